// rac_gemm.hip — rotate-project-accumulate GEMM for gfx950: the VALU tiles of
// the CORDIC and SHIFTADD MACs, and the dispatch of every product.
//
// C[M,N] = alpha * op(A) @ op(B) (+ beta * C), row-major, with the MAC of
// rac_fma_iters (rac_kernels.hip:204-219):
//   FAST     fmaf(a ^ sign(b), |b|, acc)                  == fmaf(a, b, acc)
//   CORDIC   n circular micro-rotations of (a ^ sign(b), 0), x * 1/K-hat(n),
//            projected on |b| and accumulated               (rac_math.hpp)
//   SHIFTADD acc + integer shift-add product of the top n mantissa bits of b
// op(A) = A or A^T (A stored [K,M], the TN launcher); op(B) = B or B^T
// (B stored [N,K], the NT launcher).  Each output keeps ONE accumulator over
// k = 0..K-1 in order, like every reference tile shape, so results do not
// depend on the tiling; out-of-range operands are zero-padded (a zero MAC
// leaves acc unchanged).
//
// Design: CORDIC mode costs ~2n VALU lane-ops per MAC, so the kernel is
// VALU-bound by two orders of magnitude over LDS and HBM traffic.  A 64x64
// block tile (4x4 outputs per lane, 256 lanes = 4 wave64) staged through LDS
// with BK = 16 keeps 16 independent MAC chains per lane for latency hiding
// and reads only 2 ds_read_b128 per 16 MACs; the rotations of those MACs
// advance step-major, so independent FMA chains interleave in each wave's
// instruction stream.  FAST mode (1 FMA per MAC) runs on the matrix cores
// (rac_gemm_fast.hip), here only for few k (dispatch).  Launches with fewer
// than 2 blocks of 64x64 per CU (FAST: 4) step down to 32x32 (2x2 per lane),
// so every SIMD holds several waves.  The next K-tile is
// prefetched into registers while the current one is computed.
#include <hip/hip_runtime.h>
#include <atomic>
#include "rac_act.hpp"
#include "rac_gemm.hpp"

namespace rac {

// CORDIC mode: rotations of kGroupRows tile rows (x TN columns) advance
// step-major (8 interleaved chains in the 4x4 register tile).
constexpr int kGroupRows = 2;
// Offset of a lane's i-th row (or column) inside the block tile, for the
// lane's 16-way index t.  Register tiles of 4k are split into k groups of 4
// spaced 64 apart, so a wave's float4 LDS reads of one group cover 256
// contiguous bytes (no bank conflicts for the 8x8 tile); 2 and 4 are
// contiguous.  Only the output a lane owns changes, never its arithmetic.
template <int TT>
__device__ __forceinline__ int lane_off(int t, int i) {
    if constexpr (TT % 4 == 0) return (i >> 2) * 64 + t * 4 + (i & 3);
    else return t * TT + i;
}

template <int MODE, int NITER, bool TA, bool TB, int TM, int TN>
struct GemmCfg {
    static constexpr int kThreads = 256;
    static constexpr int kBM = 16 * TM;
    static constexpr int kBN = 16 * TN;
    static constexpr int kBK = 16;
    static constexpr int kPad = 4;
    static constexpr int kALoads = kBM * kBK / kThreads;
    static constexpr int kBLoads = kBN * kBK / kThreads;
};

template <int MODE, int NITER, bool LIT = false>
__device__ __forceinline__ float mac(float a, float b, uint32_t bsign, float acc,
                                     int iters, float kinv) {
    if constexpr (MODE == kModeFast) {
        return __builtin_fmaf(a, b, acc);
    } else if constexpr (MODE == kModeCordic && LIT) {
        // the rotation as rac_kernels.hip:152-163 writes it, for inputs
        // outside the strength-reduced chain's range (cordic_needs_literal)
        const float x0 = as_f(as_u(a) ^ bsign);
        const float xr = cordic_rot_x_literal_rt(x0, NITER > 0 ? NITER : iters);
        return __builtin_fmaf(xr * kinv, __builtin_fabsf(b), acc);
    } else if constexpr (MODE == kModeCordic) {
        if constexpr (NITER > 0) {
            return mac_cordic<NITER>(a, b, bsign, acc);
        } else {
            const float x0 = as_f(as_u(a) ^ bsign);
            const float xr = cordic_rot_x_rt(x0, iters);
            return __builtin_fmaf(xr * kinv, __builtin_fabsf(b), acc);
        }
    } else {
        return acc + shiftadd_mul(a, b, iters);
    }
}

template <int MODE, int NITER, bool TA, bool TB, int TM, int TN, bool FUSED, int SCHED>
__global__ __launch_bounds__(256) void gemm_kernel(
    const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C,
    int M, int N, int K, float alpha, float beta, int iters, float kinv, long sa, long sb, long sc,
    GemmEpilogue ep, const int* k_causal, int exact_specials, int row0)
{
    using Cfg = GemmCfg<MODE, NITER, TA, TB, TM, TN>;
    constexpr int BM = Cfg::kBM, BN = Cfg::kBN, BK = Cfg::kBK, PAD = Cfg::kPad;
    // Tile schedule.  0: tile (blockIdx.y, blockIdx.x).  1 (causal attention
    // scores, square, BM == BN): only tiles on or below the diagonal, which
    // the softmax does not overwrite with -inf; workgroup (x, p) takes row p
    // col x for x <= p, else row nt-1-p col x-p-1, so every workgroup has one
    // tile and rows p and nt-1-p share a column of the grid (grid nt+1 x
    // ceil(nt/2)).  2 (causal P V): workgroup p computes row tiles p and
    // nt-1-p, whose K ranges (below) sum to a constant.  3 (causal attention
    // scores of query rows row0.. row0+M-1 against keys 0..N-1): only the
    // tiles on or below the diagonal, numbered row by row (row tile r has
    // trap_cols(r) of them), one workgroup each; consecutive workgroups go to
    // consecutive XCDs, so the trapezoid's work spreads over all of them (a
    // rectangular grid with the upper tiles skipped leaves the live ones on
    // a few XCDs).
    int tm = blockIdx.y, tn = blockIdx.x, tm2 = -1;
    if constexpr (SCHED == 3) {
        int l = blockIdx.x;
        tm = 0;
        for (;;) {
            const int c = trap_cols(row0, tm, BM, BN, N);
            if (l < c) break;
            l -= c;
            tm++;
        }
        tn = l;
    }
    if constexpr (SCHED == 1) {
        const int nt = (M + BM - 1) / BM, p = blockIdx.y, x = blockIdx.x;
        if (x > p) {
            tm = nt - 1 - p;
            tn = x - p - 1;
            if (tm == p) return;     // middle row of an odd tile count: covered by x <= p
        }
    } else if constexpr (SCHED == 2) {
        const int nt = (M + BM - 1) / BM, p = blockIdx.y;
        if (nt - 1 - p != p) tm2 = nt - 1 - p;
    }
    const long m0a = (long)tm * BM, m0b = tm2 < 0 ? -1L : (long)tm2 * BM, n0 = (long)tn * BN;
    A += (long)blockIdx.z * sa;
    B += (long)blockIdx.z * sb;
    C += (long)blockIdx.z * sc;
    __shared__ __attribute__((aligned(16))) float sA[BK][BM + PAD];
    __shared__ __attribute__((aligned(16))) float sB[BK][BN + PAD];
    // CORDIC mode: lit_pass[pass] is set when some A element of the output
    // tile's row panel lies outside the strength-reduced chain's range
    // (cordic_needs_literal); the tile is then recomputed on the literal
    // chain.  One flag per pass, so no flag is cleared while being read.
    __shared__ int lit_pass[2];

    const int tid = threadIdx.x;
    const int tx = tid % 16, ty = tid / 16;
    if constexpr (MODE == kModeCordic) {
        if (tid == 0) lit_pass[0] = lit_pass[1] = 0;   // ordered before any set by the K loop's barriers
    }

    constexpr int kPasses = SCHED == 2 ? 2 : 1;
    for (int pass = 0; pass < kPasses; pass++) {
        const long m0 = pass ? m0b : m0a;
        if (m0 < 0) break;

        float acc[TM][TN];
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = 0.0f;

        float ra[Cfg::kALoads], rb[Cfg::kBLoads];
        // Range of the A elements this lane staged, as |a| bit patterns: the
        // largest, and the smallest minus one (unsigned, so +-0 never counts).
        uint32_t a_hi = 0u, a_lo_m1 = 0xffffffffu;

        // Global -> register staging of one K-tile; element (m, k) of op(A) and
        // (k, n) of op(B), zero outside the matrix (FAST: -0 in A, so that the
        // product -0 leaves a -0 accumulator as it is too).  Index order is
        // chosen so consecutive lanes read consecutive addresses.
        auto load_tile = [&](int k0) {
#pragma unroll
            for (int r = 0; r < Cfg::kALoads; r++) {
                const int idx = tid + r * 256;
                int mm, kk;
                if constexpr (TA) { kk = idx / BM; mm = idx % BM; }
                else { mm = idx / BK; kk = idx % BK; }
                const long gm = m0 + mm, gk = (long)k0 + kk;
                float v = MODE == kModeFast ? -0.0f : 0.0f;
                if (gm < M && gk < K) v = TA ? A[gk * M + gm] : A[gm * K + gk];
                ra[r] = v;
            }
#pragma unroll
            for (int r = 0; r < Cfg::kBLoads; r++) {
                const int idx = tid + r * 256;
                int nn, kk;
                if constexpr (TB) { nn = idx / BK; kk = idx % BK; }
                else { kk = idx / BN; nn = idx % BN; }
                const long gn = n0 + nn, gk = (long)k0 + kk;
                float v = 0.0f;
                if (gn < N && gk < K) v = TB ? B[gn * K + gk] : B[gk * N + gn];
                rb[r] = v;
            }
        };
        auto store_tile = [&]() {
#pragma unroll
            for (int r = 0; r < Cfg::kALoads; r++) {
                const int idx = tid + r * 256;
                int mm, kk;
                if constexpr (TA) { kk = idx / BM; mm = idx % BM; }
                else { mm = idx / BK; kk = idx % BK; }
                sA[kk][mm] = ra[r];
                if constexpr (MODE == kModeCordic) {
                    const uint32_t u = as_u(ra[r]) & 0x7fffffffu;
                    a_hi = max(a_hi, u);
                    a_lo_m1 = min(a_lo_m1, u - 1u);
                }
            }
#pragma unroll
            for (int r = 0; r < Cfg::kBLoads; r++) {
                const int idx = tid + r * 256;
                int nn, kk;
                if constexpr (TB) { nn = idx / BK; kk = idx % BK; }
                else { kk = idx / BN; nn = idx % BN; }
                sB[kk][nn] = rb[r];
            }
        };

        // Causal P V: row t of P is exactly 0 beyond column t, and with every v
        // finite (*k_causal == 1, checked on the device) fma(0, v, acc) == acc
        // (a zero accumulator at most changes its sign), so the K loop stops
        // after the tile's last row (query position row0 + m0 + BM - 1).
        int kend = K;
        if (k_causal && *k_causal == 1) kend = (int)min((long)K, (long)row0 + m0 + BM);
        load_tile(0);
        for (int k0 = 0; k0 < kend; k0 += BK) {
            __syncthreads();            // previous tile fully consumed
            store_tile();
            __syncthreads();
            if (k0 + BK < kend) load_tile(k0 + BK);   // prefetch overlaps the MACs
            // CORDIC steps are long VALU chains and stay rolled in the plain
            // 4x4 schedules; the 2x2 register tile (4 rotations per k-step,
            // too few independent chains to cover each step's LDS reads)
            // and the square causal attention schedules take two k-steps
            // per trip (measured: 1024^3 0.616 -> 0.542 ms, the attention
            // core with P kept 9.75 -> 9.36 ms; the 4096^3 NN launch 1%
            // slower, so it keeps one).  The accumulation order is unchanged.
            constexpr int KU = (TM * TN <= 4 || SCHED == 1 || SCHED == 2) ? 2 : 1;
#pragma unroll 1
            for (int kb = 0; kb < BK; kb += KU)
#pragma unroll
            for (int ku = 0; ku < KU; ku++) {
                const int kk = kb + ku;
                float a[TM], b[TN];
                uint32_t bs[TN];
                if constexpr (TM % 4 == 0) {
#pragma unroll
                    for (int i = 0; i < TM; i += 4) {
                        const float4 v = *reinterpret_cast<const float4*>(&sA[kk][lane_off<TM>(ty, i)]);
                        a[i] = v.x; a[i + 1] = v.y; a[i + 2] = v.z; a[i + 3] = v.w;
                    }
                } else {
                    static_assert(TM == 2, "register tile");
                    const float2 v = *reinterpret_cast<const float2*>(&sA[kk][ty * TM]);
                    a[0] = v.x; a[1] = v.y;
                }
                if constexpr (TN % 4 == 0) {
#pragma unroll
                    for (int j = 0; j < TN; j += 4) {
                        const float4 v = *reinterpret_cast<const float4*>(&sB[kk][lane_off<TN>(tx, j)]);
                        b[j] = v.x; b[j + 1] = v.y; b[j + 2] = v.z; b[j + 3] = v.w;
                    }
                } else {
                    static_assert(TN == 2, "register tile");
                    const float2 v = *reinterpret_cast<const float2*>(&sB[kk][tx * TN]);
                    b[0] = v.x; b[1] = v.y;
                }
#pragma unroll
                for (int j = 0; j < TN; j++) bs[j] = as_u(b[j]) & 0x80000000u;
                if constexpr (MODE == kModeCordic && NITER > 0) {
                    // the rotations of kGroupRows x TN MACs advance step-major
                    // (independent chains interleave; same bits as mac<>)
                    constexpr int G = kGroupRows < TM ? kGroupRows : TM;
#pragma unroll
                    for (int i0 = 0; i0 < TM; i0 += G) {
                        float xr[G * TN];
#pragma unroll
                        for (int gi = 0; gi < G; gi++)
#pragma unroll
                            for (int j = 0; j < TN; j++) xr[gi * TN + j] = as_f(as_u(a[i0 + gi]) ^ bs[j]);
                        cordic_rot_x_vec<NITER, G * TN>(xr);
#pragma unroll
                        for (int gi = 0; gi < G; gi++)
#pragma unroll
                            for (int j = 0; j < TN; j++)
                                acc[i0 + gi][j] = __builtin_fmaf(xr[gi * TN + j] * cordic_kinv(NITER),
                                                                 __builtin_fabsf(b[j]), acc[i0 + gi][j]);
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < TM; i++)
#pragma unroll
                        for (int j = 0; j < TN; j++)
                            acc[i][j] = mac<MODE, NITER>(a[i], b[j], bs[j], acc[i][j], iters, kinv);
                }
            }
        }

        if constexpr (MODE == kModeCordic) {
            if (exact_specials && cordic_range_needs_literal(a_lo_m1, a_hi)) lit_pass[pass] = 1;
            __syncthreads();
            if (lit_pass[pass]) {
                // Rare: the tile's A panel holds subnormal, tiny (< 2^-105),
                // top-binade, infinite or NaN elements.  Recompute it straight
                // from global memory (zero outside the matrix, as the staged
                // tiles are): those elements' MACs on the literal chain, all
                // others on the strength-reduced one (the same bits there).
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) acc[i][j] = 0.0f;
#pragma unroll 1
                for (int k = 0; k < kend; k++) {
                    float a[TM], b[TN];
#pragma unroll
                    for (int i = 0; i < TM; i++) {
                        const long gm = m0 + lane_off<TM>(ty, i);
                        a[i] = gm < M ? (TA ? A[(long)k * M + gm] : A[gm * K + k]) : 0.0f;
                    }
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        const long gn = n0 + lane_off<TN>(tx, j);
                        b[j] = gn < N ? (TB ? B[gn * K + k] : B[(long)k * N + gn]) : 0.0f;
                    }
#pragma unroll
                    for (int i = 0; i < TM; i++) {
                        if (cordic_needs_literal(a[i])) {
#pragma unroll
                            for (int j = 0; j < TN; j++)
                                acc[i][j] = mac<MODE, NITER, true>(a[i], b[j], as_u(b[j]) & 0x80000000u, acc[i][j],
                                                                   iters, NITER > 0 ? cordic_kinv(NITER > 0 ? NITER : 1)
                                                                                    : kinv);
                        } else {
#pragma unroll
                            for (int j = 0; j < TN; j++)
                                acc[i][j] = mac<MODE, NITER>(a[i], b[j], as_u(b[j]) & 0x80000000u, acc[i][j],
                                                             iters, kinv);
                        }
                    }
                }
            }
        }

#pragma unroll
        for (int i = 0; i < TM; i++) {
            const long gm = m0 + lane_off<TM>(ty, i);
            if (gm >= M) continue;
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const long gn = n0 + lane_off<TN>(tx, j);
                if (gn >= N) continue;
                float* cp = C + gm * N + gn;
                // rac_kernels.hip:267-272
                float v = (beta != 0.0f) ? __builtin_fmaf(alpha, acc[i][j], beta * *cp)
                                         : alpha * acc[i][j];
                if constexpr (FUSED) {
                    // rac_torch.cu:770-775: + bias, then the activation in
                    // registers (the pre-activation is kept when asked for)
                    if (ep.bias) v = v + ep.bias[gn];
                    if (ep.pre) ep.pre[gm * N + gn] = v;
                    v = act_rt(v, ep.act, iters, ep.khinv);
                }
                *cp = v;
            }
        }
    }   // pass
}

// flag = 1 unless some x[i] is inf or NaN (flag must be 1 on entry; lanes
// only ever store 0, so concurrent stores agree).
__global__ __launch_bounds__(256) void all_finite_kernel(const float* __restrict__ x, long n,
                                                         int* __restrict__ flag) {
    const long stride = (long)gridDim.x * blockDim.x;
    bool ok = true;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        ok &= __builtin_isfinite(x[i]);
    if (!ok) *flag = 0;
}

__global__ void set_flag_kernel(int* flag, int v) { *flag = v; }

// flag = 1 unless some element of the four arrays (n each) is 2^57 or more
// in magnitude, infinite or NaN: then a product of two of them over up to
// 4096 k stays below 2^126, and its distance from a mean of such products
// (dP - rowsum(dP P)) below 2^127, so what a causal backward pass may skip is
// 0 times something finite.
__global__ __launch_bounds__(256) void all_bounded_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                          const float* __restrict__ c, const float* __restrict__ d,
                                                          long n, int* __restrict__ flag) {
    const float* x = blockIdx.y == 0 ? a : blockIdx.y == 1 ? b : blockIdx.y == 2 ? c : d;
    typedef float v4u __attribute__((ext_vector_type(4), aligned(4)));
    float m = 0.0f;                                      // the largest magnitude; a NaN stays
    const long n4 = n / 4, stride = (long)gridDim.x * 256;
#pragma unroll 4
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n4; i += stride) {
        const v4u q = reinterpret_cast<const v4u*>(x)[i];
#pragma unroll
        for (int e = 0; e < 4; e++) m = __builtin_elementwise_maximum(m, __builtin_fabsf(q[e]));
    }
    if (blockIdx.x == 0 && threadIdx.x < n - 4 * n4)
        m = __builtin_elementwise_maximum(m, __builtin_fabsf(x[4 * n4 + threadIdx.x]));
    if (!(m < 0x1p57f)) *flag = 0;
}

hipError_t all_bounded_launch(const float* a, const float* b, const float* c, const float* d, long n, int* flag,
                              hipStream_t s) {
    hipLaunchKernelGGL(set_flag_kernel, dim3(1), dim3(1), 0, s, flag, 1);
    const long blocks = n / 4096 + 1;
    hipLaunchKernelGGL(all_bounded_kernel, dim3((unsigned)(blocks < 1024 ? blocks : 1024), 4), dim3(256), 0, s, a, b,
                       c, d, n, flag);
    return hipGetLastError();
}

hipError_t all_finite_launch(const float* x, long n, int* flag, hipStream_t s) {
    hipLaunchKernelGGL(set_flag_kernel, dim3(1), dim3(1), 0, s, flag, 1);
    long blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(all_finite_kernel, dim3((unsigned)blocks), dim3(256), 0, s, x, n, flag);
    return hipGetLastError();
}

template <int MODE, int NITER, bool TA, bool TB, bool FUSED, int SCHED, int TM, int TN = TM>
static hipError_t launch_cfg(const GemmArgs& g, hipStream_t stream) {
    using Cfg = GemmCfg<MODE, NITER, TA, TB, TM, TN>;
    const float kinv = cordic_kinv(g.iters);
    const unsigned nt = (unsigned)((g.M + Cfg::kBM - 1) / Cfg::kBM);
    dim3 grid((unsigned)((g.N + Cfg::kBN - 1) / Cfg::kBN), nt, (unsigned)g.batch);
    if (g.sched == 1) grid = dim3(nt + 1, (nt + 1) / 2, (unsigned)g.batch);
    if (g.sched == 2) grid.y = (nt + 1) / 2;
    if (g.sched == 3) {
        long tiles = 0;
        for (unsigned r = 0; r < nt; r++) tiles += trap_cols(g.row0, (int)r, Cfg::kBM, Cfg::kBN, g.N);
        grid = dim3((unsigned)tiles, 1, (unsigned)g.batch);
    }
    hipLaunchKernelGGL((gemm_kernel<MODE, NITER, TA, TB, TM, TN, FUSED, SCHED>), grid, dim3(256), 0, stream,
                       g.A, g.B, g.C, g.M, g.N, g.K, g.alpha, g.beta, g.iters, kinv, g.sa, g.sb, g.sc,
                       g.ep, g.k_causal, g.exact_specials, g.row0);
    return hipGetLastError();
}

// Compute units of the current device (256 on MI355X), cached per device.
long device_cus() {
    static std::atomic<long> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
        (void)hipGetLastError();
        return 256;
    }
    long v = cached[dev].load(std::memory_order_relaxed);
    if (v == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
            (void)hipGetLastError();
            n = 256;
        }
        v = n;
        cached[dev].store(v, std::memory_order_relaxed);
    }
    return v;
}

// Register tile: 4x4 per lane (64x64 block), stepping down to 2x2 (32x32)
// while the launch would have too few blocks; the triangular and paired-row
// schedules keep the 64x64 tile they are written for.  The tile never
// changes a result: each output is one accumulator over k in order.
template <int MODE, int NITER, bool TA, bool TB, bool FUSED, int SCHED = 0>
static hipError_t launch_tiles(const GemmArgs& g, hipStream_t s) {
    if constexpr (SCHED == 2) {
        // Causal P V, row tiles p and nt-1-p per workgroup (equal K sums): on
        // 64x64 tiles while that gives 2 workgroups per CU, else on 32x32
        // while 4 per CU (the attention core's 512-row chunks: 4-9% faster
        // than unpaired), else unpaired (256-row chunks: no gain)
        const long cus = device_cus();
        const long pairs4 = (((g.M + 63) / 64 + 1) / 2) * ((g.N + 63) / 64) * (long)g.batch;
        if (pairs4 >= 2 * cus) return launch_cfg<MODE, NITER, TA, TB, FUSED, SCHED, 4>(g, s);
        const long pairs2 = (((g.M + 31) / 32 + 1) / 2) * ((g.N + 31) / 32) * (long)g.batch;
        if (pairs2 >= 4 * cus) return launch_cfg<MODE, NITER, TA, TB, FUSED, SCHED, 2>(g, s);
        GemmArgs h = g;
        h.sched = 0;
        return launch_tiles<MODE, NITER, TA, TB, FUSED, 0>(h, s);
    } else if constexpr (SCHED == 1) {
        return launch_cfg<MODE, NITER, TA, TB, FUSED, SCHED, 4>(g, s);
    } else {
        long tiles = 0;                      // of 64x64
        if constexpr (SCHED == 3) {          // the causal trapezoid's only
            for (long r = 0; r < (g.M + 63) / 64; r++) tiles += trap_cols(g.row0, (int)r, 64, 64, g.N);
        } else {
            tiles = (long)((g.M + 63) / 64) * ((g.N + 63) / 64);
        }
        tiles *= g.batch;
        // two 64x64 blocks per CU (2 waves per SIMD, 16 MAC chains each)
        // still beat 32x32 blocks (measured, same bits: 512-1023 blocks 5-6%
        // faster, e.g. the attention core's P V chunks 32 x 512 x 128 x K; at
        // one block per CU 43% slower).  FAST comes here with a few k only,
        // when the stores bound it: 4 blocks per CU (800 x 3913 x 1, 806
        // blocks: 9.5 us on 64x64, 7.7 on 32x32)
        if (tiles >= (MODE == kModeFast ? 4 : 2) * device_cus())
            return launch_cfg<MODE, NITER, TA, TB, FUSED, SCHED, 4>(g, s);
        return launch_cfg<MODE, NITER, TA, TB, FUSED, SCHED, 2>(g, s);
    }
}

// The fused epilogue exists for the NT layout only (input @ weight^T, the
// linear layer), the triangular and trapezoidal schedules for NT only
// (causal Q K^T) and the paired-row schedule for NN only (causal P V);
// their callers never ask for another layout.
template <int MODE, int NITER>
static hipError_t launch_layout(int ta, int tb, const GemmArgs& g, hipStream_t s) {
    if (g.fused) return launch_tiles<MODE, NITER, false, true, true>(g, s);
    if (g.sched == 1) return launch_tiles<MODE, NITER, false, true, false, 1>(g, s);   // NT only
    if (g.sched == 2) return launch_tiles<MODE, NITER, false, false, false, 2>(g, s);  // NN only
    if (g.sched == 3) return launch_tiles<MODE, NITER, false, true, false, 3>(g, s);   // NT only
    if (!ta && !tb) return launch_tiles<MODE, NITER, false, false, false>(g, s);
    if (!ta && tb) return launch_tiles<MODE, NITER, false, true, false>(g, s);
    if (ta && !tb) return launch_tiles<MODE, NITER, true, false, false>(g, s);
    return launch_tiles<MODE, NITER, true, true, false>(g, s);
}

// FAST products of few rows or columns that the few-row kernels run better
// than the matrix cores: their fold takes 4.6 cycles a k, a matrix instruction
// 8, and they start sooner, but they spread a long K's loads over fewer lanes
// and take more workgroups for the same outputs.  Both sides measured (us,
// few-row kernel / matrix cores), NT unless noted: 4 x 2036 x 64 3.1 / 3.6, x
// 200 3.8 / 4.7, x 400 5.2 / 5.8, x 512 5.5 / 5.7, x 700 7.0 / 7.2, x 1024 8.8 /
// 8.1; 3 x 6874 (430 workgroups) x 200 4.1 / 4.8, x 400 5.8 / 6.0; but 1 x 4000
// x 300 5.2 / 4.9, 16 x 6874 x 64 4.5 / 4.2, 1 x 11008 x 64 5.2 / 3.0.  One row
// times a matrix stored k by k stays ahead while that is small: 1 x 62 x 4096
// 25 / 32, 1 x 512 x 4096 24 / 26, 1 x 2048 x 1024 8.6 / 8.7, x 1500 12.4 / 11.9.
// Batches of at most 16 x 16: 60000 of 8 x 8 x 8 112 / 580 (2000 of 4 x 4 x 4 5.9,
// on the VALU tiles 7.2).
static bool fast_few_rows(int tb, const GemmArgs& g) {
    const long cus = device_cus();
    const int r = g.M <= kSkinnyMaxRows ? g.M : g.N;
    const long blocks = (long)((g.M <= kSkinnyMaxRows ? g.N : g.M) + 15) / 16 * g.batch;
    if (r > kSkinnyMaxRows) return false;
    if (g.M == 1 && !tb && blocks <= cus / 2 && (long)g.N * g.K * g.batch <= (1L << 21)) return true;
    if (g.K <= 256 && ((g.M <= 16 && g.N <= 16) || (r >= 2 && r <= 8 && blocks <= 2 * cus))) return true;
    return g.K <= 512 && blocks <= (r == 1 ? cus / 2 : cus);
}

static hipError_t dispatch(int ta, int tb, int mode, const GemmArgs& g, hipStream_t s) {
    auto skinny = [&] {
        return gemm_skinny_launch({g.A, g.B, g.C, g.M, g.N, g.K, g.alpha, g.beta, g.iters, g.batch, g.sa, g.sb, g.sc,
                                   g.ep, g.fused, tb != 0, g.k_causal, g.exact_specials, g.row0}, mode, s);
    };
    if (mode == kModeFast) {
        if (g.M == 1) ta = 0;                                // vectors
        if (g.N == 1) tb = 1;
        const bool plain = g.sched == 0 && !g.k_causal && g.k_side != 3;
        const bool few_rows = plain && !ta && fast_few_rows(tb, g);
        // up to 16 k, one K-tile, of up to 2^21 outputs are bound by the start of
        // a launch, which is shortest on the VALU tiles: 300 x 300 x 9 2.7 us, on
        // the matrix cores 3.1, 679 x 1739 x 16 4.6 against 6.3, 12 x 300 x 9 2.5
        // against 3.5 (2.9 on the few-row kernel); past them the stores dominate,
        // which the matrix-core tiles make in 16 bytes (1166 x 3868 x 9 11.8 us
        // against 8.2).  Not for SiLU, whose epilogue there has four exps in
        // flight (300 x 300 x 9 7.3 us against 4.1).
        const bool few_k = plain && g.K <= 16 && (long)g.M * g.N * g.batch <= (1L << 21) &&
                           !(g.fused && g.ep.act == kActSilu);
        // and for fewer than 4 k, which the 16-byte loads cannot read, and where
        // both operands hold 2 or 3 rows side by side
        const bool thin_a = ta && g.M > 1 && g.M < 4, thin_b = !tb && g.N > 1 && g.N < 4;
        if (few_rows && (!few_k || (g.M <= 16 && g.N <= 16 && g.batch > device_cus()))) return skinny();
        if (g.K >= 4 && !(thin_a && thin_b) && !few_k) return gemm_fast_launch(ta, tb, g, s);
        return launch_layout<kModeFast, 0>(ta, tb, g, s);
    }
    // few rows or columns (schedule 2, the causal P V, is then the plain
    // product with its causal K limit, which those kernels apply)
    if ((g.sched == 0 || g.sched == 2) && !ta && (g.M <= kSkinnyMaxRows || g.N <= kSkinnyMaxRows))
        return skinny();
    if (mode == kModeShiftAdd) return launch_layout<kModeShiftAdd, 0>(ta, tb, g, s);
    switch (g.iters) {
        case 8: return launch_layout<kModeCordic, 8>(ta, tb, g, s);
        case 16: return launch_layout<kModeCordic, 16>(ta, tb, g, s);
        case 24: return launch_layout<kModeCordic, 24>(ta, tb, g, s);
        default: return launch_layout<kModeCordic, 0>(ta, tb, g, s);
    }
}

hipError_t gemm_launch(int ta, int tb, const float* A, const float* B, float* C,
                       int M, int N, int K, float alpha, float beta, int iters, int mode,
                       hipStream_t s, int batch, long sa, long sb, long sc, int sched,
                       const int* k_causal, bool exact_specials, int row0, int k_side, int period) {
    const GemmArgs g{A, B, C, M, N, K, alpha, beta, clamp_iters(iters), batch, sa, sb, sc,
                     GemmEpilogue(), false, sched, k_causal, exact_specials ? 1 : 0, row0, k_side, period};
    return dispatch(ta, tb, mode, g, s);
}

hipError_t gemm_fused_launch(const float* A, const float* W, float* C, int M, int N, int K,
                             const GemmEpilogue& ep, int iters, int mode, hipStream_t s) {
    const GemmArgs g{A, W, C, M, N, K, 1.0f, 0.0f, clamp_iters(iters), 1, 0, 0, 0, ep, true, 0, nullptr, 1, 0, 0, 0};
    return dispatch(0, 1, mode, g, s);
}

hipError_t gemm_fused_half_launch(const void* A, const void* W, const void* bias, void* C, int M, int N, int K,
                                  const GemmEpilogue& ep, int iters, int dtype, hipStream_t s) {
    GemmEpilogue e = ep;
    e.bias = static_cast<const float*>(bias);                  // of the operands' type
    const GemmArgs g{static_cast<const float*>(A), static_cast<const float*>(W), static_cast<float*>(C), M, N, K, 1.0f,
                     0.0f, clamp_iters(iters), 1, 0, 0, 0, e, true, 0, nullptr, 1, 0, 0, 0};
    return gemm_fast_half_launch(dtype, g, s);
}

}  // namespace rac

// rac_gemm_fast.hip — the FAST-mode GEMM (one fmaf per MAC, k in order) on
// the FP32 matrix cores of gfx950.
//
// v_mfma_f32_16x16x4_f32 adds four products to each of its 16 x 16
// accumulators, one after the other in k order, each with a single IEEE
// rounding and denormals kept: the value of the chain
//   fmaf(a3, b3, fmaf(a2, b2, fmaf(a1, b1, fmaf(a0, b0, acc))))
// (checked on gfx950 against glibc's fmaf over 21 M random, subnormal,
// special and cancelling operand sets: 0 differences; the reverse order and
// separate roundings differ in millions).  Issued in k order it therefore
// gives every output the FAST MAC's accumulation chain (rac_fma_iters,
// rac_kernels.hip:204-219) bit for bit.  A single dependent chain issues at
// the full rate (32.2 cycles per instruction, measured), so a wave needs
// only one 16 x 16 tile to keep its matrix core busy, 8 cycles per k and 256
// outputs, where the 32x32x1_2b form needs 2048 outputs for it.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
#include "rac_act.hpp"
#include "rac_gemm.hpp"

namespace rac {

typedef float v4f __attribute__((ext_vector_type(4)));
// a float4 at any 4-byte boundary (global_load / store_dwordx4 need no more)
typedef float v4u __attribute__((ext_vector_type(4), aligned(4)));

// Elements of the operands and the output: float, or the 16-bit formats of a
// half-precision linear layer, widened (exactly) on the way to LDS and
// rounded to nearest even on the way out: what converting whole tensors
// before and after would give, without their passes over memory.
// Q: four elements as loaded; shifted(): the first `sh` dropped, zeros behind
// (NEG: negative ones).
struct Bf16 { uint16_t bits; };
struct F16 { uint16_t bits; };
typedef uint32_t u2a __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));

template <class T>
struct Elem;
template <>
struct Elem<float> {
    using Q = v4f;
    static __device__ __forceinline__ Q load(const float* p) {
        const v4u t = *reinterpret_cast<const v4u*>(p);
        return v4f{t.x, t.y, t.z, t.w};
    }
    static __device__ __forceinline__ v4f widen(Q v) { return v; }
    template <bool NEG>
    static __device__ __forceinline__ Q shifted(Q v, int sh) {
        constexpr float z = NEG ? -0.0f : 0.0f;
        if (sh & 1) v = v4f{v.y, v.z, v.w, z};
        if (sh & 2) v = v4f{v.z, v.w, z, z};
        if (sh & 4) v = v4f{z, z, z, z};
        return v;
    }
    static __device__ __forceinline__ float get(const float* p) { return *p; }
    static __device__ __forceinline__ void store(float* p, v4f v, int n) {
        if (n >= 4) {
            *reinterpret_cast<v4u*>(p) = v4u{v.x, v.y, v.z, v.w};
            return;
        }
        if (n > 0) p[0] = v.x;
        if (n > 1) p[1] = v.y;
        if (n > 2) p[2] = v.z;
    }
};
template <class T>
struct Elem16 {
    using Q = u2v;
    static __device__ __forceinline__ Q load(const T* p) {
        const u2a t = *reinterpret_cast<const u2a*>(p);
        return u2v{t.x, t.y};
    }
    template <bool NEG>
    static __device__ __forceinline__ Q shifted(Q v, int sh) {
        constexpr uint64_t z = NEG ? 0x8000800080008000u : 0;
        if (sh <= 0) return v;
        const uint64_t x = sh >= 4 ? z : (((uint64_t)v.y << 32) | v.x) >> (16 * sh) | z << (64 - 16 * sh);
        return u2v{(uint32_t)x, (uint32_t)(x >> 32)};
    }
};
template <>
struct Elem<Bf16> : Elem16<Bf16> {
    static __device__ __forceinline__ v4f widen(Q v) {
        return v4f{as_f(v.x << 16), as_f(v.x & 0xffff0000u), as_f(v.y << 16), as_f(v.y & 0xffff0000u)};
    }
    static __device__ __forceinline__ float get(const Bf16* p) { return as_f((uint32_t)p->bits << 16); }
    static __device__ __forceinline__ void store(Bf16* p, v4f v, int n) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const uint32_t u = as_u(v[r]);
            const uint32_t h = v[r] != v[r] ? 0x7fc0u : (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
            if (r < n) p[r].bits = (uint16_t)h;
        }
    }
};
template <>
struct Elem<F16> : Elem16<F16> {
    static __device__ __forceinline__ float widen1(uint32_t bits) {
        const uint16_t h = (uint16_t)bits;
        _Float16 f;
        __builtin_memcpy(&f, &h, 2);
        return (float)f;
    }
    static __device__ __forceinline__ v4f widen(Q v) {
        return v4f{widen1(v.x), widen1(v.x >> 16), widen1(v.y), widen1(v.y >> 16)};
    }
    static __device__ __forceinline__ float get(const F16* p) { return widen1(p->bits); }
    static __device__ __forceinline__ void store(F16* p, v4f v, int n) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const _Float16 f = (_Float16)v[r];
            if (r < n) __builtin_memcpy(&p[r].bits, &f, 2);
        }
    }
};

// One operand's K-tile (KT k x ROWS rows) of a workgroup: global ->
// registers -> LDS -> matrix-core operands.  Lane l of the instruction
// holds element (row l % 16, k = 4 t + l / 16) of step t.
//
// KC (k contiguous in memory: A, or B^T of the NT layout): LDS rows of KT +
// 8 floats, each 16-k group stored with k = 4 t + q at 4 q + t, so one
// ds_read_b128 gives a lane its elements of four consecutive steps.  Rows 8
// floats off a multiple of 16 are what keeps those reads free of bank
// conflicts (measured: 4.1-4.5 cycles an instruction, like contiguous
// lanes; 4 off 8.0, 0 off 32: 128 x 11008 x 4096 123 -> 109 us, 1024^3 24.6 ->
// 22.4); the scattering writes take 6.5 (4 off: 5.0-6.4).  Otherwise LDS rows
// are k rows of ROWS + pad floats (= 16 mod 32: the two k of a half wave on
// opposite banks), read a step at a time.
template <class T, bool KC, int ROWS, int KT, int NL, bool THIN = false>
struct FastTile {
    using El = Elem<T>;
    using Q = typename El::Q;
    static constexpr int kStride = KC ? KT + 8 : ROWS + ((48 - ROWS % 32) % 32);
    static constexpr int kFloats = (KC ? ROWS : KT) * kStride;
    static constexpr int kVecs = ROWS * KT / 4;                     // float4 of the tile
    static constexpr int kVPT = (kVecs + NL - 1) / NL;              // per lane
    static constexpr int kPer = KC ? KT / 4 : ROWS / 4;             // float4 per LDS row

    // this lane's global addresses at the next K-tile to load; rows past the
    // matrix read rows inside it (their outputs are never stored)
    const T* p[kVPT];
    long step;                                                      // one K-tile further
    int shift;                                                      // !KC: see fix_rows()

    __device__ __forceinline__ static bool on(int i) { return kVecs % NL == 0 || (int)threadIdx.x + i * NL < kVecs; }
    __device__ __forceinline__ void init(const T* P, long ld, long rows, long r0, long k0) {
        const int tid = threadIdx.x;
        step = KC ? KT : (long)KT * ld;
        shift = 0;
        long r = 0;
        if constexpr (!KC) {
            // four rows inside the matrix (it has at least 4)
            const long want = r0 + (tid % kPer) * 4;
            r = THIN ? 0 : min(want, rows - 4);
            shift = THIN ? (int)rows - 1 : (int)min(want - r, 3L);      // THIN: the last row
        }
#pragma unroll
        for (int i = 0; i < kVPT; i++) {
            const int idx = tid + i * NL;
            if constexpr (KC) p[i] = P + min(r0 + idx / kPer, rows - 1) * ld + k0 + (idx % kPer) * 4;
            else p[i] = P + (k0 + idx / kPer) * ld + r;
        }
    }
    // The K-tile at hand has only `kn` (1 .. KT - 1) of its k, and the matrix
    // at least 4: addresses move back inside K; fix_k() then puts the
    // elements where they belong and zeroes those past K, negative zeros in
    // one operand: adding the product -0 leaves every accumulator as it is,
    // the -0 of a chain of underflowed negative products too.
    __device__ __forceinline__ void retreat(int kn, long ld) {
#pragma unroll
        for (int i = 0; i < kVPT; i++) {
            const int idx = threadIdx.x + i * NL;
            if constexpr (KC) p[i] -= max(0, (idx % kPer) * 4 + 4 - kn);
            else p[i] -= max(0, idx / kPer + 1 - kn) * ld;
        }
    }
    __device__ __forceinline__ void load(Q (&v)[kVPT], int i) const {
        if constexpr (THIN) {
            if (on(i)) v[i] = v4f{p[i][0], p[i][min(1, shift)], p[i][min(2, shift)], 0.0f};
        } else if (on(i)) {
            v[i] = El::load(p[i]);
        }
    }
    __device__ __forceinline__ void advance(long by) {
#pragma unroll
        for (int i = 0; i < kVPT; i++) p[i] += by;
    }
    template <bool NEG>
    __device__ __forceinline__ static void fix_k(Q (&v)[kVPT], int kn) {
#pragma unroll
        for (int i = 0; i < kVPT; i++) {
            const int idx = threadIdx.x + i * NL;
            if constexpr (KC) v[i] = El::template shifted<NEG>(v[i], min(4, max(0, (idx % kPer) * 4 + 4 - kn)));
            else v[i] = El::template shifted<NEG>(v[i], idx / kPer >= kn ? 4 : 0);
        }
    }
    // !KC, tiles past the last row: lanes that moved back to stay inside
    // the matrix put their rows where they belong
    __device__ __forceinline__ void fix_rows(Q (&v)[kVPT]) const {
#pragma unroll
        for (int i = 0; i < kVPT; i++)
            if constexpr (!THIN) v[i] = El::template shifted<false>(v[i], shift);
    }
    __device__ __forceinline__ static void store(float* S, const Q (&q)[kVPT], int i) {
        const int idx = threadIdx.x + i * NL;
        if (!on(i)) return;
        const v4f v = El::widen(q[i]);
        if constexpr (KC) {
            const int c = idx % kPer;
            float* s = S + (idx / kPer) * kStride + (c / 4) * 16 + c % 4;
            s[0] = v.x;
            s[4] = v.y;
            s[8] = v.z;
            s[12] = v.w;
        } else {
            *reinterpret_cast<v4f*>(S + (idx / kPer) * kStride + (idx % kPer) * 4) = v;
        }
    }
    // the lane's elements of steps 4 g .. 4 g + 3 (k = 16 g .. 16 g + 15)
    // for the 16 rows at `row`
    __device__ __forceinline__ static v4f frag(const float* S, int row, int g) {
        const int l = threadIdx.x & 63;
        if constexpr (KC) {
            return *reinterpret_cast<const v4f*>(S + (row + l % 16) * kStride + 16 * g + 4 * (l / 16));
        } else {
            const float* s = S + (16 * g + l / 16) * kStride + row + l % 16;
            return v4f{s[0], s[4 * kStride], s[8 * kStride], s[12 * kStride]};
        }
    }
};

struct FastGeom {
    int M, N, K;
    long sa, sb, sc;
    float alpha, beta;
    int iters;
    GemmEpilogue ep;
    const int* k_causal;
    int k_side;           // 0: every k; 1-3: the causal limits of GemmArgs, when *k_causal holds 1
    int row0, period;
    int tiles, tiles_m;   // output tiles of one batch item, rows of them
    int batch;
    long total;           // tiles * batch
};

// alpha / beta, bias and activation of outputs (gm, gn .. gn + 3).  FUSED:
// on every lane, whose rows and columns past the matrix are copies of its
// last; only the stores look at the edges.  With the lanes past M leaving
// first, few rows paid for it (1 x 11008 x 64 with SiLU 6.7 us, 3.9 now; 4 x
// 2036 x 64 5.9, 4.6), and the activations wait on their own latency: four
// side by side, one call each (ReLU 0.3, GELU 0.2 us less than one by one).
template <bool FUSED, class T>
__device__ __forceinline__ void fast_epilogue(T* __restrict__ C, int M, int N, long gm, long gn, v4f acc,
                                              const FastGeom& g) {
    const int left = (int)min(4L, (long)N - gn);
    const bool in = gm < M && left > 0;
    if (!FUSED && !in) return;
    T* cp = C + gm * N + gn;
    v4f v;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        // rac_kernels.hip:267-272
        v[r] = g.alpha * acc[r];
        if constexpr (!FUSED) {
            if (g.beta != 0.0f && r < left) v[r] = __builtin_fmaf(g.alpha, acc[r], g.beta * cp[r]);
        }
    }
    if constexpr (FUSED) {
        // rac_torch.cu:770-775
        if (g.ep.bias) {
            const T* bias = reinterpret_cast<const T*>(g.ep.bias);
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = v[r] + Elem<T>::get(bias + min(gn + r, (long)N - 1));
        }
        if (g.ep.pre && in) Elem<float>::store(g.ep.pre + gm * N + gn, v, left);
        float x[4] = {v.x, v.y, v.z, v.w};
        if (g.ep.act == kActSilu) {
            if (g.iters == 24) {
                elt_vec<kEltSilu, 24, 4>(x, g.iters, g.ep.khinv);
            } else if (g.iters == 16) {
                elt_vec<kEltSilu, 16, 4>(x, g.iters, g.ep.khinv);
            } else {
                // one copy: x rotates
#pragma unroll 1
                for (int r = 0; r < 4; r++) {
                    const float y = act_rt(x[0], kActSilu, g.iters, g.ep.khinv);
                    x[0] = x[1];
                    x[1] = x[2];
                    x[2] = x[3];
                    x[3] = y;
                }
            }
        } else if (g.ep.act == kActGelu) {
            elt_vec<kEltGelu, 0, 4>(x, 0, 0.0f);
        } else if (g.ep.act == kActRelu) {
            elt_vec<kEltRelu, 0, 4>(x, 0, 0.0f);
        }
        v = v4f{x[0], x[1], x[2], x[3]};
        if (!in) return;
    }
    Elem<T>::store(cp, v, left);
}

// Output tile BM x BN, WR x WC waves, K-tiles of KT in two LDS buffers, PD
// K-tiles in flight in registers.  Per K-tile and buffer one barrier: while
// the MACs of one run, the next is written into the other buffer and the
// one PD further is requested.  SPREAD 0 does that ahead of the MACs, 1
// between them, 2 between them with the order held by scheduling barriers
// (a lone wave per SIMD issues them in the shadow of its matrix
// instructions: 32x4096x4096 on 32x32 tiles 34.7 -> 24.9 us).
template <bool TA, bool TB, bool FUSED, bool TRAP, int BM, int BN, int WR, int WC, int KT, int PD, int SPREAD, bool THIN, class T>
__global__ __launch_bounds__(64 * WR * WC) void gemm_fast_kernel(const T* __restrict__ A, const T* __restrict__ B,
                                                                 T* __restrict__ C, FastGeom g)
{
    constexpr int NL = 64 * WR * WC;
    using TAt = FastTile<T, !TA, BM, KT, NL, TA && THIN && BM == 16>;
    using TBt = FastTile<T, TB, BN, KT, NL, !TB && THIN && BN == 16>;
    constexpr int TM = BM / WR, TN = BN / WC, MT = TM / 16, NT = TN / 16;
    __shared__ __attribute__((aligned(16))) float sA[2][TAt::kFloats];
    __shared__ __attribute__((aligned(16))) float sB[2][TBt::kFloats];

    const long L = blockIdx.x + (long)blockIdx.y * gridDim.x;
    if (L >= g.total) return;
    const int tiles_n = TRAP ? 1 : g.tiles / g.tiles_m;
    int z, tm, tn;
    if (g.k_side == 1 || g.k_side == 2) {
        // tiles of unequal K: the longest first, one of every batch item in
        // turn (an item's tiles stay on one XCD where 8 divides the batch)
        z = (int)(L % g.batch);
        const int t = (int)(L / g.batch);
        tm = t / tiles_n;
        tn = t - tm * tiles_n;
        if (g.k_side == 1) tm = g.tiles_m - 1 - tm;
    } else {
        // The dispatcher puts workgroup L on XCD L % 8: each XCD takes one
        // contiguous range of tiles, numbered in groups of 8 row tiles
        // down, then across, so tiles that share operand panels share an L2.
        const long q = g.total / 8, r = g.total % 8, x = L % 8;
        const long id = x * q + min(x, r) + L / 8;
        z = (int)(id / g.tiles);
        int t = (int)(id - (long)z * g.tiles);
        if constexpr (TRAP) {
            tm = 0;
            for (;;) {
                const int c = trap_cols(g.row0, tm, BM, BN, g.N);
                if (t < c) break;
                t -= c;
                tm++;
            }
            tn = t;
        } else {
            const int grp = t / (8 * tiles_n), first = grp * 8, rows = min(8, g.tiles_m - first);
            t -= grp * 8 * tiles_n;
            tm = first + t % rows;
            tn = t / rows;
        }
    }
    const int M = g.M, N = g.N;
    const long m0 = (long)tm * BM, n0 = (long)tn * BN;
    A += z * g.sa;
    B += z * g.sb;
    C += z * g.sc;
    int kbeg = 0, kend = g.K;
    bool any_k = true;
    if (g.k_side && (!g.k_causal || *g.k_causal == 1)) {
        if (g.k_side == 1) kend = (int)min((long)g.K, (long)g.row0 + m0 + BM);
        else if (g.k_side == 3) {
            // the tile's last query position
            long last = m0 + BM - 1;
            if (g.period) last = m0 / g.period == last / g.period ? last % g.period : g.period - 1;
            if (n0 > g.row0 + last) return;
        }
        else if (g.k_side == 2) {
            kbeg = (int)min((long)g.K - kFastMinK, max(0L, m0 - g.row0));
            any_k = m0 - g.row0 < g.K;
        }
    }

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave / WC) * TM, wn = (wave % WC) * TN;
    v4f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    TAt ta;
    TBt tb;
    const long lda = TA ? M : g.K, ldb = TB ? g.K : N;
    ta.init(A, lda, M, m0, kbeg);
    tb.init(B, ldb, N, n0, kbeg);
    constexpr int VA = TAt::kVPT, VB = TBt::kVPT;
    typename TAt::Q va[PD][VA];
    typename TBt::Q vb[PD][VB];
    const int kn = kend - kbeg, nfull = kn / KT, tail = kn - nfull * KT, nst = nfull + (tail ? 1 : 0);
    // only a vector across the edge holds rows of the matrix elsewhere than
    // its lanes store them
    const bool edge_a = TA && m0 + BM > M && M % 4, edge_b = !TB && n0 + BN > N && N % 4;
    // before K-tile s is loaded / after (tiles past the last reload it: the
    // loads stay unconditional, so the waits stay exact)
    auto before = [&](int s) {
        if (tail && s == nfull) {
            ta.retreat(tail, lda);
            tb.retreat(tail, ldb);
        }
    };
    auto after = [&](int s) {
        const bool more = s + 1 < nst;
        ta.advance(more ? ta.step : 0);
        tb.advance(more ? tb.step : 0);
    };
    auto fix = [&](int s, int slot) {
        if (tail && s == nfull) {
            TAt::template fix_k<true>(va[slot], tail);
            TBt::template fix_k<false>(vb[slot], tail);
        }
        if constexpr (TA) if (edge_a) ta.fix_rows(va[slot]);
        if constexpr (!TB) if (edge_b) tb.fix_rows(vb[slot]);
    };
    auto frags = [&](int buf, int q, v4f (&fa)[MT], v4f (&fb)[NT]) {
#pragma unroll
        for (int i = 0; i < MT; i++) fa[i] = TAt::frag(sA[buf], wm + 16 * i, q);
#pragma unroll
        for (int j = 0; j < NT; j++) fb[j] = TBt::frag(sB[buf], wn + 16 * j, q);
    };
    // item x of a K-tile's staging: registers -> the other LDS buffer, and
    // the slot's next load
    auto stage = [&](int buf, int slot, int x, bool ld) {
        if (x < VA) {
            TAt::store(sA[buf], va[slot], x);
            if (ld) ta.load(va[slot], x);
        } else if (x < VA + VB) {
            TBt::store(sB[buf], vb[slot], x - VA);
            if (ld) tb.load(vb[slot], x - VA);
        }
    };
    // the MACs of the K-tile in LDS buffer `buf`; `staged`: with the
    // next tile's staging, ahead of them (SPREAD 0) or spread over them; else
    // the last tile's, the 16-k groups that it has
    const int last_groups = (kn - (nst - 1) * KT + 15) / 16;
    auto compute = [&](int buf, auto staged, int slot, bool ld) {
        constexpr int Q = KT / 16, X = VA + VB;
        v4f fa[2][MT], fb[2][NT];
        if constexpr (SPREAD == 0 && decltype(staged)::value) {
#pragma unroll
            for (int x = 0; x < X; x++) stage(buf ^ 1, slot, x, ld);
        }
        frags(buf, 0, fa[0], fb[0]);
#pragma unroll
        for (int q = 0; q < Q; q++) {
            if (Q > 1 && !decltype(staged)::value && q >= last_groups) break;
            if (q + 1 < Q) frags(buf, q + 1, fa[(q + 1) & 1], fb[(q + 1) & 1]);
#pragma unroll
            for (int t = 0; t < 4; t++) {
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NT; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[q & 1][j][t], fa[q & 1][i][t], acc[i][j], 0, 0, 0);
                if constexpr (SPREAD > 0 && decltype(staged)::value) {
                    const int c = 4 * q + t;
#pragma unroll
                    for (int x = c * X / (4 * Q); x < (c + 1) * X / (4 * Q); x++) stage(buf ^ 1, slot, x, ld);
                }
                if constexpr (SPREAD == 2) __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    if (KT > 16 && any_k && nst == 1) {
        // all of K in one tile: no other to load (4 x 300 x 48 3.6 us, 3.9 with
        // the last tile loaded again in its place)
        before(0);
#pragma unroll
        for (int x = 0; x < VA; x++) ta.load(va[0], x);
#pragma unroll
        for (int x = 0; x < VB; x++) tb.load(vb[0], x);
        fix(0, 0);
#pragma unroll
        for (int x = 0; x < VA + VB; x++) stage(0, 0, x, false);
        __syncthreads();
        compute(0, std::false_type(), 0, false);
    } else if (any_k) {
#pragma unroll
        for (int s = 0; s < PD; s++) {
            before(s);
#pragma unroll
            for (int x = 0; x < VA; x++) ta.load(va[s], x);
#pragma unroll
            for (int x = 0; x < VB; x++) tb.load(vb[s], x);
            after(s);
        }
        fix(0, 0);
        before(PD);
#pragma unroll
        for (int x = 0; x < VA + VB; x++) stage(0, 0, x, true);
        after(PD);
        __syncthreads();
        int s = 0;
        for (; s + 2 < nst; s += 2) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                fix(s + u + 1, (u + 1) % PD);
                before(s + u + 1 + PD);
                compute(u, std::true_type(), (u + 1) % PD, true);
                after(s + u + 1 + PD);
                __syncthreads();
            }
        }
        if (s + 1 < nst) {
            fix(s + 1, 1 % PD);
            compute(0, std::true_type(), 1 % PD, false);
            __syncthreads();
            compute(1, std::false_type(), 0, false);
        } else {
            compute(0, std::false_type(), 0, false);
        }
    }

    // the operands are passed B first, so a lane holds four consecutive
    // columns of one row: n = 4 (lane / 16) + r, m = lane % 16 of each tile
    const long em = m0 + wm + lane % 16, en = n0 + wn + 4 * (lane / 16);
    if constexpr (FUSED) {
        // one copy of the epilogue: the accumulators rotate through it
#pragma unroll 1
        for (int i = 0; i < MT * NT; i++) {
            const v4f x = acc[0][0];
            fast_epilogue<true>(C, M, N, em + 16 * (i / NT), en + 16 * (i % NT), x, g);
#pragma unroll
            for (int j = 0; j + 1 < MT * NT; j++) acc[j / NT][j % NT] = acc[(j + 1) / NT][(j + 1) % NT];
        }
    } else {
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) fast_epilogue<false>(C, M, N, em + 16 * i, en + 16 * j, acc[i][j], g);
    }
}

template <bool TA, bool TB, bool FUSED, bool TRAP, int BM, int BN, int WR, int WC, int KT, int PD, int SPREAD, bool THIN = false,
          class T = float>
static hipError_t fast_launch(const GemmArgs& a, hipStream_t s) {
    static_assert(BM <= kFastMaxTile && BN <= kFastMaxTile, "causal operands are defined to kCausalMargin only");
    FastGeom g{a.M, a.N, a.K, a.sa, a.sb, a.sc, a.alpha, a.beta, a.iters, a.ep, a.k_causal, a.k_causal || a.k_side == 3 ? a.k_side : 0,
               a.row0, a.period, 0, (a.M + BM - 1) / BM, a.batch, 0};
    if constexpr (TRAP) {
        for (int r = 0; r < g.tiles_m; r++) g.tiles += trap_cols(g.row0, r, BM, BN, g.N);
    } else {
        g.tiles = g.tiles_m * ((g.N + BN - 1) / BN);
    }
    g.total = (long)g.tiles * g.batch;
    // a grid dimension holds fewer than 2^32 lanes
    const long gx = g.total < (1L << 22) ? g.total : (1L << 22);
    hipLaunchKernelGGL((gemm_fast_kernel<TA, TB, FUSED, TRAP, BM, BN, WR, WC, KT, PD, SPREAD, THIN, T>),
                       dim3((unsigned)gx, (unsigned)((g.total + gx - 1) / gx)), dim3(64 * WR * WC), 0, s,
                       reinterpret_cast<const T*>(a.A), reinterpret_cast<const T*>(a.B), reinterpret_cast<T*>(a.C), g);
    return hipGetLastError();
}

// The output tile: the one with the least matrix-core time on the fullest
// CU.  A CU works through BM x BN x K MACs of a tile at 128 per cycle times
// the share `eff` of that rate which the tile sustains, and the fullest CU
// has ceil(tiles / CUs) of them: large tiles reuse operands best but leave
// CUs idle in the last round.  A CU that holds a single tile has nothing to
// run while that waits (`eff_alone`; 301 x 5632 x 2048 NT: 220 tiles of 64x128
// 86 us, 1760 of 32x32 68).  eff and the shapes inside a tile size are
// measured (K 1000-11008, all layouts): e.g. 2048 x 11008 x 4096 NT 1.39 ms
// on 64x128 (128x128: 1.47, 64x64: 1.46), 500 x 2048 x 5632 NT 99 us on
// 64x64 (32x64: 101, 32x32: 105), 128 x 11008 x 4096 NT 107 us on 32x64
// (32x32: 113, 64x64: 124), 1500^3 NT 68 us on 32x32 (64x64: 80).  With few
// k a 128x128 tile is mostly start and end (32 x 2048 x 2048 x 128, causal:
// 195 us, 64x128 190, 64x64 189).  A causal limit on k makes the tiles'
// work unequal (half of K on average, dispatched longest first), so a CU
// needs at least the longest tile's time: 32 x 2048 x 128 x 2048 150 us on
// 64x64 (64x128 159, 128x128 162, 32x64 227), 8 x 1000 x 64 x 1000 15.5 us
// on 32x64 (64x64 22); the larger two are never ahead there.
template <bool TA, bool TB, bool FUSED, bool TRAP, class T = float>
static hipError_t fast_tile(const GemmArgs& a, hipStream_t s) {
    struct Shape { int bm, bn; double eff, eff_alone, eff_causal; };
    constexpr Shape shapes[5] = {{128, 128, 0.93, 0.75, 0.0}, {64, 128, 0.91, 0.68, 0.0}, {64, 64, 0.87, 0.83, 0.88},
                                 {32, 64, 0.82, 0.70, 0.70}, {32, 32, 0.78, 0.65, 0.65}};
    constexpr bool KC2 = !TA && TB, KC0 = TA && !TB;      // both / neither operand k-contiguous
    const long cus = device_cus();
    const bool causal_k = a.k_causal && (a.k_side == 1 || a.k_side == 2);
    int best = -1;
    double best_cost = 0.0;
    for (int i = causal_k ? 2 : 0; i < 5; i++) {
        const long bm = shapes[i].bm, bn = shapes[i].bn, tm = (a.M + bm - 1) / bm;
        long t = tm * ((a.N + bn - 1) / bn);
        if (TRAP) {
            t = 0;
            for (long r = 0; r < tm; r++) t += trap_cols(a.row0, (int)r, (int)bm, (int)bn, a.N);
        }
        t *= a.batch;
        const double work = (double)bm * bn;
        const double eff = t <= cus ? shapes[i].eff_alone : i == 0 && a.K < 512 ? 0.80 : shapes[i].eff;
        double cost = (double)((t + cus - 1) / cus) * work / eff;
        if (causal_k) cost = std::max(0.5 * t / cus, 1.0) * work / shapes[i].eff_causal;
        if (best < 0 || cost < best_cost) {
            best = i;
            best_cost = cost;
        }
    }
#define RAC_FAST(...) return fast_launch<TA, TB, FUSED, TRAP, __VA_ARGS__, false, T>(a, s)
    // Few k for many outputs: the 64-k tiles would load and stage mostly what
    // is not there (1166 x 3868 x 24 16.3 us on 32x64 x 64 k, here 9.4; x 64
    // 16.7 against 12.9; 679 x 1739 x 24 6.6 against 5.3).  With fewer outputs
    // a CU has a tile or two, and one load of all k is the quicker start: 679
    // x 1739 x 48 with a bias 6.6 us against 7.3, 280 x 7066 x 64 8.3 against
    // 9.0; the two meet near 2^20 outputs at 32 k, 2^21 at 64.
    if (!TRAP && best >= 2 && a.K <= 64 && (long)a.M * a.N * a.batch > (long)std::max(a.K, 32) << 15)
        RAC_FAST(64, 64, 2, 2, 16, 1, 1);
    switch (best) {
    case 0:
        if constexpr (KC2) RAC_FAST(128, 128, 2, 4, 16, 1, 0);
        else if constexpr (KC0) RAC_FAST(128, 128, 2, 4, 32, 1, 0);
        else RAC_FAST(128, 128, 2, 2, 16, 1, 0);
    case 1:
        // A^T B has no 64x128 tile: its 64x64 one, of short K-tiles, runs where
        // the rule finds 64x128 best.  Left out of the rule there instead, the
        // next best lost: 1215 x 6143 x 105 27.1 -> 38.5 us on 32x64, 7333 x
        // 1011 x 444 69.0 -> 81.2, 3989 x 1795 x 136 29.7 -> 42.1 on 32x32
        // (6994 x 7356 x 614 533 -> 517 on 128x128).
        if constexpr (KC0) RAC_FAST(64, 64, 2, 2, 32, 1, 1);
        else RAC_FAST(64, 128, 2, 2, 16, 1, 1);
    case 2:
        if constexpr (KC0) RAC_FAST(64, 64, 2, 2, 32, 1, 1);
        else RAC_FAST(64, 64, 2, 2, 64, 1, 2);
    case 3: RAC_FAST(32, 64, 2, 2, 64, 2, 2);
    default: RAC_FAST(32, 32, 2, 2, 64, 2, 2);
    }
#undef RAC_FAST
}

// At most 16 rows (decode-time linears) or columns: one 16 x 16 block of
// outputs per wave, which runs at the instruction's latency, K x 8 cycles
// for any number of rows up to 16 (1 x 4096 x 4096: 23.4 us, of which 14.5
// that chain).  Four waves side by side, one per SIMD, with the deeper
// K-tile once a CU has more than one such block (1 x 32000 x 4096: 90.1
// against 95.3 us; 1 x 11008 x 4096, 172 blocks: 31.5 against 27.8); pairs
// of waves where those still fit one to a CU (4096 columns: 23.4 against
// 26.9 us; 11008, 344 blocks: 39.6, a second pair shares the first's SIMDs).
template <bool TA, bool TB, bool FUSED, class T = float>
static hipError_t fast_few(const GemmArgs& a, hipStream_t s) {
    const long cus = device_cus();
    const bool rows = a.M <= 16;
    const long n = rows ? a.N : a.M, b4 = (n + 63) / 64 * a.batch, b2 = (n + 31) / 32 * a.batch;
#define RAC_FAST(...) return fast_launch<TA, TB, FUSED, false, __VA_ARGS__, T>(a, s)
    // fewer than 4 rows stored side by side (1 is a vector, read as k-contiguous)
    if constexpr (TA) {
        if (a.M < 4) RAC_FAST(16, 64, 1, 4, 64, 2, 2, true);
    }
    if constexpr (!TB) {
        if (a.N < 4) RAC_FAST(64, 16, 4, 1, 64, 2, 2, true);
    }
    // few k of a transposed A: K-tiles no longer than they are (12 x 300 x 24
    // TN 2.9 us, on 128 k 3.6)
    if constexpr (TA) {
        if (rows && a.K <= 32) RAC_FAST(16, 32, 1, 2, 32, 1, 1, false);
        if (a.K <= 32) RAC_FAST(32, 16, 2, 1, 32, 1, 1, false);
    }
    if (rows) {
        if (b2 <= cus) RAC_FAST(16, 32, 1, 2, 128, 1, 2, false);
        if (b4 <= cus) RAC_FAST(16, 64, 1, 4, 64, 2, 2, false);
        RAC_FAST(16, 64, 1, 4, 128, 1, 2, false);
    }
    if (b2 <= cus) RAC_FAST(32, 16, 2, 1, 128, 1, 2, false);
    if (b4 <= cus) RAC_FAST(64, 16, 4, 1, 64, 2, 2, false);
    RAC_FAST(64, 16, 4, 1, 128, 1, 2, false);
#undef RAC_FAST
}

template <bool TA, bool TB, bool FUSED, class T = float>
static hipError_t fast_shape(const GemmArgs& a, hipStream_t s) {
    if (a.M <= 16 || a.N <= 16) return fast_few<TA, TB, FUSED, T>(a, s);
    return fast_tile<TA, TB, FUSED, false, T>(a, s);
}

hipError_t gemm_fast_half_launch(int dtype, const GemmArgs& g, hipStream_t s) {
    return dtype == 1 ? fast_shape<false, true, true, Bf16>(g, s) : fast_shape<false, true, true, F16>(g, s);
}

hipError_t gemm_fast_launch(int ta, int tb, const GemmArgs& g, hipStream_t s) {
    // one row or column is a vector: as well k-contiguous
    if (g.M == 1) ta = 0;
    if (g.N == 1) tb = 1;
    if (g.fused) return fast_shape<false, true, true>(g, s);                             // NT only
    if (g.sched == 1 || g.sched == 3) return fast_tile<false, true, false, true>(g, s);  // NT only
    if (!ta && !tb) return fast_shape<false, false, false>(g, s);
    if (!ta && tb) return fast_shape<false, true, false>(g, s);
    if (ta && !tb) return fast_shape<true, false, false>(g, s);
    return fast_shape<true, true, false>(g, s);
}

}  // namespace rac

// rac_rowops.hip — row-wise softmax (hyperbolic-CORDIC exp), RMSNorm and
// LayerNorm (CORDIC-vectoring rsqrt) for gfx950.
//
// A row that fits in registers (64 values per lane) is read from HBM exactly
// once, reduced and written once: 1 read + 1 write per element, the HBM
// minimum.  Longer rows take a strided loop that re-reads the row (from L2
// for rows up to a few MB).  RowLayout says which lane holds what: 16-byte
// groups where the row length and the pointers allow it, else single values,
// and a workgroup (4 wave64, a 4-entry LDS exchange) or one wave per row.
//
// Arithmetic follows rac_cpu.c:258-271 (softmax), :548-574 (RMSNorm) and
// :507-546 (LayerNorm) rounding for rounding, except the order of the row
// sums: lane l of 256 adds the float4 groups l, l + 256, ... in order (where a
// row cannot be read in float4 groups, the elements l, l + 256, ...), lanes
// combine by a wave64 XOR butterfly (offsets 32 .. 1) and the four wave
// partials in order, instead of one left-to-right sum (differences O(1e-7)
// relative).  That order is fixed, whichever layout or loop ran, so results
// do not depend on scheduling and a CPU model of it matches bit for bit.
#include <hip/hip_runtime.h>
#include <atomic>
#include <type_traits>
#include "rac_math.hpp"
#include "rac_internal.hpp"
#include "rac_rowred.hpp"

namespace rac {

template <int NITER>
__device__ __forceinline__ float exp_n(float x, int iters, float khinv) {
    if constexpr (NITER > 0) return exp_cordic<NITER>(x, khinv);
    else return exp_cordic_rt(x, iters, khinv);
}

// ── softmax ──────────────────────────────────────────────────────────────

// Attention masking of score x at (query position t, key column j), in the
// order of rac_cpu.c:668-670: causal sets -inf above the diagonal, then the
// additive mask is added (mask_ld set by the dispatcher).
__device__ __forceinline__ float mask_score(float x, long t, long j, const SoftmaxMask& mk) {
    if (mk.causal && j > t) x = -__builtin_inff();
    if (mk.mask) x += mk.mask[t * mk.mask_ld + j];
    return x;
}

// 1/sum, or 0 for a non-positive sum when the guard of rac_cpu.c:687 is on.
__device__ __forceinline__ float inv_sum(float s, int zero_guard) {
    return (zero_guard && !(s > 0.0f)) ? 0.0f : 1.0f / s;
}

// Exps of the E = 4*VPT row elements a lane holds, in the step-major form
// (the elements of a group advance one step at a time: independent chains
// interleave and constants are shared); bit-identical to one exp_cordic call
// per element.  Step counts known only at run time too: one element after the
// other, a wave's long lane of them was slower than four waves' short ones
// (1024 x 600, 12 steps: 6.9 us before rows to a wave, 9.4 with them, now
// 6.9; 4096 x 500 10.1 -> 6.4).
template <int NITER, int E, int OPT = kExpFull>
__device__ __forceinline__ void exp_lane(float* v, int iters, float khinv) {
    if constexpr (NITER > 0) {
        constexpr int G = E < 16 ? E : 16;
#pragma unroll
        for (int b = 0; b < E; b += G) exp_cordic_vec<NITER, G, OPT>(v + b, khinv);
    } else {
        constexpr int G = E < 4 ? E : E % 8 ? 4 : 8;
#pragma unroll
        for (int b = 0; b < E; b += G) exp_cordic_rt_vec<G>(v + b, iters, khinv);
    }
}

// Which elements of a row a lane holds: units of VEC values (4: 16-byte
// groups; 1: single values, for row lengths that are no multiple of 4 and
// unaligned pointers), unit l + LANES i for lane l of the W waves of the row.
//
// W = 4 is the order of the sums.  W = 1 (rows of up to 1024) has the same
// bits: the units l, l + 64, l + 128, l + 192 that its lane l holds are those
// of lane l of each of the four waves, so it keeps four sums apart, runs the
// four butterflies side by side and adds them in order.  It needs no barriers
// and leaves no wave without a row.
// VPT counts the lane's values in fours, 0 is a single one (row_values): a
// ragged row of up to LANES values.  Held in four, three of them empty, it
// took longer than in the strided loop before (900 x 130, 24 steps, 4.08 ->
// 4.43 us; masked, three of 33 x 33, 3.8 -> 4.2), now 3.5 and 3.5.
constexpr int row_values(int vpt) { return vpt ? 4 * vpt : 1; }
template <int VEC_, int W_>
struct RowLayout {
    static constexpr int VEC = VEC_, W = W_, LANES = 64 * W_;
    static constexpr int sums(int E) { return W == 4 ? 1 : E / VEC < 4 ? E / VEC : 4; }
    static __device__ __forceinline__ int lane() { return W == 4 ? threadIdx.x : threadIdx.x & 63; }
    static __device__ __forceinline__ int unit(int i) { return lane() + LANES * i; }
    static __device__ __forceinline__ int index(int e) { return VEC * unit(e / VEC) + e % VEC; }
    static constexpr int sum_of(int e) { return W == 4 ? 0 : (e / VEC) % 4; }
    // the row this thread works on (W = 1: four to a workgroup)
    static __device__ __forceinline__ long row() {
        return W == 4 ? (long)blockIdx.x : 4L * blockIdx.x + threadIdx.x / 64;
    }
    static dim3 grid(long rows) { return dim3((unsigned)(W == 4 ? rows : (rows + 3) / 4)); }
    // the row's sum of every lane's partial sums s[sums(E)]
    template <int S, bool TRAIL = false, bool LDS_ONLY = false>
    static __device__ __forceinline__ float total(const float* s, float* red) {
        if constexpr (W == 4) {
            return block_sum<TRAIL, LDS_ONLY>(s[0], red);
        } else {
            float r = wave_sum(s[0]);
#pragma unroll
            for (int i = 1; i < S; i++) r += wave_sum(s[i]);
            return r;
        }
    }
};

// Attention rows: with a causal limit or a mask, or (kGuarded) neither, only
// the zero guard of the sum.  The latter have no runs of -inf to look for,
// which took 8 heads of 2048 from 52.0 to 54.5 us, 49.0 without it; past
// 4096 the exps in the search's groups of 8 hold fewer registers and win all
// the same (1 x 6000 57.8 us against 61.0, 1 x 9000 145 against 209).
// Under a mask that search gains where the mask holds -inf (8 x 512 10.2 ->
// 7.9 us, 8 x 2048 78.1 -> 75.5) and costs where all of it is finite (8 x 2048
// 80.3 -> 86.4, 16 x 1024 43.4 -> 45.5).
constexpr int kGuarded = 1, kMasked = 2;

// Softmax of the row a workgroup (or wave) holds in registers, E values per
// lane, -inf past the row end, whose exp is +0, so the max, the lane sums
// (s + 0 == s) and the outputs are those of the elements that exist.  On
// return v holds the outputs.  t is the row's query position (masked rows
// only).
// First stage: masking (masked rows) and the lane's maximum.
template <class L, int VPT, int MASKED, bool FULL>
__device__ __forceinline__ float softmax_lane_max(float* v, long n, long t, const SoftmaxMask& mk) {
    if constexpr (MASKED == kMasked) {
#pragma unroll
        for (int i = 0; i < row_values(VPT) / L::VEC; i++) {
            const long j = (long)L::VEC * L::unit(i);
            if (FULL || j < n) {
#pragma unroll
                for (int c = 0; c < L::VEC; c++) v[L::VEC * i + c] = mask_score(v[L::VEC * i + c], t, j + c, mk);
            }
        }
    }
    float m = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < VPT; i++)
        m = fmaxf(fmaxf(fmaxf(m, v[4 * i]), fmaxf(v[4 * i + 1], v[4 * i + 2])), v[4 * i + 3]);
    if constexpr (VPT == 0) m = fmaxf(m, v[0]);
    return m;
}

// The lane's first zero (zero_key): a lane's values run in index order.
template <class L, int VPT>
__device__ __forceinline__ uint32_t lane_first_zero(const float* v) {
    uint32_t key = ~0u;
#pragma unroll
    for (int e = row_values(VPT) - 1; e >= 0; e--)
        if (v[e] == 0.0f) key = zero_key<uint32_t>(L::index(e), v[e]);
    return key;
}

// The lane's partial sums of its values.
template <class L, int E>
__device__ __forceinline__ void lane_sums(const float* v, float* s) {
#pragma unroll
    for (int i = 0; i < L::sums(E); i++) s[i] = 0.0f;
#pragma unroll
    for (int e = 0; e < E; e++) s[L::sum_of(e)] += v[e];
}

// Exps of the lane's values against the row maximum m (masked rows, and rows
// whose step count is known only at run time).
template <int VPT, int NITER, int MASKED>
__device__ __forceinline__ void softmax_lane_exps(float* v, float m, int iters, float khinv) {
    constexpr int E = row_values(VPT);
#pragma unroll
    for (int e = 0; e < E; e++) v[e] = v[e] - m;
    if constexpr (MASKED == kMasked) {
        // the exps of -inf are +0: a wave skips the runs of its values that
        // are -inf in every lane (past the diagonal of a causal row)
        constexpr int G = E < 4 ? E : E % 8 || E == 8 ? 4 : 8;
#pragma unroll
        for (int b = 0; b < E; b += G) {
            bool some = false;
#pragma unroll
            for (int e = 0; e < G; e++) some |= v[b + e] != -__builtin_inff();
            if (__any(some)) {
                exp_lane<NITER, G>(v + b, iters, khinv);
            } else {
#pragma unroll
                for (int e = 0; e < G; e++) v[b + e] = 0.0f;
            }
        }
    } else {
        exp_lane<NITER, E>(v, iters, khinv);
    }
}

// Unmasked rows with a compile-time step count.  Every x - max is <= 0 or
// NaN, and a NaN anywhere, or a maximum of +-inf, makes the reference's row
// sum NaN and with it every output (rac_cpu.c:258-271).  So:
//  - the row maximum is the NaN-propagating IEEE maximum (v_maximum3, no
//    canonicalisation of the loaded values; -0 < +0 as for v_max_f32, so
//    the maximum and every x - max equal the general path's), and a
//    non-finite maximum forces the row sum to NaN instead of a per-element
//    NaN test;
//  - the exps skip the sign-dependent rounding bias (kExpNonPos);
//  - when every x - max of the wave is >= -86 (then k >= -124), the exp's
//    (p / K_h) 2^k is p * (1/K_h 2^k) with the scale built in the exponent
//    field: one rounding of the same exact product, every intermediate
//    normal, so the bits of ldexp(p / K_h, k); otherwise ldexp and the
//    k <= -127 flush.
// Bit-identical to softmax_lane_exps<VPT, NITER, false> with kExpFlush |
// kExpNonPos exps and a NaN pass; ~5% fewer VALU instructions per element.
struct RowExtent {
    float max;   // row maximum (every lane)
    float min;   // the lane's minimum
};

// row_lds: the row in LDS in the same layout (the prefetching kernel), read
// instead of v for the rare zero-maximum scan, so that scan holds no
// registers of its own; null: scan v.
template <class L, int VPT, bool LDS_ONLY>
__device__ __forceinline__ RowExtent unmasked_row_extent(const float* v, float* red, uint32_t* zred,
                                                         const float* row_lds = nullptr) {
    constexpr int E = row_values(VPT);
    float mx = v[0], mn = v[0];
#pragma unroll
    for (int e = 1; e < E; e++) {
        mx = maximum(mx, v[e]);
        mn = fminf(mn, v[e]);
    }
    if constexpr (L::W == 1) mx = wave_maximum(mx);
    else mx = block_maximum<false, LDS_ONLY>(mx, red);
    if (mx == 0.0f) {
        uint32_t key = ~0u;
        if (row_lds) {
            for (int e = 0; e < E && key == ~0u; e++) {
                const int idx = L::index(e);
                if (row_lds[idx] == 0.0f) key = zero_key<uint32_t>(idx, row_lds[idx]);
            }
        } else {
            key = lane_first_zero<L, VPT>(v);
        }
        if constexpr (L::W == 1) mx = wave_first_zero_max(key);
        else mx = first_zero_max<LDS_ONLY>(key, zred);
    }
    return {mx, mn};
}

template <int N, int G>
__device__ __forceinline__ void unmasked_exp_group(float* v, float khinv, bool fused) {
    int k[G];
    float p[G], z[G];
#pragma unroll
    for (int e = 0; e < G; e++) {
        k[e] = cvt_i32_sat(__builtin_fmaf(v[e], kInvLn2, -0.5f));
        z[e] = __builtin_fmaf(-(float)k[e], kLn2, v[e]);
        p[e] = 1.0f;
    }
    HypStepV<N, 0, G>::run(p, z);
    if (fused) {
#pragma unroll
        for (int e = 0; e < G; e++) v[e] = p[e] * as_f(as_u(khinv) + ((uint32_t)k[e] << 23));
    } else {
#pragma unroll
        for (int e = 0; e < G; e++) {
            const float res = __builtin_ldexpf(p[e] * khinv, k[e]);
            v[e] = (k[e] <= -127) ? 0.0f : res;
        }
    }
}

template <int NITER, int E>
__device__ __forceinline__ void unmasked_lane_exps(float* v, RowExtent r, float khinv) {
    const bool fused = __all((r.min - r.max) >= -86.0f);
#pragma unroll
    for (int e = 0; e < E; e++) v[e] = v[e] - r.max;
    constexpr int G = E < 16 ? E : 16;
#pragma unroll
    for (int b = 0; b + G <= E; b += G) unmasked_exp_group<NITER, G>(v + b, khinv, fused);
}
__device__ __forceinline__ float unmasked_lane_sum(float s, RowExtent r) {
    if (!(__builtin_fabsf(r.max) < __builtin_inff())) s = __builtin_nanf("");
    return s;
}

// red: 2 kRowWaves floats (max and sum partials apart, so neither reduction
// needs a trailing barrier; a kernel handles one row per workgroup).
template <class L, int VPT, int NITER, int MASKED, bool FULL>
__device__ __forceinline__ void softmax_row_regs(float* v, long n, long t, int iters, float khinv,
                                                 const SoftmaxMask& mk, float* red, uint32_t* zred) {
    constexpr int E = row_values(VPT), S = L::sums(E);
    float s[S], inv;
    if constexpr (!MASKED && NITER > 0) {
        const RowExtent r = unmasked_row_extent<L, VPT, false>(v, red, zred);
        unmasked_lane_exps<NITER, E>(v, r, khinv);
        lane_sums<L, E>(v, s);
        s[0] = unmasked_lane_sum(s[0], r);
        inv = inv_sum(L::template total<S>(s, red + kRowWaves), 0);
    } else {
        float m = softmax_lane_max<L, VPT, MASKED, FULL>(v, n, t, mk);
        if constexpr (L::W == 1) {
            m = wave_max(m);
            if (m == 0.0f) m = wave_first_zero_max(lane_first_zero<L, VPT>(v));
        } else {
            m = block_max<false>(m, red);
            if (m == 0.0f) m = first_zero_max<false>(lane_first_zero<L, VPT>(v), zred);
        }
        softmax_lane_exps<VPT, NITER, MASKED>(v, m, iters, khinv);
        lane_sums<L, E>(v, s);
        inv = inv_sum(L::template total<S>(s, red + kRowWaves), MASKED ? mk.zero_guard : 0);
    }
#pragma unroll
    for (int e = 0; e < E; e++) v[e] = v[e] * inv;
}

// last: the last column needed (causal rows: the query position; the mask
// puts -inf past it whatever was there).  pad: in place of what is not there.
template <class L, int VPT, bool FULL, bool MASKED = false>
__device__ __forceinline__ void load_row_regs(const float* xr, long n, float* v, float pad, long last = 0) {
#pragma unroll
    for (int i = 0; i < row_values(VPT) / L::VEC; i++) {
        const long j = (long)L::VEC * L::unit(i);
        const bool in = (FULL || j < n) && (!MASKED || j <= last);
        if constexpr (L::VEC == 4) {
            float4 t = make_float4(pad, pad, pad, pad);
            if (in) t = ld4_stream(reinterpret_cast<const float4*>(xr + j));
            v[4 * i] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w;
        } else {
            v[i] = in ? xr[j] : pad;
        }
    }
}

template <int VEC>
__device__ __forceinline__ void store_unit(float* y, const float* v) {
    if constexpr (VEC == 4) st4_stream(reinterpret_cast<float4*>(y), make_float4(v[0], v[1], v[2], v[3]));
    else *y = *v;
}
template <class L, int VPT, bool FULL>
__device__ __forceinline__ void store_row_regs(float* yr, long n, const float* v) {
#pragma unroll
    for (int i = 0; i < row_values(VPT) / L::VEC; i++) {
        const long j = (long)L::VEC * L::unit(i);
        if (FULL || j < n) store_unit<L::VEC>(yr + j, v + L::VEC * i);
    }
}

// Rows held in registers: read once, reduced, exponentiated and written once.
// FULL: n == 4 LANES VPT exactly, so no lane needs a bounds check.
template <class L, int VPT, int NITER, int MASKED, bool FULL>
__global__ __launch_bounds__(kRowThreads) void softmax_reg_kernel(
    const float* x, float* y, long rows, long n, int iters, float khinv,
    SoftmaxMask mk)
{
    __shared__ float red[2 * kRowWaves];
    __shared__ uint32_t zred[kRowWaves];
    const long row = L::row();
    if (L::W == 1 && row >= rows) return;
    float v[row_values(VPT)];
    const long t = MASKED ? mk.row0 + row % mk.seq : 0;
    load_row_regs<L, VPT, FULL, MASKED == kMasked>(x + row * n, n, v, -__builtin_inff(), MASKED && mk.causal ? t : n);
    softmax_row_regs<L, VPT, NITER, MASKED, FULL>(v, n, t, iters, khinv, mk, red, zred);
    store_row_regs<L, VPT, FULL>(y + row * n, n, v);
}

// Unmasked rows of exactly 1024 VPT floats, persistent: workgroup g takes
// rows g, g + G, g + 2G, ... (G = gridDim.x).  While a row's exps run, the
// next row is already on its way from HBM into LDS (global_load_lds, which
// holds no VGPRs), so each workgroup keeps one row of loads in flight
// through its whole lifetime instead of waiting for its row at start-up.
// The row reductions use LDS-only barriers (lds_barrier): the previous
// row's stores stay in flight across them; the barrier of the row sum
// waits for the prefetch (an LDS write), which has had the exps to land.
// Same arithmetic as softmax_reg_kernel<RowLayout<4, 4>, VPT, ..>, so the
// same bits.  Used where the exps are short (n = 8): at 16 and 24 steps the
// one-row-per-workgroup kernel is faster (measured on 4096 x 4096: n = 8
// 23.6 -> 22.2 us; n = 16 25.0 against 26.3, n = 24 31.1 against 32.2).
template <int VPT, int NITER>
__global__ __launch_bounds__(kRowThreads, 6) void softmax_prefetch_kernel(
    const float* x, float* y, long rows, float khinv)
{
    using L = RowLayout<4, 4>;
    constexpr long n = 1024L * VPT;
    constexpr int E = 4 * VPT;
    __shared__ __attribute__((aligned(16))) float row_lds[n];
    __shared__ float red[2 * kRowWaves];
    __shared__ uint32_t zred[kRowWaves];
    const int t = threadIdx.x, w = t >> 6;
    const long G = gridDim.x;
    long row = blockIdx.x;
    // lane t of wave w copies the float4 groups t + 256 i of row r to the
    // same group index in row_lds; each instruction fills 1 KB at the
    // wave's base (64 lanes x 16 bytes)
    auto prefetch = [&](long r) {
        const float* src = x + r * n;
#pragma unroll
        for (int i = 0; i < VPT; i++)
            __builtin_amdgcn_global_load_lds(src + 4 * (t + kRowThreads * i),
                                             (__attribute__((address_space(3))) void*)(row_lds + 4 * (kRowThreads * i + 64 * w)),
                                             16, 0, 0);
    };
    prefetch(row);
    lds_barrier();
    for (; row < rows; row += G) {
        float v[E];
#pragma unroll
        for (int i = 0; i < VPT; i++) {
            const float4 q = *reinterpret_cast<const float4*>(row_lds + 4 * (t + kRowThreads * i));
            v[4 * i] = q.x; v[4 * i + 1] = q.y; v[4 * i + 2] = q.z; v[4 * i + 3] = q.w;
        }
        // every wave has read row_lds (its lane maximum needs the values)
        // once the barrier inside block_maximum is passed
        const RowExtent r = unmasked_row_extent<L, VPT, true>(v, red, zred, row_lds);
        if (row + G < rows) prefetch(row + G);
        unmasked_lane_exps<NITER, E>(v, r, khinv);
        float s;
        lane_sums<L, E>(v, &s);
        s = unmasked_lane_sum(s, r);
        // the prefetch has landed before the barrier below (the LDS fence
        // waits for it too; this states it, and the operand keeps the wait
        // after the exps)
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(s));
        s = L::total<1, false, true>(&s, red + kRowWaves);
        const float inv = inv_sum(s, 0);
#pragma unroll
        for (int e = 0; e < E; e++) v[e] = v[e] * inv;
        store_row_regs<L, VPT, true>(y + row * n, n, v);
    }
}

// Workgroups of softmax_prefetch_kernel<VPT, NITER> resident per CU.
template <int VPT, int NITER>
static int softmax_prefetch_occupancy() {
    static std::atomic<int> cached{0};
    int v = cached.load(std::memory_order_relaxed);
    if (v == 0) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, softmax_prefetch_kernel<VPT, NITER>, kRowThreads, 0) !=
                hipSuccess || v < 1) {
            (void)hipGetLastError();
            v = 1;
        }
        cached.store(v, std::memory_order_relaxed);
    }
    return v;
}

template <int NITER, bool MASKED>
__global__ __launch_bounds__(kRowThreads) void softmax_loop_kernel(
    const float* x, float* y, long n, int iters, float khinv,
    SoftmaxMask mk)
{
    __shared__ float red[kRowWaves];
    const long row = blockIdx.x;
    const long t = MASKED ? mk.row0 + row % mk.seq : 0;
    const float* xr = x + row * n;
    float* yr = y + row * n;
    float m = -__builtin_inff();
    for (long i = threadIdx.x; i < n; i += kRowThreads) {
        float v = xr[i];
        if constexpr (MASKED) v = mask_score(v, t, i, mk);
        m = fmaxf(m, v);
    }
    m = block_max(m, red);
    if (m == 0.0f) {
        __shared__ uint64_t zred[kRowWaves];
        uint64_t key = ~0ull;
        for (long i = threadIdx.x; i < n; i += kRowThreads) {
            float v = xr[i];
            if constexpr (MASKED) v = mask_score(v, t, i, mk);
            if (v == 0.0f) {
                key = zero_key<uint64_t>(i, v);
                break;
            }
        }
        m = first_zero_max<false>(key, zred);
    }
    float s = 0.0f;
    for (long i = threadIdx.x; i < n; i += kRowThreads) {
        float v = xr[i];
        if constexpr (MASKED) v = mask_score(v, t, i, mk);
        const float e = exp_n<NITER>(v - m, iters, khinv);
        yr[i] = e;
        s += e;
    }
    s = block_sum(s, red);
    const float inv = inv_sum(s, MASKED ? mk.zero_guard : 0);
    for (long i = threadIdx.x; i < n; i += kRowThreads) yr[i] = yr[i] * inv;
}

// Workgroups per CU of the unmasked register kernel with compile-time steps.
// Its leaner arithmetic needs fewer VGPRs than the general form (59 / 82 /
// 113 at VPT 4 / 8 / 16 against 74 / 120 / 137), which would raise
// residency from 6 / 4 / 3 to 8 / 5 / 4 workgroups per CU.  At VPT 4 that
// was measured slower (softmax 4096 x 4096, n = 16: 8 per CU ran 29.2 µs
// median against 25.4 at 6 on one box, 0.97x on another; 6 per CU with the
// lean arithmetic: 0.95-0.99x of the general form), so the launch keeps the
// general form's residency by requesting unused dynamic LDS: 160 KB / cap
// minus 1 KB lets exactly `cap` workgroups share a CU's 160 KB.
constexpr long kCuLdsBytes = 160L * 1024;
constexpr int unmasked_reg_cap(int vpt) { return vpt <= 2 ? 0 : vpt == 4 ? 6 : vpt == 8 ? 4 : 3; }

template <class L, int VPT, int NITER, int MASKED>
static void softmax_reg_launch(hipStream_t s, const float* x, float* y, long rows, long n, int iters,
                               float khinv, const SoftmaxMask& mk) {
    constexpr int cap = (!MASKED && NITER > 0 && L::W == 4) ? unmasked_reg_cap(VPT) : 0;
    constexpr size_t lds = cap ? (size_t)(kCuLdsBytes / cap - 1024) : 0;
    if constexpr (L::VEC == 4) {
        if (n == 4L * VPT * L::LANES) {
            hipLaunchKernelGGL((softmax_reg_kernel<L, VPT, NITER, MASKED, true>), L::grid(rows), dim3(kRowThreads),
                               lds, s, x, y, rows, n, iters, khinv, mk);
            return;
        }
    }
    hipLaunchKernelGGL((softmax_reg_kernel<L, VPT, NITER, MASKED, false>), L::grid(rows), dim3(kRowThreads), lds, s,
                       x, y, rows, n, iters, khinv, mk);
}

// Calls f(layout, VPT) for the layout of rows of n values (vec: 16-byte
// groups) and returns true, or returns false where a row does not fit.
// A wave takes a row of up to 768 once there are 4 rows per CU (fewer rows
// need the four waves each): softmax n = 16 against a workgroup per row
// 16000 x 500 25.6 -> 15.1 us, 8192 x 100 13.7 -> 5.6, 4096 x 700 9.3 -> 7.7,
// 1024 x 256 4.0 -> 2.9; RMSNorm 16000 x 500 19.6 -> 12.7, LayerNorm
// 22.4 -> 13.1.  Past 768 its 16 values per lane leave too few waves in
// flight until there are `wide` rows per CU (softmax 32: 4096 x 1000
// 9.7 against 9.9, 16000 x 1000 29.3 against 26.5; the norms 16:
// RMSNorm 2048 x 1000 4.95 against 5.25, 4096 x 1000 8.9 against 6.9).
// Rows that cannot be read in 16-byte groups (the strided loop before):
// softmax 4096 x 4095 69.5 -> 29.3 us (4096 x 4096: 25.1), RMSNorm 40.4 ->
// 28.3, LayerNorm 49.3 -> 28.9.
template <class F>
static bool with_row_layout(long rows, long n, bool vec, long wide, F f) {
    const long per_cu = rows / device_cus();
    auto at = [&](auto vec_c) {
        constexpr int VEC = decltype(vec_c)::value;
        using L1 = RowLayout<VEC, 1>;
        using L4 = RowLayout<VEC, 4>;
#define RAC_VPT(L, k) f(L(), std::integral_constant<int, (k) == 0 && VEC == 4 ? 1 : (k)>())
        if (n <= 1024 && per_cu >= (n <= 768 ? 4 : wide)) {
            if (VEC == 1 && n <= 64) RAC_VPT(L1, 0);
            else if (n <= 256) RAC_VPT(L1, 1);
            else if (n <= 512) RAC_VPT(L1, 2);
            else if (n <= 768) RAC_VPT(L1, 3);
            else RAC_VPT(L1, 4);
        } else if (VEC == 1 && n <= 256) RAC_VPT(L4, 0);
        else if (n <= 1024) RAC_VPT(L4, 1);
        else if (n <= 2048) RAC_VPT(L4, 2);
        else if (n <= 4096) RAC_VPT(L4, 4);
        else if (n <= 8192) RAC_VPT(L4, 8);
        else if (n <= 16384) RAC_VPT(L4, 16);
        else return false;
#undef RAC_VPT
        return true;
    };
    return vec ? at(std::integral_constant<int, 4>()) : at(std::integral_constant<int, 1>());
}

template <int NITER, int MASKED>
static hipError_t softmax_dispatch(const float* x, float* y, long rows, long n, int iters,
                                   float khinv, hipStream_t s, const SoftmaxMask& mk) {
    const bool vec_ok = (n % 4 == 0) && ((reinterpret_cast<uintptr_t>(x) & 15) == 0) &&
                        ((reinterpret_cast<uintptr_t>(y) & 15) == 0);
    dim3 grid((unsigned)rows), block(kRowThreads);
    if constexpr (!MASKED && NITER > 0 && NITER <= 8) {
        // short exps: the persistent prefetching kernel, where every
        // workgroup gets at least two rows
        auto prefetch_launch = [&](auto vpt) -> bool {
            constexpr int VPT = decltype(vpt)::value;
            if (n != 1024L * VPT) return false;
            const long g = (long)softmax_prefetch_occupancy<VPT, NITER>() * device_cus();
            if (rows < 2 * g) return false;
            hipLaunchKernelGGL((softmax_prefetch_kernel<VPT, NITER>), dim3((unsigned)g), block, 0, s, x, y, rows,
                               khinv);
            return true;
        };
        if (vec_ok && (prefetch_launch(std::integral_constant<int, 1>{}) ||
                       prefetch_launch(std::integral_constant<int, 2>{}) ||
                       prefetch_launch(std::integral_constant<int, 4>{})))
            return hipGetLastError();
    }
    if (!with_row_layout(rows, n, vec_ok, 32, [&](auto l, auto vpt) {
            if constexpr (MASKED != kGuarded || decltype(vpt)::value <= 4)
                softmax_reg_launch<decltype(l), decltype(vpt)::value, NITER, MASKED>(s, x, y, rows, n, iters, khinv, mk);
        }))
        hipLaunchKernelGGL((softmax_loop_kernel<NITER, MASKED != 0>), grid, block, 0, s, x, y, n, iters, khinv, mk);
    return hipGetLastError();
}

template <int NITER>
static hipError_t softmax_mask_dispatch(const float* x, float* y, long rows, long n, int iters,
                                        float khinv, hipStream_t s, const SoftmaxMask& mk) {
    if (mk.mask || mk.causal || mk.zero_guard) {
        SoftmaxMask m2 = mk;
        if (m2.seq <= 0) m2.seq = n;   // square scores: row length = sequence length
        if (m2.mask_ld <= 0) m2.mask_ld = n;
        if (mk.mask || mk.causal || n > 4096)
            return softmax_dispatch<NITER, kMasked>(x, y, rows, n, iters, khinv, s, m2);
        return softmax_dispatch<NITER, kGuarded>(x, y, rows, n, iters, khinv, s, m2);
    }
    return softmax_dispatch<NITER, 0>(x, y, rows, n, iters, khinv, s, mk);
}

hipError_t softmax_launch(const float* x, float* y, long rows, long n, int iters, hipStream_t s,
                          const SoftmaxMask& mk) {
    iters = clamp_iters(iters);
    const float khinv = host_consts().exp_khinv[iters];
    switch (iters) {
        case 8: return softmax_mask_dispatch<8>(x, y, rows, n, iters, khinv, s, mk);
        case 16: return softmax_mask_dispatch<16>(x, y, rows, n, iters, khinv, s, mk);
        case 24: return softmax_mask_dispatch<24>(x, y, rows, n, iters, khinv, s, mk);
        default: return softmax_mask_dispatch<0>(x, y, rows, n, iters, khinv, s, mk);
    }
}

// ── RMSNorm / LayerNorm ──────────────────────────────────────────────────

// The VEC values of a weight row at column j (gamma null: 1; beta null: 0).
template <int VEC>
__device__ __forceinline__ void load_weights(const float* w, long j, float none, float* v) {
    if constexpr (VEC == 4) {
        const float4 q = w ? *reinterpret_cast<const float4*>(w + j) : make_float4(none, none, none, none);
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else {
        v[0] = w ? w[j] : none;
    }
}

// Rows of 64 values a lane store each unit as it is done, which frees its
// registers; shorter ones all at the end: behind a store in between, the next
// weights' load waits for it (8192 x 700 7.7 us against 8.5; but wide 1000 x
// 15001 47.1 stored at the end, 43.0 so).
constexpr bool wide_row(int vpt) { return vpt >= 16; }

template <class L, int VPT>
__global__ __launch_bounds__(kRowThreads) void rmsnorm_reg_kernel(
    const float* __restrict__ x, float* __restrict__ y, const float* __restrict__ gamma,
    float eps, long rows, long d, float khinv16)
{
    constexpr int E = row_values(VPT), S = L::sums(E);
    constexpr bool kWide = wide_row(VPT);
    __shared__ float red[kRowWaves];
    const long row = L::row();
    if (L::W == 1 && row >= rows) return;
    float v[E], ss[S] = {};
    load_row_regs<L, VPT, false>(x + row * d, d, v, 0.0f);
#pragma unroll
    for (int e = 0; e < E; e++) ss[L::sum_of(e)] = __builtin_fmaf(v[e], v[e], ss[L::sum_of(e)]);
    const float ms = L::template total<S, kWide>(ss, red) / (float)d;
    const float inv = rsqrt_cordic(ms + eps, khinv16);
#pragma unroll
    for (int i = 0; i < E / L::VEC; i++) {
        const long j = (long)L::VEC * L::unit(i);
        if (j < d) {
            float g[L::VEC];
            load_weights<L::VEC>(gamma, j, 1.0f, g);
#pragma unroll
            for (int c = 0; c < L::VEC; c++) v[L::VEC * i + c] = v[L::VEC * i + c] * inv * g[c];
            if constexpr (kWide) store_unit<L::VEC>(y + row * d + j, v + L::VEC * i);
        }
    }
    if constexpr (!kWide) store_row_regs<L, VPT, false>(y + row * d, d, v);
}

__global__ __launch_bounds__(kRowThreads) void rmsnorm_loop_kernel(
    const float* __restrict__ x, float* __restrict__ y, const float* __restrict__ gamma,
    float eps, long d, float khinv16)
{
    __shared__ float red[kRowWaves];
    const long row = blockIdx.x;
    const float* xr = x + row * d;
    float* yr = y + row * d;
    float ss = 0.0f;
    for (long i = threadIdx.x; i < d; i += kRowThreads) ss = __builtin_fmaf(xr[i], xr[i], ss);
    const float ms = block_sum(ss, red) / (float)d;
    const float inv = rsqrt_cordic(ms + eps, khinv16);
    for (long i = threadIdx.x; i < d; i += kRowThreads) {
        const float g = gamma ? gamma[i] : 1.0f;
        yr[i] = xr[i] * inv * g;
    }
}

template <class L, int VPT>
__global__ __launch_bounds__(kRowThreads) void layernorm_reg_kernel(
    const float* __restrict__ x, float* __restrict__ y, const float* __restrict__ gamma,
    const float* __restrict__ beta, float eps, long rows, long d, float khinv16)
{
    constexpr int E = row_values(VPT), S = L::sums(E);
    constexpr bool kWide = wide_row(VPT);
    __shared__ float red[2 * kRowWaves];
    const long row = L::row();
    if (L::W == 1 && row >= rows) return;
    float v[E], sm[S], sv[S] = {};
    load_row_regs<L, VPT, false>(x + row * d, d, v, 0.0f);
    lane_sums<L, E>(v, sm);
    const float mean = L::template total<S>(sm, red) / (float)d;
    // one bounds check a unit: one for each value cost a wide row 34 registers
    // and a wave per SIMD (1000 x 16384 28.0 us, 21.2 so)
#pragma unroll
    for (int i = 0; i < E / L::VEC; i++) {
        if ((long)L::VEC * L::unit(i) < d) {
#pragma unroll
            for (int e = L::VEC * i; e < L::VEC * (i + 1); e++) {
                const float z = v[e] - mean;
                sv[L::sum_of(e)] = __builtin_fmaf(z, z, sv[L::sum_of(e)]);
            }
        }
    }
    const float var = L::template total<S>(sv, red + kRowWaves) / (float)d;
    const float inv = rsqrt_cordic(var + eps, khinv16);
#pragma unroll
    for (int i = 0; i < E / L::VEC; i++) {
        const long j = (long)L::VEC * L::unit(i);
        if (j < d) {
            float g[L::VEC], b[L::VEC];
            load_weights<L::VEC>(gamma, j, 1.0f, g);
            load_weights<L::VEC>(beta, j, 0.0f, b);
#pragma unroll
            for (int c = 0; c < L::VEC; c++) {
                float& o = v[L::VEC * i + c];
                o = __builtin_fmaf(g[c], (o - mean) * inv, b[c]);
            }
            if constexpr (kWide) store_unit<L::VEC>(y + row * d + j, v + L::VEC * i);
        }
    }
    if constexpr (!kWide) store_row_regs<L, VPT, false>(y + row * d, d, v);
}

__global__ __launch_bounds__(kRowThreads) void layernorm_loop_kernel(
    const float* __restrict__ x, float* __restrict__ y, const float* __restrict__ gamma,
    const float* __restrict__ beta, float eps, long d, float khinv16)
{
    __shared__ float red[kRowWaves];
    const long row = blockIdx.x;
    const float* xr = x + row * d;
    float* yr = y + row * d;
    float sm = 0.0f;
    for (long i = threadIdx.x; i < d; i += kRowThreads) sm += xr[i];
    const float mean = block_sum(sm, red) / (float)d;
    float sv = 0.0f;
    for (long i = threadIdx.x; i < d; i += kRowThreads) {
        const float z = xr[i] - mean;
        sv = __builtin_fmaf(z, z, sv);
    }
    const float var = block_sum(sv, red) / (float)d;
    const float inv = rsqrt_cordic(var + eps, khinv16);
    for (long i = threadIdx.x; i < d; i += kRowThreads) {
        const float g = gamma ? gamma[i] : 1.0f;
        const float b = beta ? beta[i] : 0.0f;
        yr[i] = __builtin_fmaf(g, (xr[i] - mean) * inv, b);
    }
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

hipError_t rmsnorm_launch(const float* x, float* y, const float* gamma, float eps,
                          long rows, long d, hipStream_t s) {
    const float k = host_consts().rsqrt_khinv;
    const bool vec_ok = (d % 4 == 0) && aligned16(x) && aligned16(y) && (!gamma || aligned16(gamma));
    if (!with_row_layout(rows, d, vec_ok, 16, [&](auto l, auto vpt) {
            using L = decltype(l);
            hipLaunchKernelGGL((rmsnorm_reg_kernel<L, decltype(vpt)::value>), L::grid(rows), dim3(kRowThreads), 0, s,
                               x, y, gamma, eps, rows, d, k);
        }))
        hipLaunchKernelGGL(rmsnorm_loop_kernel, dim3((unsigned)rows), dim3(kRowThreads), 0, s, x, y, gamma, eps, d, k);
    return hipGetLastError();
}

hipError_t layernorm_launch(const float* x, float* y, const float* gamma, const float* beta,
                            float eps, long rows, long d, hipStream_t s) {
    const float k = host_consts().rsqrt_khinv;
    const bool vec_ok = (d % 4 == 0) && aligned16(x) && aligned16(y) &&
                        (!gamma || aligned16(gamma)) && (!beta || aligned16(beta));
    if (!with_row_layout(rows, d, vec_ok, 16, [&](auto l, auto vpt) {
            using L = decltype(l);
            hipLaunchKernelGGL((layernorm_reg_kernel<L, decltype(vpt)::value>), L::grid(rows), dim3(kRowThreads), 0, s,
                               x, y, gamma, beta, eps, rows, d, k);
        }))
        hipLaunchKernelGGL(layernorm_loop_kernel, dim3((unsigned)rows), dim3(kRowThreads), 0, s, x, y, gamma, beta, eps, d, k);
    return hipGetLastError();
}

// ── the attention backward's score gradients ─────────────────────────────

// dS = P (dP - rowsum(dP P)), in place of dP, in one pass: both rows are held
// in registers (4 VPT values of each per lane) between the sum and the
// products, where separate elementwise passes move each matrix six times.
// W waves per row (1: rows of up to 512, four to a workgroup).  Bound by
// memory: [32, 2048, 2048] in 155 us causal (804 MB: half of each matrix).
// With *flag == 1 (causal P, nothing past the diagonal but zeros) row t reads
// columns 0 .. t and also writes zeros to t + kCausalMargin, as far as the
// products look past the diagonal.
template <int W, int VPT>
__global__ __launch_bounds__(256) void attn_dscore_kernel(const float* __restrict__ P, float* dP, long rows, long n,
                                                          long c, long row0, const int* flag) {
    constexpr int LANES = 64 * W;
    __shared__ float red[kRowWaves];
    const int lane = threadIdx.x % LANES;
    const long row = (long)blockIdx.x * (256 / LANES) + threadIdx.x / LANES;
    if (W == 1 && row >= rows) return;
    const bool causal = flag && *flag == 1;
    const long t = row0 + row % c;
    const long have = causal ? min(n, t + 1) : n, want = causal ? min(n, t + 1 + kCausalMargin) : n;
    const float* p = P + row * n;
    float* d = dP + row * n;
    // 16-byte accesses at any 4-byte boundary
    typedef float v4u __attribute__((ext_vector_type(4), aligned(4)));
    auto get = [&](const float* x, long j, float* v) {
        if (j + 3 < have) {
            const v4u q = *reinterpret_cast<const v4u*>(x + j);
            v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = j + e < have ? x[j + e] : 0.0f;
        }
    };
    auto put = [&](long j, const float* pv, const float* dv, float s) {
        v4u o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = j + e < have ? pv[e] * (dv[e] - s) : 0.0f;
        if (j + 3 < want) {
            *reinterpret_cast<v4u*>(d + j) = o;
        } else {
#pragma unroll
            for (int e = 0; e < 3; e++)
                if (j + e < want) d[j + e] = o[e];
        }
    };
    float s = 0.0f;
    if constexpr (VPT > 0) {
        float pv[4 * VPT], dv[4 * VPT];
#pragma unroll
        for (int i = 0; i < VPT; i++) {
            const long j = 4L * (lane + i * LANES);
            get(p, j, pv + 4 * i);
            get(d, j, dv + 4 * i);
        }
#pragma unroll
        for (int e = 0; e < 4 * VPT; e++) s = __builtin_fmaf(dv[e], pv[e], s);
        if constexpr (W == 1) s = wave_sum(s);
        else s = block_sum<false>(s, red);
#pragma unroll
        for (int i = 0; i < VPT; i++) {
            const long j = 4L * (lane + i * LANES);
            if (j < want) put(j, pv + 4 * i, dv + 4 * i, s);
        }
    } else {
        for (long j = 4L * lane; j < have; j += 4L * LANES) {
            float pv[4], dv[4];
            get(p, j, pv);
            get(d, j, dv);
#pragma unroll
            for (int e = 0; e < 4; e++) s = __builtin_fmaf(dv[e], pv[e], s);
        }
        s = block_sum<false>(s, red);
        for (long j = 4L * lane; j < want; j += 4L * LANES) {
            float pv[4], dv[4];
            get(p, j, pv);
            get(d, j, dv);
            put(j, pv, dv, s);
        }
    }
}

hipError_t attn_dscore_launch(const float* P, float* dP, long rows, long seq, long c, long row0, const int* flag,
                              hipStream_t s) {
#define RAC_DSCORE(W, VPT)                                                                                     \
    hipLaunchKernelGGL((attn_dscore_kernel<W, VPT>), dim3((unsigned)((rows * W + 3) / 4)), dim3(256), 0, s, P, \
                       dP, rows, seq, c, row0, flag)
    if (seq <= 256) RAC_DSCORE(1, 1);
    else if (seq <= 512) RAC_DSCORE(1, 2);
    else if (seq <= 1024) RAC_DSCORE(4, 1);
    else if (seq <= 2048) RAC_DSCORE(4, 2);
    else if (seq <= 4096) RAC_DSCORE(4, 4);
    else if (seq <= 8192) RAC_DSCORE(4, 8);
    else RAC_DSCORE(4, 0);
#undef RAC_DSCORE
    return hipGetLastError();
}

}  // namespace rac

// rac_decode.hip — the per-token pieces of a decoder layer's decode step
// that are not GEMVs or row norms (bench/bench_rac_transformer.c
// decoder_forward_kv :557-616 with T_new = 1): the key/value cache append,
// grouped-query attention of the new token over the cache, SiLU(gate) * up,
// and the cache position's advance.
//
// The token's position lives in device memory (one int) and every kernel
// here reads it there, so the launches of a whole decode step have fixed
// arguments: the step can be recorded once as a HIP graph and replayed per
// token, the position advancing inside the graph.
//
// Attention is one workgroup per query head h, reading key /
// value head g = h / rep of a cache laid out [n_kv_heads, t_cap, d_head]
// (each head's keys a row-major matrix).  Its arithmetic is that of the
// composition  scores = alpha * (q K^T) (FAST MAC: one fmaf chain over
// d_head in order, from +0), softmax by the row kernel, out = P V (one fmaf
// chain over the positions in order)  with the softmax row padded with -inf
// to a multiple of 4 (the row kernel's 16-byte form: lane l sums the
// elements 4 g .. 4 g + 3 of its groups g = l, l + 256, ... in order, then
// the fixed wave and block combination); P V over the padded length equals
// the unpadded one, since the padded probabilities are +0.  So the output
// is bit-identical to bmm -> softmax -> bmm on the padded scores.
#include <hip/hip_runtime.h>
#include "rac_act.hpp"
#include "rac_internal.hpp"
#include "rac_math.hpp"
#include "rac_rowred.hpp"

namespace rac {

// softmax exps of 4 values x - max (<= 0 or NaN), as the row kernel's
// unmasked form: step-major CORDIC for compile-time step counts (kLean:
// NaN is forced into the row sum separately), the runtime loop otherwise
template <int NITER>
__device__ __forceinline__ void dec_exp4(float* v, int iters, float khinv) {
    if constexpr (NITER > 0) {
        exp_cordic_vec<NITER, 4, kExpFlush | kExpNonPos>(v, khinv);
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = exp_cordic_rt(v[e], iters, khinv);
    }
}

// V tile staged in LDS for the P V chains: kDecTile floats (16 KB)
constexpr int kDecTile = 4096;

// Any d_head (those the matrix-core kernel below does not take): one
// workgroup per query head.
// Scores: lane t computes positions t, t + 256, ... (one fmaf chain each).  Softmax:
// lane l takes the groups l, l + 256, ... as the row kernel.  P V: the
// value rows pass through LDS a tile at a time (every lane loads, the next
// tile's loads are in flight during the chains), and lane c < d_head runs
// output column c's chain over the tile.
template <int NITER>
__global__ __launch_bounds__(kRowThreads) void decode_attention_kernel(
    const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc,
    float* __restrict__ out, int rep, int dh, long t_cap, const int* __restrict__ pos_dev, float scale,
    int iters, float khinv)
{
    __shared__ __attribute__((aligned(16))) float sq[kDecodeMaxHead];
    __shared__ __attribute__((aligned(16))) float sp[kDecodeMaxLen];
    __shared__ __attribute__((aligned(16))) float sv[kDecTile];
    __shared__ float red[2 * kRowWaves];
    const int tid = threadIdx.x;
    const int h = blockIdx.x;
    const long g = h / rep;
    const int pos = *pos_dev;
    float* o = out + (long)h * dh;
    if (pos < 0 || pos >= t_cap || pos >= kDecodeMaxLen) {
        // a position outside the cache: NaN output, nothing read
        for (int c = tid; c < dh; c += kRowThreads) o[c] = __builtin_nanf("");
        return;
    }
    const int n = pos + 1;                 // positions 0 .. pos, the new token's included
    const int n4 = (n + 3) / 4;
    const float* K = kc + g * t_cap * dh;
    const float* V = vc + g * t_cap * dh;
    for (int c = tid; c < dh; c += kRowThreads) sq[c] = q[(long)h * dh + c];
    __syncthreads();

    for (int j = tid; j < n; j += kRowThreads) {
        const float* kr = K + (long)j * dh;
        float acc = 0.0f;
        for (int k = 0; k < dh; k++) acc = __builtin_fmaf(sq[k], kr[k], acc);
        sp[j] = scale * acc;
    }
    if (tid < 4 * n4 - n) sp[n + tid] = -__builtin_inff();       // the row's -inf padding
    __syncthreads();

    // the lane's maximum, exps and sum over its groups, in group order
    float m = -__builtin_inff();
    for (int gi = tid; gi < n4; gi += kRowThreads) {
#pragma unroll
        for (int c = 0; c < 4; c++) m = fmaxf(m, sp[4 * gi + c]);
    }
    m = block_max<false>(m, red);
    if (m == 0.0f) {
        // the signed zero the reference's scan ends on (first_zero_max)
        __shared__ uint32_t zred[kRowWaves];
        uint32_t key = ~0u;
        for (int gi = tid; gi < n4 && key == ~0u; gi += kRowThreads) {
#pragma unroll
            for (int c = 3; c >= 0; c--)
                if (sp[4 * gi + c] == 0.0f) key = zero_key<uint32_t>(4 * gi + c, sp[4 * gi + c]);
        }
        m = first_zero_max<false>(key, zred);
    }
    constexpr bool kLean = NITER > 0;
    float nanp = -__builtin_inff();
    float s = 0.0f;
    for (int gi = tid; gi < n4; gi += kRowThreads) {
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            v[c] = sp[4 * gi + c] - m;
            if constexpr (kLean) nanp = __builtin_elementwise_maximum(nanp, v[c]);
        }
        dec_exp4<NITER>(v, iters, khinv);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            s += v[c];
            sp[4 * gi + c] = v[c];
        }
    }
    if constexpr (kLean) {
        if (nanp != nanp) s = __builtin_nanf("");
    }
    s = block_sum<false>(s, red + kRowWaves);
    const float inv = 1.0f / s;
    for (int gi = tid; gi < n4; gi += kRowThreads) {
#pragma unroll
        for (int c = 0; c < 4; c++) sp[4 * gi + c] = sp[4 * gi + c] * inv;
    }

    // out[c] = sum_j p_j V[j][c], one chain per output column in j order
    const int tj = kDecTile / dh;                        // value rows per tile
    constexpr int kF4 = kDecTile / 4 / kRowThreads;      // tile float4 per lane
    float4 pre[kF4];
    auto fetch = [&](int j0) {                           // rows j0 .. of the tile into registers
        const int cnt = (n - j0 < tj ? n - j0 : tj) * dh;
        const float* src = V + (long)j0 * dh;
#pragma unroll
        for (int i = 0; i < kF4; i++) {
            const int e = (tid + i * kRowThreads) * 4;
            pre[i].x = e < cnt ? src[e] : 0.0f;
            pre[i].y = e + 1 < cnt ? src[e + 1] : 0.0f;
            pre[i].z = e + 2 < cnt ? src[e + 2] : 0.0f;
            pre[i].w = e + 3 < cnt ? src[e + 3] : 0.0f;
        }
    };
    float acc = 0.0f;
    fetch(0);
    for (int j0 = 0; j0 < n; j0 += tj) {
        __syncthreads();                                 // previous tile's chains done (and sp final)
#pragma unroll
        for (int i = 0; i < kF4; i++) reinterpret_cast<float4*>(sv)[tid + i * kRowThreads] = pre[i];
        __syncthreads();
        if (j0 + tj < n) fetch(j0 + tj);                 // in flight during the chains
        const int cnt = n - j0 < tj ? n - j0 : tj;
        if (tid < dh) {
            int u = 0;
            for (; u + 8 <= cnt; u += 8) {
#pragma unroll
                for (int w = 0; w < 8; w++) acc = __builtin_fmaf(sp[j0 + u + w], sv[(u + w) * dh + tid], acc);
            }
            for (; u < cnt; u++) acc = __builtin_fmaf(sp[j0 + u], sv[u * dh + tid], acc);
        }
    }
    if (tid < dh) o[tid] = acc;
}

// ── the same on the matrix cores (d_head 32, 64, 128) ────────────────────
//
// One workgroup of 16 waves per query head.  Every chain of the form above is
// kept, four k per instruction: a 16x16x4 matrix instruction is four in-order
// fmaf steps on each of 16 x 16 outputs (rac_gemm_fast.hip), here on 16
// positions (scores) or 16 columns (P V) of one head.  What bounds a step of
// a few hundred positions is latency, so each stage spreads over the waves
// and its loads are requested stages ahead:
//   scores   a wave takes 16 positions at a time, two such tiles in flight:
//            its key rows come by 16-byte loads of whole rows and pass through
//            a piece of LDS of its own (permuted as below; no barrier).
//            Loaded as the instruction wants them, 16 rows by 64 bytes, four
//            neighbouring lanes touch four cache lines: 132 KB of keys took
//            4.7 us to request, against 3.1;
//   softmax  one exp per lane and 1024 positions; the row sum on four waves
//            in the row kernel's order; the probabilities go to LDS permuted,
//            k = 4 t + q of a 16-k group at 4 q + t, so that one ds_read_b128
//            feeds four instructions;
//   P V      a wave per 16 columns; its values, kDecAhead groups of 16
//            positions in flight from before the scores on, go straight to
//            the instruction: 10-14 cycles per position of the chain, where a
//            lane of the VALU form took ~35 (its fmaf, its LDS reads).
// The softmax loops over the lanes' positions, its values in LDS: held in
// registers (2 or, in caches of more than 2048 positions, 8 to a lane) its
// unrolled stages cost a short row the instruction fetches of all 8, d_head 64
// at length 16 4.45 us against 3.96.
// Replayed in a graph (32 heads over 4, d_head 64, any cache length), one
// workgroup of 4 waves on the VALU before -> now: length 1 3.9 -> 3.7, 256 8.5
// -> 6.3, 516 14.6 -> 9.8, 2047 46.7 -> 28.8 us (d_head 128: 4.3 -> 4.2, 11.7
// -> 9.0, 21.3 -> 15.6, 75.7 -> 48.9).  Four heads to a workgroup (one reading
// of the keys for them) were slower: 12.6 us at 516, the exps of all four
// being on one CU.
typedef float v4f __attribute__((ext_vector_type(4)));
// the same at any 4-byte boundary (global_load / store_dwordx4 need no more):
// every alignment of the queries, the caches and the output runs here
typedef float v4u __attribute__((ext_vector_type(4), aligned(4)));
constexpr int kDecWaves = 16, kDecThreads = 64 * kDecWaves;

template <int NITER, int DH>
__global__ __launch_bounds__(kDecThreads) void decode_attention_mfma_kernel(
    const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc,
    float* __restrict__ out, int rep, long t_cap, const int* __restrict__ pos_dev, float scale, int iters,
    float khinv)
{
    constexpr int DF = DH / 16, kDecTiles = DH == 128 ? 1 : 2, kDecAhead = DH == 128 ? 6 : 8;
    // a wave's key staging: 16 rows of KP floats (a row, or half a long one)
    constexpr int KP = DH < 64 ? DH : 64, KR = KP + 8, PARTS = DH / KP, VECS = KP / 16;
    __shared__ __attribute__((aligned(16))) float sk[kDecWaves][16 * KR];
    __shared__ __attribute__((aligned(16))) float sp[kDecodeMaxLen];
    __shared__ __attribute__((aligned(16))) float rmax[kDecWaves];
    __shared__ __attribute__((aligned(16))) uint32_t rzero[kDecWaves];
    __shared__ float rsum[kRowWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane % 16, lq = lane / 16;
    // workgroup L runs on XCD L % 8: neighbouring heads, which share keys and
    // values, on one XCD and its L2
    const int nh = gridDim.x, h = nh % 8 ? blockIdx.x : (blockIdx.x % 8) * (nh / 8) + blockIdx.x / 8, g = h / rep;
    const int pos = *pos_dev;
    if (pos < 0 || pos >= t_cap || pos >= kDecodeMaxLen) {
        // a position outside the cache: NaN output, nothing read
        for (int c = tid; c < DH; c += kDecThreads) out[(long)h * DH + c] = __builtin_nanf("");
        return;
    }
    const int n = pos + 1, n4 = (n + 3) / 4, n16 = (n + 15) / 16;
    const float* K = kc + (long)g * t_cap * DH;
    const float* V = vc + (long)g * t_cap * DH;

    // keys of positions 16 b ..: part h (KP columns), 16-byte vector lane + 64 i
    v4f kf[kDecTiles][DF];
    auto kload = [&](int b, v4f (&f)[DF]) {
#pragma unroll
        for (int h = 0; h < PARTS; h++)
#pragma unroll
            for (int i = 0; i < VECS; i++) {
                const int v = lane + 64 * i;
                f[h * VECS + i] = *reinterpret_cast<const v4u*>(
                    K + (long)min(16 * b + v / (KP / 4), n - 1) * DH + h * KP + 4 * (v % (KP / 4)));
            }
    };
    float* skw = sk[wave];
    const v4f q4 = *reinterpret_cast<const v4u*>(q + (long)h * DH + 4 * (lane % (DH / 4)));
#pragma unroll
    for (int u = 0; u < kDecTiles; u++)
        if (wave + kDecWaves * u < n16) kload(wave + kDecWaves * u, kf[u]);

    // P V's values, group of 16 positions b: V[16 b + 4 t + lq][16 wave + li],
    // the last, partial group apart (-0 past the row: times the probability 0
    // there it leaves every accumulator as it is, -0 too)
    const bool pv_wave = wave < DF;
    const int nf = n / 16;
    v4f vr[kDecAhead], vt = {-0.0f, -0.0f, -0.0f, -0.0f};
    const uint32_t voff = (uint32_t)(lq * DH + 16 * wave + li) * 4u;
    auto vload = [&](int b) {
        const char* base = reinterpret_cast<const char*>(V + (long)b * 16 * DH);
        v4f v;
#pragma unroll
        for (int t = 0; t < 4; t++) v[t] = *reinterpret_cast<const float*>(base + 16 * t * DH + voff);
        return v;
    };
    if (pv_wave) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int j = 16 * nf + 4 * t + lq;
            if (j < n) vt[t] = V[(long)j * DH + 16 * wave + li];
        }
        if (nf) {
#pragma unroll
            for (int u = 0; u < kDecAhead; u++) vr[u] = vload(min(u, nf - 1));
        }
    }

    // scores: every column of the instruction's output is this head; the
    // query passes through the staging as the keys do
    auto own_lds = [&]() {
        // the wave's own writes, read back by other lanes
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    };
    v4f qf[DF];                                                   // q[16 c + 4 t + lq]
    if (lane < DH / 4) {
#pragma unroll
        for (int e = 0; e < 4; e++) skw[(lane / 4) * 16 + lane % 4 + 4 * e] = q4[e];
    }
    own_lds();
#pragma unroll
    for (int c = 0; c < DF; c++) qf[c] = *reinterpret_cast<const v4f*>(skw + 16 * c + 4 * lq);
    own_lds();
    for (int b0 = wave; b0 < n16; b0 += kDecWaves * kDecTiles) {
#pragma unroll
        for (int u = 0; u < kDecTiles; u++) {
            const int b = b0 + kDecWaves * u;
            if (b < n16) {
                v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int p = 0; p < PARTS; p++) {
#pragma unroll
                    for (int i = 0; i < VECS; i++) {
                        const int v = lane + 64 * i, c = v % (KP / 4);
                        float* o = skw + (v / (KP / 4)) * KR + (c / 4) * 16 + c % 4;
#pragma unroll
                        for (int e = 0; e < 4; e++) o[4 * e] = kf[u][p * VECS + i][e];
                    }
                    own_lds();
                    v4f a[VECS];
#pragma unroll
                    for (int c = 0; c < VECS; c++)
                        a[c] = *reinterpret_cast<const v4f*>(skw + li * KR + 16 * c + 4 * lq);
#pragma unroll
                    for (int c = 0; c < VECS; c++)
#pragma unroll
                        for (int t = 0; t < 4; t++)
                            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[c][t], qf[p * VECS + c][t], acc, 0, 0, 0);
                    own_lds();
                }
                if (b + kDecWaves * kDecTiles < n16) kload(b + kDecWaves * kDecTiles, kf[u]);
                // positions j .. j + 3; -inf past the row
                const int j = 16 * b + 4 * lq;
                v4f v;
#pragma unroll
                for (int r = 0; r < 4; r++) v[r] = j + r < n ? scale * acc[r] : -__builtin_inff();
                if (li == 0) *reinterpret_cast<v4f*>(&sp[j]) = v;
            }
        }
    }
    __syncthreads();

    // row maximum; a zero maximum takes the sign of the row's first zero
    // (first_zero_max)
    float m = -__builtin_inff();
    for (int j = tid; j < n; j += kDecThreads) m = fmaxf(m, sp[j]);
    m = wave_max_valu(m);
    uint32_t key = ~0u;
    if (m == 0.0f) {
        for (int j = tid; j < n; j += kDecThreads)
            if (sp[j] == 0.0f) {
                key = zero_key<uint32_t>(j, sp[j]);
                break;
            }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) key = min(key, (uint32_t)__shfl_xor((int)key, off, 64));
    }
    if (lane == 0) {
        rmax[wave] = m;
        rzero[wave] = key;
    }
    __syncthreads();
    m = rmax[0];
#pragma unroll
    for (int i = 1; i < kDecWaves; i++) m = fmaxf(m, rmax[i]);
    if (m == 0.0f) {
        key = rzero[0];
#pragma unroll
        for (int i = 1; i < kDecWaves; i++) key = min(key, rzero[i]);
        m = (key & 1) ? -0.0f : 0.0f;
    }

    // exps, of the -inf up to the last group of four too; a NaN score stays
    // NaN and makes the row's sum, and every probability, NaN
    for (int j = tid; j < 4 * n4; j += kDecThreads) {
        float v[1] = {sp[j] - m};
        const bool nan = v[0] != v[0];
        if constexpr (NITER > 0) exp_cordic_vec<NITER, 1, kExpFlush | kExpNonPos>(v, khinv);
        else v[0] = exp_cordic_rt(v[0], iters, khinv);
        sp[j] = nan ? __builtin_nanf("") : v[0];
    }
    __syncthreads();
    if (tid < kRowThreads) {
        float s = 0.0f;
        for (int gi = tid; gi < n4; gi += kRowThreads) {
            const v4f v = *reinterpret_cast<const v4f*>(&sp[4 * gi]);
#pragma unroll
            for (int c = 0; c < 4; c++) s += v[c];
        }
        s = wave_sum_valu(s);
        if (lane == 0) rsum[wave] = s;
    }
    __syncthreads();
    float s = rsum[0];
#pragma unroll
    for (int i = 1; i < kRowWaves; i++) s += rsum[i];
    const float inv = 1.0f / s;
    // permuted within groups of 16, which a wave reads and writes as a whole
    for (int j = tid; j < 16 * n16; j += kDecThreads) {
        const float v = j < n ? sp[j] * inv : 0.0f;
        own_lds();
        sp[(j & ~15) + 4 * (j & 3) + ((j >> 2) & 3)] = v;
    }
    __syncthreads();

    if (pv_wave) {
        const float* prow = sp + 4 * lq;
        v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
        auto mac = [&](v4f p, v4f v) {
#pragma unroll
            for (int t = 0; t < 4; t++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t], p[t], acc, 0, 0, 0);
        };
        auto probs = [&](int b) { return *reinterpret_cast<const v4f*>(prow + 16 * b); };
        v4f p = probs(0);
        int b0 = 0;
        for (; b0 + kDecAhead < nf; b0 += kDecAhead) {
#pragma unroll
            for (int u = 0; u < kDecAhead; u++) {
                const v4f pn = probs(b0 + u + 1);
                mac(p, vr[u]);
                vr[u] = vload(min(b0 + u + kDecAhead, nf - 1));
                p = pn;
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int u = 0; u < kDecAhead; u++)
            if (b0 + u < nf) {
                mac(p, vr[u]);
                p = probs(min(b0 + u + 1, n16 - 1));
            }
        if (nf < n16) mac(p, vt);
        if (li == 0) *reinterpret_cast<v4u*>(out + (long)h * DH + 16 * wave + 4 * lq) = acc;
    }
}

template <int NITER>
static hipError_t decode_attention_dh(int dh, const float* q, const float* kc, const float* vc,
                                      float* out, int n_heads, int rep, long t_cap, const int* pos, float scale,
                                      int iters, float khinv, hipStream_t s) {
#define RAC_DEC_ATT(D)                                                                                         \
    hipLaunchKernelGGL((decode_attention_mfma_kernel<NITER, D>), dim3(n_heads), dim3(kDecThreads), 0, s, q, kc, \
                       vc, out, rep, t_cap, pos, scale, iters, khinv)
    if (dh == 64) RAC_DEC_ATT(64);
    else if (dh == 128) RAC_DEC_ATT(128);
    else if (dh == 32) RAC_DEC_ATT(32);
    else
        hipLaunchKernelGGL((decode_attention_kernel<NITER>), dim3(n_heads), dim3(kRowThreads), 0, s, q, kc, vc, out,
                           rep, dh, t_cap, pos, scale, iters, khinv);
#undef RAC_DEC_ATT
    return hipGetLastError();
}

hipError_t decode_attention_launch(const float* q, const float* kc, const float* vc, float* out, int n_heads,
                                   int n_kv_heads, int dh, long t_cap, const int* pos, float scale, int iters,
                                   hipStream_t s) {
    iters = clamp_iters(iters);
    const float khinv = host_consts().exp_khinv[iters];
    const int rep = n_heads / n_kv_heads;
    switch (iters) {
        case 8: return decode_attention_dh<8>(dh, q, kc, vc, out, n_heads, rep, t_cap, pos, scale, iters, khinv, s);
        case 16: return decode_attention_dh<16>(dh, q, kc, vc, out, n_heads, rep, t_cap, pos, scale, iters, khinv, s);
        case 24: return decode_attention_dh<24>(dh, q, kc, vc, out, n_heads, rep, t_cap, pos, scale, iters, khinv, s);
        default: return decode_attention_dh<0>(dh, q, kc, vc, out, n_heads, rep, t_cap, pos, scale, iters, khinv, s);
    }
}

// ── cache append ─────────────────────────────────────────────────────────

// kv = [k (n_kv_heads * d_head) | v (n_kv_heads * d_head)] of the new token
// (the K and V projections' outputs, adjacent); written at the position
// *pos of every head's rows.  A position outside the cache writes nothing.
__global__ __launch_bounds__(256) void kv_append_kernel(const float* __restrict__ kv, float* __restrict__ kc,
                                                       float* __restrict__ vc, long w, int dh, long t_cap,
                                                       const int* __restrict__ pos_dev) {
    const int pos = *pos_dev;
    if (pos < 0 || pos >= t_cap) return;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < 2 * w; i += (long)gridDim.x * 256) {
        const long r = i < w ? i : i - w;
        const long g = r / dh, c = r - g * dh;
        (i < w ? kc : vc)[(g * t_cap + pos) * dh + c] = kv[i];
    }
}

hipError_t kv_append_launch(const float* kv, float* kc, float* vc, int n_kv_heads, int dh, long t_cap,
                            const int* pos, hipStream_t s) {
    const long w = (long)n_kv_heads * dh;
    const long blocks = (2 * w + 255) / 256;
    hipLaunchKernelGGL(kv_append_kernel, dim3((unsigned)(blocks < 1024 ? blocks : 1024)), dim3(256), 0, s, kv, kc,
                       vc, w, dh, t_cap, pos);
    return hipGetLastError();
}

__global__ void position_advance_kernel(int* pos, int by) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *pos += by;
}

hipError_t position_advance_launch(int* pos, int by, hipStream_t s) {
    hipLaunchKernelGGL(position_advance_kernel, dim3(1), dim3(64), 0, s, pos, by);
    return hipGetLastError();
}

// ── SiLU(gate) * up ──────────────────────────────────────────────────────

// out[i] = silu(gu[i]) * gu[n + i]: the gate and up projections stacked in
// one vector; SiLU by the CORDIC exp of the elementwise kernels (same bits).
template <int NITER>
__global__ __launch_bounds__(256) void swiglu_kernel(const float* __restrict__ gu, float* __restrict__ out, long n,
                                                    int iters, float khinv) {
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256)
        out[i] = elt<kEltSilu, NITER>(gu[i], iters, khinv) * gu[n + i];
}

hipError_t swiglu_launch(const float* gu, float* out, long n, int iters, hipStream_t s) {
    iters = clamp_iters(iters);
    const float khinv = host_consts().exp_khinv[iters];
    const long blocks = (n + 255) / 256;
    const dim3 grid((unsigned)(blocks < 4096 ? blocks : 4096));
    switch (iters) {
        case 8: hipLaunchKernelGGL((swiglu_kernel<8>), grid, dim3(256), 0, s, gu, out, n, iters, khinv); break;
        case 16: hipLaunchKernelGGL((swiglu_kernel<16>), grid, dim3(256), 0, s, gu, out, n, iters, khinv); break;
        case 24: hipLaunchKernelGGL((swiglu_kernel<24>), grid, dim3(256), 0, s, gu, out, n, iters, khinv); break;
        default: hipLaunchKernelGGL((swiglu_kernel<0>), grid, dim3(256), 0, s, gu, out, n, iters, khinv); break;
    }
    return hipGetLastError();
}

}  // namespace rac

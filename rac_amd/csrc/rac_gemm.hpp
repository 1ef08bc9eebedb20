// rac_gemm.hpp — what the GEMM kernel files share: a launch's arguments and
// the causal score trapezoid.
#pragma once
#include <hip/hip_runtime.h>
#include "rac_internal.hpp"

namespace rac {

struct GemmArgs {
    const float* A;
    const float* B;
    float* C;
    int M, N, K;
    float alpha, beta;
    int iters;
    int batch;
    long sa, sb, sc;
    GemmEpilogue ep;
    bool fused;
    int sched;
    const int* k_causal;
    int exact_specials;
    int row0;
    // with k_causal: 1, row tile m sums k only up to its last query position
    // row0 + m*BM + BM - 1 (P V); 2, only from k = m*BM - row0 on (P^T dO: row
    // s of P^T is 0 before query position s, k = 0 being position row0); 3,
    // tiles wholly above the diagonal are left unwritten (dO V^T, rows from
    // query position row0; without k_causal too).  2 and 3 in FAST mode only.
    int k_side;
    int period;      // k_side 3: row m is at query position row0 + m % period (0: row0 + m)
};

// Column tiles of row tile r in a causal score trapezoid (query rows
// row0 + r*BM .. row0 + r*BM + BM - 1, keys 0 .. N-1): those holding a key
// position not past the row tile's last query position.
__host__ __device__ __forceinline__ int trap_cols(int row0, int r, int BM, int BN, int N) {
    const long last = (long)row0 + (long)(r + 1) * BM - 1;
    const long c = last / BN + 1;
    const long ntn = (N + BN - 1) / BN;
    return (int)(c < ntn ? c : ntn);
}

// FAST mode on the matrix cores (rac_gemm_fast.hip): K >= 4; at most one
// operand stored with its rows side by side (A of ta, B of !tb) has 2 or 3.
hipError_t gemm_fast_launch(int ta, int tb, const GemmArgs& g, hipStream_t s);
// The fused linear layer (NT) with A, B, C and the bias in bf16 (dtype 1) or
// fp16 (2), K >= 4; the products and sums in fp32, ep.pre in fp32.
hipError_t gemm_fast_half_launch(int dtype, const GemmArgs& g, hipStream_t s);

}  // namespace rac

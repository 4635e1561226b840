// fp32 products on the matrix cores (f32_gemm.hip), for the fp32 Medusa block and the chain cell.
#pragma once

#include "fg_common.h"

namespace fg {

// C[z] = A[z] . B[z]^T for z < batch: A [M, K] (row stride lda, batches a_batch apart), B [N, K].
// K and N multiples of 4, 16-byte aligned rows. With B2, B's columns from k_b2 (a multiple of 4) on
// are those of B2 [N, K - k_b2], of the same row stride.
struct F32Gemm {
  const float* A;
  int64_t lda, a_batch;
  const float* B;
  int64_t ldb, b_batch;
  int M, N, K, batch;
  const float* B2 = nullptr;
  int k_b2 = 0;
};

// Parts of K (at most 16): the count with the least (rounds of workgroups over the CUs) x (steps of
// a part, 2 more for its start and end), a lone round counting half again, as nothing then covers
// a wave's waits. 768 x 512 x 8192: 8 parts, three whole rounds (5 parts, 1.9 rounds: 71 us to 67).
int f32_splits(int M, int N, int K, int batch);
// parts[p][z][m][n]: the sums of part p, `splits` as f32_splits gives it.
int f32_gemm_parts(const F32Gemm& g, int splits, float* parts, hipStream_t s);

// fg_chain_cell_norm with token rows of their own dtype (layers.hip): that of the state and the
// weights, or bf16.
int chain_cell_norm(const void* state, int64_t ld_state, int dtype, const void* token, int64_t ld_token,
                    int token_dtype, int rows, int hidden, const void* state_w, const void* state_b,
                    const void* token_w, const void* token_b, float eps, void* out, hipStream_t s);

}  // namespace fg

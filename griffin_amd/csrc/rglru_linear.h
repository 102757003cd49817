// Shared by the matrix products of the Linear layers (rglru_linear.hip: fp32 and the forward; rglru_linear16.hip: the gradients in bf16).
#pragma once

#include <hip/hip_runtime.h>

#include "rglru_device.h"
#include "rglru_host.h"

namespace rglru {

struct LinearArgs {
  // `batch` equal problem sets side by side, operands a_step, b_step and c_step elements on: the gate blocks of the RG-LRU
  long long a_step, b_step, c_step;
  int batch, accumulate;             // accumulate: c += product, rounded once
  int partial_ld;                    // partial: [split][batch][problem][partial_ld][partial_ld] where set, else [split][problem][M][N]
  const void* a[2]; const void* b[2]; const void* bias[2]; void* c[2];
  const unsigned char* active;       // one byte per token, or null: inactive rows of the result are zero (weight gradient: rows of A count as zero)
  float* partial;                    // [split][problem][M][N] instead of c where the contraction is split
  float* colsum;                     // weight gradient: [split][problem][M] column sums of A, or null
  long long lda, ldb, ldc;           // elements between rows in memory
  int M, N, K;                       // of one problem; K of one segment (input gradient)
  int tiles_m, tiles_n, problems, segments, splits, k_per_split, total;
};

// Four consecutive elements (N is a multiple of a 16-byte vector, so they lie wholly inside or outside a row).
template <typename IO> RGLRU_DEVICE auto buf_load_four(rsrc_t r, unsigned voff) {
  typedef IO io4 __attribute__((ext_vector_type(4)));
  if constexpr (sizeof(IO) == 2) return __builtin_bit_cast(io4, __builtin_amdgcn_raw_buffer_load_b64(r, voff, 0, 0));
  else return __builtin_bit_cast(io4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
}

// How a product is cut up: edge of the square tiles, and workgroups that share a contraction.
struct LinearPlan { int edge, splits; };

// rglru_linear16.hip: input gradients (kind RGLRU_LINEAR_INPUT_GRAD) and weight gradients in bf16
void linear16_launch(LinearArgs& a, int kind, int edge, hipStream_t s);

}  // namespace rglru

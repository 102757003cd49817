// Shared by the matrix products of the Linear layers (rglru_linear.hip: fp32 and the forward; rglru_linear16.hip: the gradients in bf16).
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/rglru_hip.h"
#include "rglru_device.h"
#include "rglru_host.h"

namespace rglru {

// What the block forward of an inference call needs in front of it: the flag bytes of every token (reset at position 0, in bits 2-3 the
// lags that reach in front of the document), each row's last position and the cleared part of the workspace.  It rides on the launch of
// the two input projections (block prefill B3 T777 D768 W1024: 48.6 us with a launch of its own, 46.9 so; without a cache 47.6 and 44.1
// beside the plain forward kernel), or is a launch of its own.
struct PositionArgs {
  const long long* prev; const long long* segpos; unsigned char* flags; long long* last;
  uint4* clear; long long clear_n;
  int B, T;
};
RGLRU_DEVICE void token_positions(const PositionArgs& p, long long first, long long stride) {
  const long long n = p.flags ? (long long)p.B * p.T : 0;
  for (long long i = first; i < p.clear_n; i += stride) p.clear[i] = make_uint4(0u, 0u, 0u, 0u);
  for (long long i = first; i < n; i += stride) {
    const int b = (int)(i / p.T), t = (int)(i - (long long)b * p.T);
    const long long pos = p.segpos ? p.segpos[i] : p.prev[b] + 1 + t;
    const unsigned near = pos < 0 ? 3u : pos < 3 ? (unsigned)(3 - pos) : 0u;
    p.flags[i] = (unsigned char)((pos == 0 ? RGLRU_FLAG_RESET : 0u) | (near << RGLRU_FLAG_CONV_SHIFT));
  }
  if (p.last)
    for (long long b = first; b < p.B; b += stride)
      p.last[b] = p.segpos ? p.segpos[b * p.T + p.T - 1] : (p.prev ? p.prev[b] : -1ll) + p.T;
}

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
  PositionArgs positions;            // forward in 16 bits: B > 0: work on the side
  int M, N, K;                       // of one problem; K of one segment (input gradient)
  int tiles_m, tiles_n, problems, segments, splits, k_per_split, total;
};

// Four consecutive elements (N is a multiple of a 16-byte vector, so they lie wholly inside or outside a row).
template <typename IO> RGLRU_DEVICE auto buf_load_four(rsrc_t r, unsigned voff) {
  typedef IO io4 __attribute__((ext_vector_type(4)));
  if constexpr (sizeof(IO) == 2) return __builtin_bit_cast(io4, __builtin_amdgcn_raw_buffer_load_b64(r, voff, 0, 0));
  else return __builtin_bit_cast(io4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
}

// How a product is cut up: rows (and columns, where no others are given) of a tile, and workgroups that share a contraction.
struct LinearPlan { int edge, splits, columns = 0; };

// rglru_linear.hip: two products of one input, u and v, with the positions of an inference call
int linear_pair_with_positions(const void* x, const void* w0, const void* w1, const void* bias0, const void* bias1, void* u, void* v, int64_t M,
                               int64_t N, int64_t K, int dtype, const PositionArgs& positions, void* stream);

// rglru_linear16.hip: input gradients (kind RGLRU_LINEAR_INPUT_GRAD) and weight gradients in bf16
void linear16_launch(LinearArgs& a, int kind, int edge, hipStream_t s);

}  // namespace rglru

// Last step of the reductions whose first step leaves partial results in memory: sums over `sets` arrays of n elements
// each, in a fixed order, written in the gradient's type.  Several of them (and the gate gradients' own) share a launch:
// each is a few microseconds of memory latency, so side by side they cost what the longest of them does.
#pragma once

#include <hip/hip_runtime.h>

#include <cstring>

#include "rglru_device.h"
#include "rglru_host.h"

namespace rglru {

struct SumJob {
  const void* src; void* dst;
  long long n;                       // elements of a set; set s starts at src + s * n
  int sets, src_bf16, dst_bf16;
  int taps, width;                   // convolution: n = (taps + 1 or 2) * width, element j * width + c goes to dst[c * taps + j], ...
  void* dst_bias; void* dst_du;      // ... those of j = taps to dst_bias[c] and of j = taps + 1 to dst_du[c]; any may be null
  int vec;                           // elements per thread of the streaming form (8 or 1), 0: the column form
  int blocks;                        // workgroups of 256 threads
};

// Few sets of many elements (weight gradients) are streamed, `vec` consecutive elements a thread, eight sets in flight.  Many
// sets of a few thousand columns (bias gradients) are latency: a workgroup takes 32 columns, eight threads share a column
// with sixteen loads in flight each.
inline void plan_sum_job(SumJob& j) {
  if (j.taps || (j.sets > 32 && !j.src_bf16)) {
    j.vec = 0; j.blocks = (int)((j.n + 31) / 32);
  } else {
    j.vec = (j.n % 8 == 0 && (uintptr_t)j.src % 16 == 0 && (uintptr_t)j.dst % 16 == 0) ? 8 : 1;
    j.blocks = (int)((j.n / j.vec + 255) / 256);
  }
}

RGLRU_DEVICE void sum_job_store(const SumJob& j, void* dst, long long at, float v) {
  if (j.dst_bf16) ((__bf16*)dst)[at] = (__bf16)v; else ((float*)dst)[at] = v;
}

template <typename SRC>
RGLRU_DEVICE void sum_job_stream8(const SumJob& j, long long i) {
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  const SRC* src = (const SRC*)j.src + i;
  for (int s0 = 0; s0 < j.sets; s0 += 8) {
    float v[8][8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int s = s0 + q < j.sets ? s0 + q : j.sets - 1;  // a set past the last is asked again and not added
      if constexpr (sizeof(SRC) == 2) {
        const bf16x8 f = *reinterpret_cast<const bf16x8*>(src + (long long)s * j.n);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[q][e] = (float)f[e];
      } else {
        const f32x4 lo = *reinterpret_cast<const f32x4*>(src + (long long)s * j.n), hi = *reinterpret_cast<const f32x4*>(src + (long long)s * j.n + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) { v[q][e] = lo[e]; v[q][4 + e] = hi[e]; }
      }
    }
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (s0 + q < j.sets) {
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += v[q][e];
      }
  }
  if (j.dst_bf16) {
    bf16x8 out;
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = (__bf16)acc[e];
    *reinterpret_cast<bf16x8*>((__bf16*)j.dst + i) = out;
  } else {
    *reinterpret_cast<f32x4*>((float*)j.dst + i) = (f32x4){acc[0], acc[1], acc[2], acc[3]};
    *reinterpret_cast<f32x4*>((float*)j.dst + i + 4) = (f32x4){acc[4], acc[5], acc[6], acc[7]};
  }
}

// Workgroup `block` of the job (256 threads, all of them).
RGLRU_DEVICE void run_sum_job(const SumJob& j, int block, float (&red)[8][32]) {
  if (j.vec) {
    const long long i = ((long long)block * 256 + threadIdx.x) * j.vec;
    if (i >= j.n) return;
    if (j.vec == 8) {
      if (j.src_bf16) sum_job_stream8<__bf16>(j, i); else sum_job_stream8<float>(j, i);
    } else {
      float acc = 0.f;
      for (int s = 0; s < j.sets; ++s)
        acc += j.src_bf16 ? (float)((const __bf16*)j.src)[(long long)s * j.n + i] : ((const float*)j.src)[(long long)s * j.n + i];
      sum_job_store(j, j.dst, i, acc);
    }
    return;
  }
  const int col = threadIdx.x & 31, share = threadIdx.x >> 5;
  const long long c = (long long)block * 32 + col;
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  if (c < j.n) {
    const float* src = (const float*)j.src + c;
    int n = share;
    for (; n + 120 < j.sets; n += 128) {
      float v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = src[(long long)(n + 8 * u) * j.n];
#pragma unroll
      for (int u = 0; u < 16; u += 4) { s0 += v[u]; s1 += v[u + 1]; s2 += v[u + 2]; s3 += v[u + 3]; }
    }
    for (; n + 24 < j.sets; n += 32) {
      s0 += src[(long long)n * j.n]; s1 += src[(long long)(n + 8) * j.n];
      s2 += src[(long long)(n + 16) * j.n]; s3 += src[(long long)(n + 24) * j.n];
    }
    for (; n < j.sets; n += 8) s0 += src[(long long)n * j.n];
  }
  red[share][col] = (s0 + s1) + (s2 + s3);
  __syncthreads();
  if (share != 0 || c >= j.n) return;
  float s = 0.f;
#pragma unroll
  for (int q = 0; q < 8; ++q) s += red[q][col];
  if (!j.taps) { sum_job_store(j, j.dst, c, s); return; }
  const int t = (int)(c / j.width), ch = (int)(c - (long long)t * j.width);
  if (t < j.taps) { if (j.dst) sum_job_store(j, j.dst, (long long)ch * j.taps + t, s); }
  else if (void* dst = t == j.taps ? j.dst_bias : j.dst_du) sum_job_store(j, dst, ch, s);
}

// A convolution's tap and bias gradients from the per-run partials [slots][K + 1][W] (K + 2 rows with the column
// sums of du).
inline SumJob conv_sum_job(const float* partial, void* dtaps, void* dbias, int64_t W, int64_t K, int64_t slots, int grad_dtype,
                           void* du_sums = nullptr) {
  SumJob j;
  memset(&j, 0, sizeof(j));
  j.src = partial; j.dst = dtaps; j.dst_bias = dbias; j.dst_du = du_sums; j.n = (K + (du_sums ? 2 : 1)) * W; j.sets = (int)slots; j.dst_bf16 = grad_dtype == RGLRU_BF16;
  j.taps = (int)K; j.width = (int)W;
  return j;
}

// Reverse mode of the convolution without that last step (rglru_block_ops.hip): the partials stay in `scratch`.
int64_t conv_partial_sets(int64_t B, int64_t T);
int conv_bwd_partials(const void* u, const void* state, const void* taps, const int64_t* segment_pos, const int32_t* rows,
                      const void* dout, void* scratch, void* du, int64_t du_stride, void* dstate,
                      int64_t B, int64_t T, int64_t W, int64_t K, int dtype, int vec_dtype, bool sum_du, void* stream);

}  // namespace rglru

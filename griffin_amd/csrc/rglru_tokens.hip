// Per-token bookkeeping of the recurrent block: what an activity mask, segment positions and a carried position say about
// every token (griffin/griffin.py:309-358, :459-510), in one launch instead of a dozen elementwise ones, and the row
// masks around it.  Bytes of bookkeeping per token are nothing next to its channels: these kernels are launch latency.

#include <hip/hip_runtime.h>

#include <cstring>

#include "rglru_device.h"
#include "rglru_host.h"

namespace rglru {

constexpr int kTokenThreads = 256;
constexpr int kTokenRun = 8;                    // consecutive tokens per thread

struct TokenArgs {
  const unsigned char* active; const long long* segpos; const long long* prev;
  long long* pos; unsigned char* flags; long long* conv_pos; int* rows; long long* last; unsigned* host;
  int B, T;
};

// Inclusive scans over the workgroup, one value per thread: a wave by shuffles, the waves through LDS.
template <typename Op>
RGLRU_DEVICE int block_scan(int v, int identity, int* lds, Op op, int* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(v, d);
    if (lane >= d) v = op(v, u);
  }
  __syncthreads();                              // the area may still be read from the scan before
  if (lane == 63) lds[wave] = v;
  __syncthreads();
  int before = identity, all = identity;
#pragma unroll
  for (int w = 0; w < kTokenThreads / 64; ++w) {
    if (w < wave) before = op(before, lds[w]);
    all = op(all, lds[w]);
  }
  *total = all;
  return op(v, before);
}

// One workgroup per row; a thread owns eight consecutive tokens, so 2048 tokens are one pass of two scans: the ordinals of
// the active tokens (sum) and the ordinal at which the document of each token started (maximum; -1: before this call).
__global__ __launch_bounds__(kTokenThreads) void token_facts_kernel(TokenArgs p) {
  __shared__ int lds[kTokenThreads / 64];
  __shared__ int s_last_t;
  __shared__ long long s_last_pos;
  const int b = blockIdx.x;
  const long long row = (long long)b * p.T;
  const long long prev = p.prev ? p.prev[b] : -1;
  int count = 0, doc = -1;                      // of the passes before
  if (threadIdx.x == 0) { s_last_t = -1; s_last_pos = prev; }
  const bool words = (p.T % 8 == 0) && ((uintptr_t)p.active % 8 == 0) && ((uintptr_t)p.flags % 8 == 0);
  for (int base = 0; base < p.T; base += kTokenThreads * kTokenRun) {
    const int t0 = base + (int)threadIdx.x * kTokenRun;
    unsigned act = 0u;                          // bit i: token t0 + i takes part
    long long given[kTokenRun];
    if (words) {
      const unsigned long long w = t0 < p.T ? *reinterpret_cast<const unsigned long long*>(p.active + row + t0) : 0ull;
#pragma unroll
      for (int i = 0; i < kTokenRun; ++i) act |= ((w >> (8 * i)) & 0xffull) ? 1u << i : 0u;
    } else {
#pragma unroll
      for (int i = 0; i < kTokenRun; ++i) act |= (t0 + i < p.T && p.active[row + t0 + i]) ? 1u << i : 0u;
    }
    if (p.segpos) {
#pragma unroll
      for (int i = 0; i < kTokenRun; ++i) given[i] = p.segpos[row + (t0 + i < p.T ? t0 + i : p.T - 1)];
    }
    int total;
    const int mine = __popc(act);
    const int upto = block_scan(mine, 0, lds, [](int x, int y) { return x + y; }, &total);
    const int first = count + upto - mine;      // ordinal of this thread's first active token
    // positions of the eight tokens, and the last document start among them
    long long pos[kTokenRun];
    int start = -1, ord = first;
#pragma unroll
    for (int i = 0; i < kTokenRun; ++i) {
      const bool a = (act >> i) & 1u;
      pos[i] = p.segpos ? given[i] : prev + ord + (a ? 1 : 0);
      if (a && pos[i] == 0) start = ord;
      ord += a ? 1 : 0;
    }
    int last_start;
    const int reached = block_scan(start, -1, lds, [](int x, int y) { return x > y ? x : y; }, &last_start);
    int s = __shfl_up(reached, 1);              // the scan up to the thread before
    if ((threadIdx.x & 63) == 0) {
      s = -1;
      for (int w = 0; w < (int)(threadIdx.x >> 6); ++w) s = s > lds[w] ? s : lds[w];
    }
    s = s > doc ? s : doc;
    ord = first;
    unsigned long long packed = 0ull;
#pragma unroll
    for (int i = 0; i < kTokenRun; ++i) {
      const bool a = (act >> i) & 1u;
      if (a && pos[i] == 0) s = ord;
      const int behind = ord - s;               // of an active token: tokens of its document in front of it
      const unsigned near = !a ? 3u : s < 0 ? 0u : behind < 3 ? 3u - (unsigned)behind : 0u;
      const unsigned char f = (unsigned char)((pos[i] == 0 ? RGLRU_FLAG_RESET : 0u) | (a ? 0u : RGLRU_FLAG_INACTIVE) | (near << RGLRU_FLAG_CONV_SHIFT));
      packed |= (unsigned long long)f << (8 * i);
      if (t0 + i < p.T) {
        if (!words) p.flags[row + t0 + i] = f;
        if (p.pos) p.pos[row + t0 + i] = pos[i];
        if (p.conv_pos) p.conv_pos[row + t0 + i] = s < 0 ? (1ll << 30) : (long long)behind;
      }
      ord += a ? 1 : 0;
    }
    if (words && t0 < p.T) *reinterpret_cast<unsigned long long*>(p.flags + row + t0) = packed;
    if (mine && first + mine == count + total) {                // this thread holds the pass's last active token
      const int i = 31 - __clz(act);
      s_last_t = t0 + i;
#pragma unroll
      for (int j = 0; j < kTokenRun; ++j) if (j == i) s_last_pos = pos[j];
    }
    count += total;
    doc = last_start > doc ? last_start : doc;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int prefix = count == s_last_t + 1 ? 1 : 0;           // the active tokens are the row's first ones
    p.rows[b] = count; p.rows[p.B + b] = doc; p.rows[2 * p.B + b] = prefix;
    if (p.last) p.last[b] = s_last_pos;
    if (p.host) p.host[b] = (count == p.T ? 1u : 0u) | (prefix ? 2u : 0u) | ((unsigned)count << 2);
  }
}

// Flag bytes from the two masks of the RG-LRU (either may be null).
__global__ __launch_bounds__(256) void pack_flags_kernel(const unsigned char* reset, const unsigned char* active, unsigned char* flags,
                                                         long long n, int words) {
  const long long stride = (long long)gridDim.x * 256;
  if (words) {                                  // eight tokens at a time
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n / 8; i += stride) {
      const unsigned long long r = reset ? reinterpret_cast<const unsigned long long*>(reset)[i] : 0ull;
      const unsigned long long a = active ? reinterpret_cast<const unsigned long long*>(active)[i] : ~0ull;
      unsigned long long f = 0ull;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        f |= (unsigned long long)((((r >> (8 * j)) & 0xffull) ? RGLRU_FLAG_RESET : 0u) | (((a >> (8 * j)) & 0xffull) ? 0u : RGLRU_FLAG_INACTIVE)) << (8 * j);
      reinterpret_cast<unsigned long long*>(flags)[i] = f;
    }
    return;
  }
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
    flags[i] = (unsigned char)((reset && reset[i] ? RGLRU_FLAG_RESET : 0u) | (active && !active[i] ? RGLRU_FLAG_INACTIVE : 0u));
}

// Rows of `bytes` bytes: those of inactive tokens become zero, the others are copied, or left alone where source and
// destination are one buffer (only the padding is written then).  V: 16 bytes, or one element.
struct MaskRowsArgs { const void* src; const unsigned char* active; void* dst; long long rows; int per_row; int in_place; };
template <typename V>
__global__ __launch_bounds__(256) void mask_rows_kernel(MaskRowsArgs p) {
  constexpr int AHEAD = 4;
  const long long n = p.rows * p.per_row, stride = (long long)gridDim.x * 256;
  const V* src = (const V*)p.src;
  V* dst = (V*)p.dst;
  for (long long i0 = (long long)blockIdx.x * 256 + threadIdx.x; i0 < n; i0 += stride * AHEAD) {
    bool live[AHEAD];
    V v[AHEAD];
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) {
      const long long i = i0 + q * stride;
      live[q] = i < n && p.active[(unsigned long long)i / (unsigned)p.per_row] != 0;
    }
    if (!p.in_place) {
#pragma unroll
      for (int q = 0; q < AHEAD; ++q) if (live[q]) v[q] = src[i0 + q * stride];
    }
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) {
      const long long i = i0 + q * stride;
      if (i < n && !(live[q] && p.in_place)) dst[i] = live[q] ? v[q] : V{};
    }
  }
}

// Right-padded rows without their padding, one behind the other: rows of `bytes` bytes (whole 16-byte vectors) of [B, T] tokens to
// `packed` rows and back.  A workgroup has sixteen tokens of a row; where the row lies follows from the counts of the rows in front of it.  What
// is left behind the last row is one more row, of zeros.  PACK: up to two arrays, and the positions and flags (as
// rglru_hip_block_fwd takes them) of tokens whose rows are documents from their beginning.  Else: one array, padding becomes zero.
// Streaming, a batch of eight vectors in flight per thread; what lies past the ends is dropped by the descriptors.  Counts that do not fit (more
// than T, or more than `packed` together) lose their tail: nothing outside the arrays is read or written whatever they say.
struct PackArgs {
  const int* counts; const f32x4* src[2]; f32x4* dst[2]; int per_row[2];
  long long* pos; unsigned char* flags; int B, T, packed, chunks;
};
constexpr int kPackTokens = 16;
template <bool PACK>
__global__ __launch_bounds__(256) void pack_rows_kernel(PackArgs p) {
  constexpr int kTokens = kPackTokens, AHEAD = 8;
  __shared__ int lds[4];
  const int b = blockIdx.x / p.chunks, chunk = blockIdx.x - b * p.chunks;
  auto count = [&](int i) { return min(max(p.counts[i], 0), p.T); };
  int before = 0;
  for (int i = threadIdx.x; i < b; i += 256) before += count(i);
#pragma unroll
  for (int d = 32; d; d >>= 1) before += __shfl_xor(before, d);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = before;
  __syncthreads();
  const int first = lds[0] + lds[1] + lds[2] + lds[3];
  const bool tail = b == p.B;                   // PACK only
  // tokens of the row that exist, and those that this launch writes
  const int there = tail ? 0 : count(b), rows = PACK ? (tail ? p.packed - first : there) : p.T;
  for (int t0 = chunk * kTokens; t0 < rows; t0 += p.chunks * kTokens) {
    const int n = rows - t0 < kTokens ? rows - t0 : kTokens;
    const long long wide = (long long)b * p.T + t0, narrow = (long long)first + t0;
#pragma unroll
    for (int a = 0; a < (PACK ? 2 : 1); ++a) {
      if (!p.dst[a]) continue;
      const unsigned per_row = (unsigned)p.per_row[a], all = (unsigned)n * per_row;
      const f32x4* src = p.src[a] + (PACK ? wide : narrow) * per_row;
      f32x4* dst = p.dst[a] + (PACK ? narrow : wide) * per_row;
      // vectors that exist, and that may be written
      const int left = there - t0 < n ? there - t0 : n, fit = p.packed - narrow < n ? (int)(p.packed - narrow) : n;
      const int from_rows = PACK ? left : min(left, fit), to_rows = PACK ? fit : n;
      const unsigned live = from_rows > 0 ? (unsigned)from_rows * per_row : 0u, room = to_rows > 0 ? (unsigned)to_rows * per_row : 0u;
      const rsrc_t from = make_rsrc(src, live * 16u), to = make_rsrc(dst, room * 16u);
      for (unsigned i0 = threadIdx.x; i0 < all; i0 += 256 * AHEAD) {
        i32x4 v[AHEAD];
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) v[q] = __builtin_amdgcn_raw_buffer_load_b128(from, (i0 + q * 256) * 16u, 0, 0);
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) buf_store_b128(v[q], to, (i0 + q * 256) * 16u);
      }
    }
    if (PACK && p.pos && (int)threadIdx.x < n && narrow + threadIdx.x < p.packed) {
      const int t = t0 + (int)threadIdx.x;
      p.pos[narrow + threadIdx.x] = t;
      p.flags[narrow + threadIdx.x] = (unsigned char)((t == 0 ? RGLRU_FLAG_RESET : 0u) | ((t < 3 ? 3u - (unsigned)t : 0u) << RGLRU_FLAG_CONV_SHIFT));
    }
  }
}

// Carried rows of the padded convolution where the active tokens are a prefix of each row: the last K - 1 inputs of the
// row's document, oldest first, reaching into the rows carried so far where no document started in this call.
struct CarryArgs { const void* u; const void* state; const int* rows; void* out; long long ldu; int B, T, W, K; };
template <typename IO>
__global__ __launch_bounds__(256) void conv_carry_kernel(CarryArgs p) {
  const int K1 = p.K - 1;
  const long long n = (long long)p.B * K1 * p.W;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int c = (int)(i % p.W), j = (int)(i / p.W % K1), b = (int)(i / p.W / K1);
  const int count = p.rows[b], doc = p.rows[p.B + b];
  const int t = count - K1 + j;                 // the token this row holds, negative: carried row K1 + t
  IO v = (IO)0.0f;
  if (t >= 0 && t >= doc) v = ((const IO*)p.u)[((long long)b * p.T + t) * p.ldu + c];
  else if (t < 0 && doc < 0 && p.state) v = ((const IO*)p.state)[((long long)b * K1 + K1 + t) * p.W + c];
  ((IO*)p.out)[i] = v;
}

}  // namespace rglru

using namespace rglru;

extern "C" {

int rglru_hip_token_facts(const uint8_t* active, const int64_t* segment_pos, const int64_t* prev_pos, int64_t* pos, uint8_t* flags,
                          int64_t* conv_pos, int32_t* rows, int64_t* last_pos, uint32_t* host_facts, int64_t B, int64_t T,
                          void* stream) {
  if (!active || !flags || !rows) return fail(RGLRU_E_ARG, "token_facts: null pointer");
  if (B <= 0 || T <= 0) return fail(RGLRU_E_ARG, "token_facts: empty shape B=%lld T=%lld", (long long)B, (long long)T);
  if (T >= (1ll << 30) || B >= (1ll << 30)) return fail(RGLRU_E_UNSUPPORTED, "token_facts: too large");
  TokenArgs a;
  a.active = active; a.segpos = (const long long*)segment_pos; a.prev = (const long long*)prev_pos; a.pos = (long long*)pos;
  a.flags = flags; a.conv_pos = (long long*)conv_pos; a.rows = rows; a.last = (long long*)last_pos; a.host = host_facts;
  a.B = (int)B; a.T = (int)T;
  hipLaunchKernelGGL(token_facts_kernel, dim3((unsigned)B), dim3(kTokenThreads), 0, (hipStream_t)stream, a);
  return check_launch("token_facts");
}

int rglru_hip_pack_flags(const uint8_t* reset, const uint8_t* active, uint8_t* flags, int64_t n, void* stream) {
  if ((!reset && !active) || !flags) return fail(RGLRU_E_ARG, "pack_flags: null pointer");
  if (n <= 0) return fail(RGLRU_E_ARG, "pack_flags: empty mask");
  const int words = n % 8 == 0 && (uintptr_t)reset % 8 == 0 && (uintptr_t)active % 8 == 0 && (uintptr_t)flags % 8 == 0;
  long long blocks = ((words ? n / 8 : n) + 255) / 256; if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(pack_flags_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, reset, active, flags, (long long)n, words);
  return check_launch("pack_flags");
}

int rglru_hip_mask_rows(const void* src, const uint8_t* active, void* dst, int64_t rows, int64_t D, int dtype, void* stream) {
  if (!src || !active || !dst) return fail(RGLRU_E_ARG, "mask_rows: null pointer");
  if (dtype != RGLRU_F32 && dtype != RGLRU_BF16) return fail(RGLRU_E_ARG, "mask_rows: unknown dtype %d", dtype);
  if (rows <= 0 || D <= 0) return fail(RGLRU_E_ARG, "mask_rows: empty shape");
  const int64_t es = dtype == RGLRU_BF16 ? 2 : 4, row_bytes = D * es;
  const bool vec = row_bytes % 16 == 0 && (uintptr_t)src % 16 == 0 && (uintptr_t)dst % 16 == 0;
  const int64_t per_row = vec ? row_bytes / 16 : D;
  if (per_row >= (1ll << 31) || rows >= (1ll << 40) / D) return fail(RGLRU_E_UNSUPPORTED, "mask_rows: too large");
  MaskRowsArgs a{src, active, dst, (long long)rows, (int)per_row, src == dst};
  long long blocks = (rows * per_row + 1023) / 1024; if (blocks > 8ll * num_compute_units()) blocks = 8ll * num_compute_units();
  const dim3 grid((unsigned)(blocks < 1 ? 1 : blocks));
  hipStream_t s = (hipStream_t)stream;
  if (vec) hipLaunchKernelGGL((mask_rows_kernel<f32x4>), grid, dim3(256), 0, s, a);
  else if (es == 2) hipLaunchKernelGGL((mask_rows_kernel<short>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((mask_rows_kernel<float>), grid, dim3(256), 0, s, a);
  return check_launch("mask_rows");
}

static int pack_args(const char* who, PackArgs& a, const int32_t* counts, int64_t B, int64_t T, int64_t packed) {
  if (!counts) return fail(RGLRU_E_ARG, "%s: null pointer", who);
  if (B <= 0 || T <= 0 || packed <= 0) return fail(RGLRU_E_ARG, "%s: empty shape", who);
  if (B * T >= (1ll << 30) || packed >= (1ll << 30)) return fail(RGLRU_E_UNSUPPORTED, "%s: too large", who);
  a.counts = counts; a.B = (int)B; a.T = (int)T; a.packed = (int)packed; a.chunks = (int)((T + kPackTokens - 1) / kPackTokens);
  return RGLRU_OK;
}
static int pack_array(const char* who, PackArgs& a, int i, const void* src, void* dst, int64_t bytes) {
  if (!src || !dst) return fail(RGLRU_E_ARG, "%s: null pointer", who);
  if (bytes <= 0 || bytes % 16 || (uintptr_t)src % 16 || (uintptr_t)dst % 16) return fail(RGLRU_E_UNSUPPORTED, "%s: rows must be whole 16-byte vectors", who);
  if (bytes >= (1ll << 28)) return fail(RGLRU_E_UNSUPPORTED, "%s: too large", who);
  a.src[i] = (const f32x4*)src; a.dst[i] = (f32x4*)dst; a.per_row[i] = (int)(bytes / 16);
  return RGLRU_OK;
}

int rglru_hip_pack_rows(const int32_t* counts, const void* src0, void* dst0, int64_t bytes0, const void* src1, void* dst1, int64_t bytes1,
                        int64_t* pos, uint8_t* flags, int64_t B, int64_t T, int64_t packed, void* stream) {
  PackArgs a;
  memset(&a, 0, sizeof(a));
  int rc = pack_args("pack_rows", a, counts, B, T, packed);
  if (!rc) rc = pack_array("pack_rows", a, 0, src0, dst0, bytes0);
  if (!rc && dst1) rc = pack_array("pack_rows", a, 1, src1, dst1, bytes1);
  if (rc) return rc;
  if (!pos != !flags) return fail(RGLRU_E_ARG, "pack_rows: positions and flags go together");
  a.pos = (long long*)pos; a.flags = flags;
  const long long blocks = (long long)(B + 1) * a.chunks;
  hipLaunchKernelGGL((pack_rows_kernel<true>), dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, a);
  return check_launch("pack_rows");
}

int rglru_hip_unpack_rows(const int32_t* counts, const void* src, void* dst, int64_t bytes, int64_t B, int64_t T, int64_t packed, void* stream) {
  PackArgs a;
  memset(&a, 0, sizeof(a));
  int rc = pack_args("unpack_rows", a, counts, B, T, packed);
  if (!rc) rc = pack_array("unpack_rows", a, 0, src, dst, bytes);
  if (rc) return rc;
  hipLaunchKernelGGL((pack_rows_kernel<false>), dim3((unsigned)(B * a.chunks)), dim3(256), 0, (hipStream_t)stream, a);
  return check_launch("unpack_rows");
}

int rglru_hip_conv_carry(const void* u, int64_t u_stride, const void* state, const int32_t* rows, void* new_state, int64_t B, int64_t T,
                         int64_t W, int64_t K, int dtype, void* stream) {
  if (!u || !rows || !new_state) return fail(RGLRU_E_ARG, "conv_carry: null pointer");
  if (dtype != RGLRU_F32 && dtype != RGLRU_BF16) return fail(RGLRU_E_ARG, "conv_carry: unknown dtype %d", dtype);
  if (B <= 0 || T <= 0 || W <= 0 || K < 2 || u_stride < W) return fail(RGLRU_E_ARG, "conv_carry: bad shape");
  const long long n = B * (K - 1) * W, blocks = (n + 255) / 256;
  if (blocks >= (1ll << 31) || T >= (1ll << 30)) return fail(RGLRU_E_UNSUPPORTED, "conv_carry: too large");
  CarryArgs a{u, state, rows, new_state, (long long)u_stride, (int)B, (int)T, (int)W, (int)K};
  hipStream_t s = (hipStream_t)stream;
  if (dtype == RGLRU_BF16) hipLaunchKernelGGL((conv_carry_kernel<__bf16>), dim3((unsigned)blocks), dim3(256), 0, s, a);
  else hipLaunchKernelGGL((conv_carry_kernel<float>), dim3((unsigned)blocks), dim3(256), 0, s, a);
  return check_launch("conv_carry");
}

}  // extern "C"

// Linear layers of a single-token step of the recurrent block (griffin/griffin.py:379-389 with one token per row): the
// two input projections with everything in front of the RG-LRU step (positions, causal convolution against the carried
// rows, shifted cache) in one launch, and the output projection.
//
// A decode step multiplies a few rows by matrices of a few megabytes: latency, not arithmetic.  A workgroup owns
// 16 CT output features x 16 RT rows and its four waves split the contraction, taking turns by steps of 64 bytes per
// row, so the four together read whole cache lines and each has all operands of a batch of steps in flight at once;
// the partial tiles meet in LDS.  Operands go from memory straight into MFMA fragments (16 rows x 64 bytes per load
// instruction, what the texture path takes at full rate).
//
// Measured (MI355X, eager, one token of RMSNorm + RecurrentBlock(768, 1024)): see decode_project / decode_linear below.
#include "rglru_fused.h"
#include "rglru_rows.h"

namespace rglru {

struct DecodeLinearArgs {
  const void* x; long long ldx;                 // [B, K] rows ldx elements apart
  const void* w[2]; const void* bias[2];        // one or two weight matrices [N, K], each with its bias or null
  void* y; long long ldy;                       // plain epilogue: [B, N] (of the second matrix in the projection)
  const unsigned char* active;                  // plain epilogue: rows with a zero byte are written as zeros (or null)
  int B, N, K, tiles;                           // tiles: column tiles per matrix
  // projection epilogue of the first matrix (see rglru_hip_decode_prepare for the meaning)
  const void* state; const void* taps; const void* conv_bias;
  const long long* prev_pos; const long long* seg_pos;
  void* x_conv; void* new_state; long long* new_pos; unsigned char* flags;
  int taps_count;
};

template <typename IO> struct SkinnyMma;
template <> struct SkinnyMma<__bf16> {
  static constexpr int STEP = 32;               // K elements per step: 8 per lane, four lane groups
  static RGLRU_DEVICE void mma(f32x4& acc, const bf16x8& a, const bf16x8& b) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
  }
};
template <> struct SkinnyMma<float> {
  static constexpr int STEP = 16;               // 4 per lane: element j of all lanes forms one K = 4 product
  static RGLRU_DEVICE void mma(f32x4& acc, const f32x4& a, const f32x4& b) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], acc, 0, 0, 0);
  }
};

constexpr int kMaxTaps = 4;

template <typename IO, int RT, int CT, bool PROJECT>
__global__ __launch_bounds__(kThreads) void decode_linear_kernel(DecodeLinearArgs p) {
  typedef typename Io<IO>::Frag Frag;
  typedef SkinnyMma<IO> M;
  constexpr int HW = Io<IO>::HW;
  constexpr int ROWS = 16 * RT, COLS = 16 * CT, ELEMS = ROWS * COLS / kThreads;
  constexpr int BATCH = RT * CT == 1 ? 6 : RT * CT == 2 ? 4 : 2;            // steps whose operands are in flight together
  __shared__ float red[kWaves][ROWS][COLS + 1];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, q = lane >> 4;
  const int which = PROJECT && (int)blockIdx.x >= p.tiles ? 1 : 0;
  const int col0 = ((int)blockIdx.x - which * p.tiles) * COLS;
  const long long row0 = (long long)blockIdx.y * ROWS;
  const bool conv = PROJECT && which == 0;

  // Epilogue operands of the elements this thread finishes: carried rows, taps, positions.
  int er[ELEMS], ec[ELEMS];
  bool eok[ELEMS];
#pragma unroll
  for (int i = 0; i < ELEMS; ++i) {
    const int e = (int)threadIdx.x + i * kThreads;
    er[i] = e / COLS; ec[i] = e % COLS;
    eok[i] = row0 + er[i] < p.B && col0 + ec[i] < p.N;
  }
  // All of them are loaded on every path, from x where there is no such tensor (the value is not used then): a load under
  // a condition of its own waits for its data before the next one is issued.
  IO hist[ELEMS][kMaxTaps - 1], tap[ELEMS][kMaxTaps], cbias[ELEMS], bias[ELEMS];
  unsigned char act[ELEMS];
  long long before[ELEMS], explicit_pos[ELEMS];
  const int K1 = p.taps_count - 1;
  const unsigned char* act_src = p.active ? p.active : (const unsigned char*)p.x;
  const IO* bias_src = (const IO*)(p.bias[which] ? p.bias[which] : p.x);
  const long long* before_src = p.prev_pos ? p.prev_pos : (const long long*)p.x;
  const long long* pos_src = p.seg_pos ? p.seg_pos : (const long long*)p.x;
  const IO* state_src = (const IO*)(p.state ? p.state : p.x);
  const IO* cbias_src = (const IO*)(p.conv_bias ? p.conv_bias : p.x);
  auto request = [&]() {
#pragma unroll
    for (int i = 0; i < ELEMS; ++i) {
      const long long b = eok[i] ? row0 + er[i] : 0;
      const int c = eok[i] ? col0 + ec[i] : 0;
      act[i] = act_src[p.active ? b : 0];
      bias[i] = bias_src[p.bias[which] ? c : 0];
      if (conv) {
        before[i] = before_src[p.prev_pos ? b : 0];
        explicit_pos[i] = pos_src[p.seg_pos ? b : 0];
        cbias[i] = cbias_src[p.conv_bias ? c : 0];
#pragma unroll
        for (int j = 0; j < kMaxTaps; ++j) {
          if (j < kMaxTaps - 1) hist[i][j] = state_src[p.state && j < K1 ? (b * K1 + j) * p.N + c : 0];
          tap[i][j] = ((const IO*)p.taps)[(long long)c * p.taps_count + (j < p.taps_count ? j : 0)];
        }
      }
    }
  };
  if constexpr (ELEMS <= 2) request();           // with more of them they would take the registers of the products

  // Products.  Rows and columns past the end read the last one that exists; K past the end reads zero.
  const IO* xr[RT];
  const IO* wr[CT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const long long r = row0 + 16 * t + n;
    xr[t] = (const IO*)p.x + (r < p.B ? r : p.B - 1) * p.ldx;
  }
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    const int c = col0 + 16 * t + n;
    wr[t] = (const IO*)p.w[which] + (long long)(c < p.N ? c : p.N - 1) * p.K;
  }
  f32x4 acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (p.K + M::STEP - 1) / M::STEP;
  for (int s0 = wave; s0 < steps; s0 += kWaves * BATCH) {
    Frag xa[BATCH][RT], wb[BATCH][CT];
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      const int k = (s0 + u * kWaves) * M::STEP;
      const int kk = row_vector(k, q, HW, p.K);                             // K is a multiple of a lane's vector
#pragma unroll
      for (int t = 0; t < CT; ++t) wb[u][t] = *reinterpret_cast<const Frag*>(wr[t] + kk);
#pragma unroll
      for (int t = 0; t < RT; ++t) xa[u][t] = *reinterpret_cast<const Frag*>(xr[t] + kk);
    }
    __builtin_amdgcn_sched_barrier(0);           // the whole batch in flight before the first product
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      if ((s0 + u * kWaves) * M::STEP + q * HW >= p.K) {                    // both: zero times what is not a number would count
#pragma unroll
        for (int t = 0; t < RT; ++t) xa[u][t] = Io<IO>::zero();
#pragma unroll
        for (int t = 0; t < CT; ++t) wb[u][t] = Io<IO>::zero();
      }
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) M::mma(acc[i][j], xa[u][i], wb[u][j]);
    }
  }
  if constexpr (ELEMS > 2) request();
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[wave][16 * i + 4 * q + v][16 * j + n] = acc[i][j][v];
  __syncthreads();

#pragma unroll
  for (int i = 0; i < ELEMS; ++i) {
    if (!eok[i]) continue;
    const long long b = row0 + er[i];
    const int c = col0 + ec[i];
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s += red[w][er[i]][ec[i]];
    if (p.bias[which]) s += (float)bias[i];
    const bool live = p.active ? act[i] != 0 : true;
    if (!conv) {
      ((IO*)p.y)[b * p.ldy + c] = (IO)(PROJECT || live ? s : 0.f);
      continue;
    }
    // griffin/griffin.py:309-358 (position), :474-510 (convolution over the carried rows and this token)
    const float cur = (float)(IO)s;                                          // the projection as stored
    const long long prev = p.prev_pos ? before[i] : -1;
    const long long pos = p.seg_pos ? explicit_pos[i] : prev + (live ? 1 : 0);
    const bool padded = p.active != nullptr;
    const bool fresh = padded && live && pos == 0;                           // a document starts: the window is cleared
    float a = p.conv_bias ? (float)cbias[i] : 0.f;
    float h[kMaxTaps - 1];
#pragma unroll
    for (int j = 0; j < kMaxTaps - 1; ++j) h[j] = (p.state && j < K1 && !fresh) ? (float)hist[i][j] : 0.f;
    float last = 0.f;
#pragma unroll
    for (int j = 0; j < kMaxTaps; ++j) if (j == K1) last = (float)tap[i][j];
    if (padded || pos >= 0) a = fmaf(cur, last, a);
#pragma unroll
    for (int lag = 1; lag < kMaxTaps; ++lag) {
      if (lag > K1 || !(padded || pos >= lag)) continue;
      float t = 0.f, v = 0.f;
#pragma unroll
      for (int j = 0; j < kMaxTaps - 1; ++j) if (j == K1 - lag) { t = (float)tap[i][j]; v = h[j]; }
      a = fmaf(v, t, a);
    }
    ((IO*)p.x_conv)[b * p.N + c] = (IO)(live ? a : 0.f);
#pragma unroll
    for (int j = 0; j < kMaxTaps - 1; ++j) {
      if (j >= K1) continue;
      const float shifted = j + 1 < K1 ? h[j + 1 < kMaxTaps - 1 ? j + 1 : 0] : cur;
      ((IO*)p.new_state)[(b * K1 + j) * p.N + c] = (IO)(live ? shifted : h[j]);
    }
    if (c == 0) {
      p.new_pos[b] = live ? pos : prev;
      p.flags[b] = (unsigned char)((live && pos == 0 ? RGLRU_FLAG_RESET : 0u) | (live ? 0u : RGLRU_FLAG_INACTIVE));
    }
  }
}

// Rows per workgroup: as many as there are up to 64, so that a weight fragment is used for all of them; two column tiles
// where the launch still fills the chip (each x fragment is then used twice).
template <typename IO, bool PROJECT>
static void launch_decode_linear(DecodeLinearArgs& a, hipStream_t s) {
  const int matrices = PROJECT ? 2 : 1;
  auto go = [&](auto kernel, int rows, int cols) {
    a.tiles = (a.N + cols - 1) / cols;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(a.tiles * matrices), (unsigned)((a.B + rows - 1) / rows)), dim3(kThreads), 0, s, a);
  };
  const long long wide = (long long)((a.N + 31) / 32) * matrices * ((a.B + 63) / 64);
  if (a.B <= 16) go(decode_linear_kernel<IO, 1, 1, PROJECT>, 16, 16);
  else if (a.B <= 32) go(decode_linear_kernel<IO, 2, 1, PROJECT>, 32, 16);
  else if (wide < num_compute_units()) go(decode_linear_kernel<IO, 4, 1, PROJECT>, 64, 16);
  else go(decode_linear_kernel<IO, 4, 2, PROJECT>, 64, 32);
}

static int decode_linear_check(const char* what, int64_t B, int64_t N, int64_t K, int64_t ldx, const void* x, const void* w, int dtype) {
  if (dtype != RGLRU_F32 && dtype != RGLRU_BF16) return fail(RGLRU_E_ARG, "%s: unknown dtype %d", what, dtype);
  if (B <= 0 || N <= 0 || K <= 0) return fail(RGLRU_E_ARG, "%s: sizes must be positive", what);
  const int64_t es = dtype == RGLRU_BF16 ? 2 : 4;
  if ((K * es) % 16 || (ldx * es) % 16 || ((uintptr_t)x % 16) || ((uintptr_t)w % 16))
    return fail(RGLRU_E_UNSUPPORTED, "%s: rows must start on 16-byte boundaries", what);
  if (ldx < K) return fail(RGLRU_E_ARG, "%s: row stride smaller than the row", what);
  if (B >= (1ll << 22) || N >= (1ll << 24) || K >= (1ll << 24)) return fail(RGLRU_E_UNSUPPORTED, "%s: too large", what);
  return RGLRU_OK;
}

}  // namespace rglru

using namespace rglru;

extern "C" {

int rglru_hip_decode_linear(const void* x, int64_t x_stride, const void* w, const void* bias, const uint8_t* active, void* y,
                            int64_t B, int64_t N, int64_t K, int dtype, void* stream) {
  if (!x || !w || !y) return fail(RGLRU_E_ARG, "decode_linear: null pointer");
  int rc = decode_linear_check("decode_linear", B, N, K, x_stride, x, w, dtype);
  if (rc) return rc;
  DecodeLinearArgs a;
  memset(&a, 0, sizeof(a));
  a.x = x; a.ldx = x_stride; a.w[0] = w; a.bias[0] = bias; a.active = active; a.y = y; a.ldy = N;
  a.B = (int)B; a.N = (int)N; a.K = (int)K;
  if (dtype == RGLRU_BF16) launch_decode_linear<__bf16, false>(a, (hipStream_t)stream);
  else launch_decode_linear<float, false>(a, (hipStream_t)stream);
  return check_launch("decode_linear");
}

int rglru_hip_decode_project(const void* x, int64_t x_stride, const void* w_x, const void* b_x, const void* w_y, const void* b_y,
                             const void* conv_state, const void* taps, const void* conv_bias, const int64_t* prev_pos,
                             const int64_t* segment_pos, const uint8_t* active, void* x_conv, void* v, void* new_conv_state,
                             int64_t* new_pos, uint8_t* flags, int64_t B, int64_t D, int64_t W, int64_t K, int dtype,
                             void* stream) {
  if (!x || !w_x || !w_y || !taps || !x_conv || !v || !new_pos || !flags || (K > 1 && !new_conv_state))
    return fail(RGLRU_E_ARG, "decode_project: null pointer");
  int rc = decode_linear_check("decode_project", B, W, D, x_stride, x, w_x, dtype);
  if (rc) return rc;
  if ((uintptr_t)w_y % 16) return fail(RGLRU_E_UNSUPPORTED, "decode_project: rows must start on 16-byte boundaries");
  if (K < 1 || K > kMaxTaps) return fail(RGLRU_E_UNSUPPORTED, "decode_project: kernel size %lld", (long long)K);
  DecodeLinearArgs a;
  memset(&a, 0, sizeof(a));
  a.x = x; a.ldx = x_stride; a.w[0] = w_x; a.w[1] = w_y; a.bias[0] = b_x; a.bias[1] = b_y; a.active = active; a.y = v; a.ldy = W;
  a.B = (int)B; a.N = (int)W; a.K = (int)D;
  a.state = conv_state; a.taps = taps; a.conv_bias = conv_bias; a.prev_pos = (const long long*)prev_pos;
  a.seg_pos = (const long long*)segment_pos; a.x_conv = x_conv; a.new_state = new_conv_state; a.new_pos = (long long*)new_pos;
  a.flags = flags; a.taps_count = (int)K;
  if (dtype == RGLRU_BF16) launch_decode_linear<__bf16, true>(a, (hipStream_t)stream);
  else launch_decode_linear<float, true>(a, (hipStream_t)stream);
  return check_launch("decode_project");
}

}  // extern "C"

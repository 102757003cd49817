// Gradients of the Linear layers in bf16 (input: one or two products into one result; weight: contraction over the tokens), whose
// operands do not both lie with the contraction index contiguous.
#include <hip/hip_runtime.h>

#include "../../include/rglru_hip.h"
#include "rglru_linear.h"

namespace rglru {

// Slice of one operand, moved from memory to LDS without passing through registers.  T: a line of the slice is one contraction index
// (ROWS result indices), else one result index (BK contraction indices).  Lines lie without padding, so their 16-byte vectors are
// permuted against bank conflicts: vector c of line l is at place c ^ swizzle(l).  Lines of 128 (64) bytes are read by rows, sixteen
// at a time, which the LDS serves together: two (four) of them fill its banks, so every two (four) have another permutation.  Lines of
// ROWS results are read by the transposing loads, four lines of 64 bytes at a time: these land in different quarters of the banks.
template <bool T, int ROWS, int BK, int THREADS>
struct SliceTile {
  static constexpr int VPL = (T ? ROWS : BK) / 8, LINES = T ? BK : ROWS, NV = LINES * VPL / THREADS, kBytes = ROWS * BK * 2;
  static constexpr int kLineStep = THREADS / VPL;              // lines between a thread's vectors
  static_assert(LINES * VPL % THREADS == 0 && THREADS % VPL == 0 && kLineStep % 16 == (T ? kLineStep % 16 : 0), "a thread's vectors lie in one column");
  static_assert(!T || kLineStep % 4 == 0, "... and have one permutation");
  unsigned off, step;                                          // byte offset of the thread's first vector; bytes between its vectors
  int c, line;                                                 // place of the first vector in the slice
  static RGLRU_DEVICE unsigned swizzle(int l) { return T ? (VPL == 8 ? (unsigned)(l & 2) << 1 : (unsigned)(l & 3) << 2) : VPL == 8 ? (unsigned)(l >> 1) & 7u : (unsigned)(l >> 2) & 3u; }
  // limit: result indices left
  RGLRU_DEVICE void setup(int tid, long long ld, int limit) {
    line = tid / VPL;
    c = (tid % VPL) ^ (int)swizzle(line);
    off = !T || c * 8 < limit ? (unsigned)line * (unsigned)(ld * 2) + (unsigned)c * 16u : kOutOfRange;
    step = (unsigned)kLineStep * (unsigned)(ld * 2);
  }
  // bytes from the slice's first element to the end of its last line
  static RGLRU_DEVICE unsigned extent(long long ld, int k_left, int limit) {
    const int lines = T ? (k_left < BK ? k_left : BK) : (limit < ROWS ? limit : ROWS);
    return k_left > 0 ? (unsigned)((long long)lines * ld) * 2u : 0u;
  }
  // Vector i of the slice behind `r` to LDS at `lds` (the wave's part of the slice, uniform).  The compiler neither counts these loads nor
  // knows their hazards: the caller waits for them, and gives the descriptor its wait states.
  RGLRU_DEVICE void request(int i, i32x4 r, int k_left, unsigned lds, bool live = true) const {
    const bool inside = (T || c * 8 < k_left) && live;
    const unsigned at = inside && off != kOutOfRange ? off + (unsigned)i * step : kOutOfRange;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :: "s"(lds + (unsigned)(i * THREADS) * 16u), "v"(at), "s"(r) : "memory", "m0");
  }
  // fragment of 32 result indices from `first`, sixteen contraction indices from 16 kg
  static RGLRU_DEVICE bf16x8 fragment(const unsigned char* lds, int first, int kg, int lane) {
    if constexpr (!T) {
      const unsigned r = lane & 31, hf = lane >> 5;
      return *reinterpret_cast<const bf16x8*>(lds + ((unsigned)first + r) * (unsigned)(BK * 2) + (((2u * kg + hf) ^ swizzle(r)) * 16u));
    } else {                                                   // as lds_transposed_frag, with the permutation
      typedef __attribute__((address_space(3))) bf16x4_lds* lds_ptr_t;
      const int i = lane & 15, g = lane >> 4, l = kg * 16 + 8 * (g >> 1) + (i >> 2);
      const unsigned v = (unsigned)(first / 8 + 2 * (g & 1) + ((i & 3) >> 1));
      const unsigned char* src = lds + l * (ROWS * 2) + ((v ^ swizzle(l)) * 16u) + (i & 1) * 8;
      const bf16x4_lds lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_ptr_t)(src));
      const bf16x4_lds hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_ptr_t)(src + 4 * (ROWS * 2)));
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  }
};

RGLRU_DEVICE i32x4 uniform_rsrc(const void* base, unsigned bytes) {
  const unsigned long long at = (unsigned long long)base;
  i32x4 r;
  r[0] = __builtin_amdgcn_readfirstlane((int)(unsigned)at);
  r[1] = __builtin_amdgcn_readfirstlane((int)((unsigned)(at >> 32) & 0xffffu));
  r[2] = __builtin_amdgcn_readfirstlane((int)bytes);
  r[3] = 0x00020000;
  return r;
}

// Tiles of EDGE x EDGE by WM x WN waves.  Two forms of the loop over the slices:
//  * EDGE 64 and 128: slices of 64 contraction indices, fetched one (128) or two (64) ahead; fragments one K group ahead inside a
//    slice.  Two or three workgroups a compute unit cover each other's barriers.
//  * EDGE 256: one workgroup of eight waves a compute unit, so nothing else covers a wait: slices of 32, fetched three ahead, fragments one
//    K group ahead across slices, and reads and requests issued between the products.
// us, slices through registers (the kernels before) -> here: input gradient 2331 x 768 of two segments of 1024 20.7 -> 16.7, 8704 40.2 -> 30.9, 8704
// x 1024 x 768 29.8 -> 22.7; weight gradient of two of 1024 x 768 at 2331 tokens 27.4 -> 17.9, 8704 64.5 -> 39.1, 16384 114 -> 58.5 (BLAS library:
// 51.6 where the tokens divide into its batches, 66 at 8704, where they do not).
// What bounds them: 256 x 256 keeps the matrix units 63 % busy (counters, 16384 x 2048 x 2048), at a clock that the load draws down
// to 1.6-1.8 GHz; LDS reads are 768 of a slice's 1024 matrix clocks.  128 x 128 reads a third more of LDS per product.
template <bool TA, int EDGE, int WM, int WN, int BK, int STAGES>
__global__ __launch_bounds__(64 * WM * WN, 2) void linear16_kernel(LinearArgs p) {
  constexpr bool TB = true, AHEAD = EDGE == 256;
  constexpr int THREADS = 64 * WM * WN, MI = EDGE / WM / 32, NI = EDGE / WN / 32, KGS = BK / 16;
  typedef SliceTile<TA, EDGE, BK, THREADS> TileA;
  typedef SliceTile<TB, EDGE, BK, THREADS> TileB;
  constexpr int kStage = TileA::kBytes + TileB::kBytes, LOADS = TileA::NV + TileB::NV;
  constexpr int kRow = EDGE / WN + 4, kOut = WM * WN * 32 * kRow * 4;          // epilogue: 32 rows of a wave's tile, fp32
  __shared__ __attribute__((aligned(1024))) unsigned char lds[STAGES * kStage > kOut ? STAGES * kStage : kOut];

  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, hf = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  // workgroups go to the eight XCDs round-robin; each XCD gets a contiguous run of tiles (columns fastest)
  const int per_xcd = (p.total + 7) >> 3;
  int t = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || t >= p.total) return;
  const int tn = t % p.tiles_n; t /= p.tiles_n;
  const int problem = t % p.problems; t /= p.problems;
  const int tm = t % p.tiles_m; t /= p.tiles_m;
  const int item = t % p.batch, split = t / p.batch;
  const int m0 = tm * EDGE, n0 = tn * EDGE, m_left = p.M - m0, n_left = p.N - n0;
  const int k_begin = split * p.k_per_split, k_end = (k_begin + p.k_per_split) < p.K ? (k_begin + p.k_per_split) : p.K;
  const int slices = k_end > k_begin ? (k_end - k_begin + BK - 1) / BK : 0, total = slices * p.segments;
  const bool two = p.segments > 1;
  const long long lda = p.lda, ldb = p.ldb;
  const __bf16* const a_first = (const __bf16*)p.a[TA ? problem : 0] + item * p.a_step + (TA ? k_begin * lda + m0 : m0 * lda + k_begin);
  const __bf16* const b_first = (const __bf16*)p.b[0] + item * p.b_step + k_begin * ldb + n0;
  const __bf16* const a_second = two ? (const __bf16*)p.a[1] + item * p.a_step + (TA ? k_begin * lda + m0 : m0 * lda + k_begin) : a_first;
  const __bf16* const b_second = two ? (const __bf16*)p.b[1] + item * p.b_step + k_begin * ldb + n0 : b_first;
  const unsigned char* const active = TA ? p.active : nullptr;

  TileA ta;
  TileB tb;
  ta.setup(tid, lda, m_left);
  tb.setup(tid, ldb, n_left);
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)lds + (unsigned)wave * 1024u;

  // One slice on its way: descriptors, and which of the thread's tokens take part (masked weight gradient).
  struct Slice { i32x4 ra, rb; int left; unsigned lds; };
  unsigned live = ~0u;
  auto slice_at = [&](int s, unsigned stage) {
    Slice f;
    const bool second = s >= slices;
    const int q = second ? s - slices : s, k = q * BK;
    f.left = s < total ? k_end - k_begin - k : 0;
    const long long from = s < total ? k : 0;
    f.ra = uniform_rsrc((second ? a_second : a_first) + (TA ? from * lda : from), TileA::extent(lda, f.left, m_left));
    f.rb = uniform_rsrc((second ? b_second : b_first) + from * ldb, TileB::extent(ldb, f.left, n_left));
    f.lds = __builtin_amdgcn_readfirstlane(lds0 + stage * (unsigned)kStage);
    asm volatile("s_nop 4" :: "s"(f.ra), "s"(f.rb));
    if (active) {
      const rsrc_t rl = make_rsrc(active + k_begin + from, f.left > 0 ? (unsigned)(f.left < BK ? f.left : BK) : 0u);
      live = 0u;
#pragma unroll
      for (int i = 0; i < TileA::NV; ++i)
        live |= (__builtin_amdgcn_raw_buffer_load_b8(rl, (unsigned)(ta.line + i * TileA::kLineStep), 0, 0) & 0xff) ? 1u << i : 0u;
    }
    return f;
  };
  auto request = [&](const Slice& f, int l) {
    if (l < TileA::NV) ta.request(l, f.ra, f.left, f.lds, !TA || ((live >> l) & 1u));
    else tb.request(l - TileA::NV, f.rb, f.left, f.lds + TileA::kBytes);
  };
  auto fetch = [&](int s, unsigned stage) {
    const Slice f = slice_at(s, stage);
#pragma unroll
    for (int l = 0; l < LOADS; ++l) request(f, l);
  };

  f32x16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  const int row0 = wm * (EDGE / WM), col0 = wn * (EDGE / WN);
  typedef __bf16 io4 __attribute__((ext_vector_type(4)));
  // The second operand's fragments come first in the products, so an accumulator's lane has ONE row of the result (m = r) and runs of four
  // columns (n = 8 (v / 4) + 4 hf + v % 4).
  if (p.accumulate) {
    const rsrc_t rc = make_rsrc((const __bf16*)p.c[problem] + item * p.c_step + (long long)m0 * p.ldc + n0, (unsigned)((long long)(m_left < EDGE ? m_left : EDGE) * p.ldc) * 2u);
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int n = col0 + 32 * j + 8 * g + 4 * hf, m = row0 + 32 * i + r;
          const io4 c = buf_load_four<__bf16>(rc, n < n_left ? ((unsigned)m * (unsigned)p.ldc + (unsigned)n) * 2u : kOutOfRange);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][j][4 * g + e] = (float)c[e];
        }
  }
  // column sums of A: products with ones, 32 columns to each of the waves that share them (so that no wave has much more to do)
  static_assert(MI <= WN, "a wave for every 32 columns");
  f32x16 sum;
  bf16x8 ones;
#pragma unroll
  for (int v = 0; v < 16; ++v) sum[v] = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (__bf16)1.0f;
  const bool sums = TA && p.colsum && tn == 0 && wn < MI;
  auto add_up = [&](const bf16x8 (&fa)[MI]) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
      if (wn == i) Io<__bf16>::mma(sum, ones, fa[i]);
  };

#pragma unroll
  for (int q = 0; q < STAGES - 1; ++q) fetch(q, q);
  unsigned stage = 0;
  bf16x8 fa[2][MI], fb[2][NI];
  if constexpr (!AHEAD) {
    for (int s = 0; s < total; ++s) {
      // a slice has landed when every wave has waited for its own part of it
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((STAGES - 2) * LOADS) : "memory");
      fetch(s + STAGES - 1, stage == 0 ? STAGES - 1 : stage - 1);              // read in the pass before
      const unsigned char* cur = lds + stage * (unsigned)kStage;
      auto read = [&](int kg) {
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[kg & 1][i] = TileA::fragment(cur, row0 + 32 * i, kg, lane);
#pragma unroll
        for (int j = 0; j < NI; ++j) fb[kg & 1][j] = TileB::fragment(cur + TileA::kBytes, col0 + 32 * j, kg, lane);
      };
      read(0);
#pragma unroll
      for (int kg = 0; kg < KGS; ++kg) {
        if (kg + 1 < KGS) read(kg + 1);
        __builtin_amdgcn_sched_barrier(0);                     // or the reads sink to their use, and the products wait for them
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) Io<__bf16>::mma(acc[i][j], fb[kg & 1][j], fa[kg & 1][i]);
        if (sums) add_up(fa[kg & 1]);
      }
      stage = stage + 1 == STAGES ? 0u : stage + 1;
    }
  } else {
    static_assert(STAGES >= 4, "the slice behind the current one has landed, one more is on its way");
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((STAGES - 2) * LOADS) : "memory");
#pragma unroll
    for (int i = 0; i < MI; ++i) fa[0][i] = TileA::fragment(lds, row0 + 32 * i, 0, lane);
#pragma unroll
    for (int j = 0; j < NI; ++j) fb[0][j] = TileB::fragment(lds + TileA::kBytes, col0 + 32 * j, 0, lane);
    for (int s = 0; s < total; ++s) {
      const unsigned next = stage + 1 == STAGES ? 0u : stage + 1;
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((STAGES - 3) * LOADS) : "memory");
      const Slice f = slice_at(s + STAGES - 1, stage == 0 ? STAGES - 1 : stage - 1);   // its reads ended in the pass before
      const unsigned char *cur = lds + stage * (unsigned)kStage, *nxt = lds + next * (unsigned)kStage;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kg = 0; kg < KGS; ++kg) {
        constexpr int NM = MI * NI, PER = (LOADS + KGS - 1) / KGS;
        const unsigned char* from = kg + 1 < KGS ? cur : nxt;
        const int kn = kg + 1 < KGS ? kg + 1 : 0, now = kg & 1;
        if (sums) add_up(fa[now]);
#pragma unroll
        for (int m = 0; m < NM; ++m) {
          if (m < MI) fa[now ^ 1][m] = TileA::fragment(from, row0 + 32 * m, kn, lane);
          else if (m < MI + NI) fb[now ^ 1][m - MI] = TileB::fragment(from + TileA::kBytes, col0 + 32 * (m - MI), kn, lane);
          if (m >= NM - PER && kg * PER + m - (NM - PER) < LOADS) request(f, kg * PER + m - (NM - PER));
          Io<__bf16>::mma(acc[m / NI][m % NI], fb[now][m % NI], fa[now][m / NI]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      stage = next;
    }
  }
  // nothing may land over the epilogue's staging, and every wave has read its last fragments
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  if (sums) {                                                  // all rows of the product are the sums
    const int m = row0 + 32 * wn + r;
    if (hf == 0 && m < m_left) p.colsum[((long long)split * p.problems + problem) * p.M + m0 + m] = sum[0];
  }
  // Results leave through LDS, 32 rows of the wave's tile at a time: fp32 partial sums of a split contraction, or the storage type.
  // Written through the L2s (kWriteThrough).
  float* out = reinterpret_cast<float*>(lds) + wave * 32 * kRow;
  const bool partial = TA && p.partial;
  const int ld = p.partial_ld ? p.partial_ld : p.N, rows = p.partial_ld ? p.partial_ld : p.M;
  const unsigned lines = (unsigned)(m_left < EDGE ? m_left : EDGE);
  const rsrc_t rc = partial ? make_rsrc(p.partial + ((((long long)split * p.batch + item) * p.problems + problem) * rows + m0) * ld + n0, lines * (unsigned)ld * 4u)
                            : make_rsrc((__bf16*)p.c[problem] + item * p.c_step + (long long)m0 * p.ldc + n0, lines * (unsigned)p.ldc * 2u);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 c;
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] = acc[i][j][4 * g + e];
        *reinterpret_cast<f32x4*>(out + r * kRow + 32 * j + 8 * g + 4 * hf) = c;
      }
    wave_lds_fence();
    if (partial) {
      constexpr int VPR = (EDGE / WN) / 4, ROWS = 64 / VPR;
#pragma unroll
      for (int q = 0; q < 32 / ROWS; ++q) {
        const int m = q * ROWS + lane / VPR, cv = lane % VPR, row = row0 + 32 * i + m, n = col0 + cv * 4;
        const i32x4 c = *reinterpret_cast<const i32x4*>(out + m * kRow + cv * 4);
        buf_store_b128<kWriteThrough>(c, rc, n < n_left && row < m_left ? ((unsigned)row * (unsigned)ld + (unsigned)n) * 4u : kOutOfRange);
      }
    } else {
      constexpr int VPR = (EDGE / WN) / 8, ROWS = 64 / VPR;
#pragma unroll
      for (int q = 0; q < 32 / ROWS; ++q) {
        const int m = q * ROWS + lane / VPR, cv = lane % VPR, row = row0 + 32 * i + m, n = col0 + cv * 8;
        const f32x4 lo = *reinterpret_cast<const f32x4*>(out + m * kRow + cv * 8), hi = *reinterpret_cast<const f32x4*>(out + m * kRow + cv * 8 + 4);
        bf16x8 f;
#pragma unroll
        for (int e = 0; e < 4; ++e) { f[e] = (__bf16)lo[e]; f[e + 4] = (__bf16)hi[e]; }
        if (!TA && p.active && row < m_left && !p.active[m0 + row]) f = Io<__bf16>::zero();
        buf_store_b128<kWriteThrough>(__builtin_bit_cast(i32x4, f), rc, n < n_left && row < m_left ? ((unsigned)row * (unsigned)p.ldc + (unsigned)n) * 2u : kOutOfRange);
      }
    }
    wave_lds_fence();
  }
}

template <bool TA>
static void launch(LinearArgs& a, int edge, hipStream_t s) {
  const dim3 grid((unsigned)(8 * ((a.total + 7) / 8)));
  if (edge == 256) hipLaunchKernelGGL((linear16_kernel<TA, 256, 2, 4, 32, 4>), grid, dim3(512), 0, s, a);
  else if (edge == 128) hipLaunchKernelGGL((linear16_kernel<TA, 128, 2, 2, 64, 2>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((linear16_kernel<TA, 64, 2, 2, 64, 3>), grid, dim3(256), 0, s, a);
}

void linear16_launch(LinearArgs& a, int kind, int edge, hipStream_t s) {
  a.tiles_m = (a.M + edge - 1) / edge;
  a.tiles_n = (a.N + edge - 1) / edge;
  a.total = a.tiles_m * a.tiles_n * a.problems * a.batch * a.splits;
  if (kind == RGLRU_LINEAR_WEIGHT_GRAD) launch<true>(a, edge, s);
  else launch<false>(a, edge, s);
}

}  // namespace rglru

// Matrix products of the recurrent block's Linear layers (griffin/griffin.py:379-389 and their reverse mode) on the matrix
// unit, as kernels of this library:
//
//   forward      C_i[m, n] = sum_k X[m, k] W_i[n, k] + b_i[n]         one or two weights on one input
//   input grad   C[m, n]   = sum_i sum_k A_i[m, k] W_i[k, n]          one or two products into one result
//   weight grad  C_i[m, n] = sum_k A_i[k, m] X[k, n]                  contraction over the tokens, split over workgroups;
//                            the column sums of A_i (the bias gradient) come with it
//
// Why not the BLAS library alone: a call of it costs the host 17 us, seven calls of it are a third of the host time of a
// training step of the block, which is what bounds such a step up to several thousand tokens; and it takes no row mask and
// returns no column sums.  For long products it is faster (16384 x 1024 x 768 twice in bf16: 57 us against 67 us), so callers choose by the
// size of the product.
//
// Here: fp32, and the forward in bf16 (the gradients in bf16: rglru_linear16.hip).  A workgroup of four waves owns a BM x BN tile of C; K is
// walked in slices of 128 bytes, one barrier a slice.  Where both operands
// lie with their contraction index contiguous (forward) a slice goes from memory to LDS directly (DirectTile), one slice ahead
// or (64 x 64) two.  Otherwise it goes through registers (requested one slice ahead) into one of two LDS buffers: an
// operand with its contraction index contiguous is read back as 16-byte rows (row stride 144 bytes: no bank conflicts); one that
// lies the other way round is read element by element.
// Edges of M, N and K are masked through the offsets of buffer loads, so any size works as long as rows are whole 16-byte
// vectors.
// What bounds it, forward: with slices through registers the LDS writes (13.8 clocks a KB on a compute unit, reads 4.3) were most
// of the 0.9 us a slice.  Direct, two products of 2331 x 1024 x 768 in bf16 take 14.8 us: 1.5 us launch, 3 us until the first slice is
// there, 4 us for the results (timing builds), the rest MFMAs of the 48 compute units that have two of the 304 tiles.  us before ->
// with direct slices, bias asked for in front of them: 2331 x 2 x 1024 x 768 20.3 -> 14.8, x 768 x 1024 11.6 -> 9.8; 4096 x 2 x 1024 x 768
// 22.4 -> 18.9; 8192 41.5 -> 34.4; 16384 x 2048 x 2048 166 -> 136 (1012 TFLOP/s).  fp32, bound by its MFMAs: 34.1 -> 32.8 at 800
// x 2 x 1024 x 768, 389 -> 387 at 16384.  Three or four slices of 128 x 128 (one workgroup a compute unit): 23.0, 16.4 against 16.6;
// both operands' tiles per XCD in another order: no change.  Sizes of the tiles: forward16_plan.
// The gradients, through registers: the order of a slice below, operand pointers outside the loop and results staged four columns
// at a time took the gate gradients of B4 T1024 W1024 in fp32 from 39.5 to 37 us; more slices in flight (3, 4 or 6) gained nothing.
#include <hip/hip_runtime.h>

#include <cstring>
#include <initializer_list>
#include <type_traits>

#include "rglru_device.h"
#include "rglru_host.h"
#include "rglru_layout.h"
#include "rglru_linear.h"

namespace rglru {

// Tile of one operand: ROWS rows of the result's index (m or n) x BK of the contraction index.  T: in memory (and in LDS) a row
// is one contraction index, else one result index.
template <typename IO, bool T, int ROWS, int THREADS>
struct OperandTile {
  static constexpr int RING = 2;     // slices on their way from memory
  typedef Io<IO> Tr;
  typedef typename Tr::Frag Frag;
  static constexpr int HW = Tr::HW, BK = 8 * HW;                              // 128 bytes
  static constexpr int kLines = T ? BK : ROWS, kLineElems = T ? ROWS : BK;    // memory rows of the tile, elements of each
  // transposed: the two halves of a wave read rows four apart, half the banks away
  static constexpr int kStride = T ? ROWS + 8 : BK + HW;
  static constexpr int kElems = kLines * kStride;
  static constexpr int VPR = kLineElems / HW, NV = kLines * VPR / THREADS;
  static_assert(kLines * VPR % THREADS == 0, "whole vectors per thread");
  Frag v[RING][NV];
  unsigned off[NV];                  // lane offsets in bytes, kOutOfRange past the last result index
  unsigned live[RING];               // masked weight gradient: bit i = the token of vector i takes part

  RGLRU_DEVICE void setup(int tid, long long ld, int limit) {               // limit: result indices left in the tile
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + i * THREADS, line = idx / VPR, cv = idx - line * VPR;
      const int index = T ? cv * HW : line;
      off[i] = index < limit ? (unsigned)((long long)line * ld * (int)sizeof(IO)) + (unsigned)(cv * HW) * (unsigned)sizeof(IO) : kOutOfRange;
    }
    live[0] = live[1] = ~0u;
  }
  // q: slot of the ring; base: first element of the slice (uniform); k_left: contraction indices left
  RGLRU_DEVICE void request(int q, const IO* base, long long ld, int k_left, int limit, int tid, const unsigned char* active = nullptr) {
    const int lines = T ? (k_left < BK ? (k_left < 0 ? 0 : k_left) : BK) : (limit < ROWS ? limit : ROWS);
    const rsrc_t r = make_rsrc(base, k_left > 0 ? (unsigned)((long long)lines * ld) * (unsigned)sizeof(IO) : 0u);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      unsigned o = off[i];
      if constexpr (!T) {
        const int cv = (tid + i * THREADS) % VPR;
        if (cv * HW >= k_left) o = kOutOfRange;
      }
      v[q][i] = buf_load_frag<Frag>(r, o);
    }
    if (T && active) {
      const rsrc_t ra = make_rsrc(active, (unsigned)lines);
      live[q] = 0u;
#pragma unroll
      for (int i = 0; i < NV; ++i)
        live[q] |= (__builtin_amdgcn_raw_buffer_load_b8(ra, (unsigned)((tid + i * THREADS) / VPR), 0, 0) & 0xff) ? 1u << i : 0u;
    }
  }
  RGLRU_DEVICE void deposit(int q, IO* lds, int tid, bool masked = false) const {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + i * THREADS, line = idx / VPR, cv = idx - line * VPR;
      Frag f = v[q][i];
      if (T && masked && !((live[q] >> i) & 1u)) f = Tr::zero();
      *reinterpret_cast<Frag*>(lds + line * kStride + cv * HW) = f;
    }
  }
  // fragment of 32 result indices from `first`, K group kg
  static RGLRU_DEVICE Frag fragment(const IO* lds, int first, int kg, int lane) {
    const int r = lane & 31, hf = lane >> 5;
    if constexpr (!T) {
      return *reinterpret_cast<const Frag*>(lds + (first + r) * kStride + kg * Tr::KG + hf * HW);
    } else {
      static_assert(sizeof(IO) == 4, "16-bit types: rglru_linear16.hip");
      Frag f;
#pragma unroll
      for (int i = 0; i < HW; ++i) f[i] = lds[(kg * Tr::KG + hf * HW + i) * kStride + first + r];
      return f;
    }
  }
};

constexpr int kLinearThreads = 256;

// Tile of an operand whose rows are result indices, moved from memory to LDS without passing through registers (1 KB a wave
// instruction: eight rows of 128 bytes).  The rows lie without padding, so the 16-byte vectors of row r are permuted: vector c is at
// place c ^ ((r / 2) % 8), and the sixteen rows that the LDS serves at once fall on different banks.
template <typename IO, int ROWS>
struct DirectTile {
  typedef Io<IO> Tr;
  typedef typename Tr::Frag Frag;
  static constexpr int HW = Tr::HW, BK = 8 * HW, kBytes = ROWS * 128, NV = ROWS / 32;
  unsigned off, cv;                  // the lane's first vector: offset in memory, its place in the slice
  unsigned place[4];                 // the lane's vector of a fragment in LDS, by K group
  RGLRU_DEVICE void setup(int wave, int lane, long long ld) {
    const unsigned row = (unsigned)wave * 8u + (unsigned)(lane >> 3);
    cv = (unsigned)(lane & 7) ^ ((row >> 1) & 7u);
    off = row * (unsigned)(ld * (int)sizeof(IO)) + cv * 16u;
    const unsigned r = lane & 31, hf = lane >> 5;
#pragma unroll
    for (unsigned kg = 0; kg < 4; ++kg) place[kg] = r * 128u + (((2u * kg + hf) ^ ((r >> 1) & 7u)) * 16u);
  }
  // Slice at `base` with k_left contraction indices into LDS at byte address `lds`; rows past
  // `limit` and indices past k_left become zeros, as masked loads do everywhere.  The compiler neither counts these loads nor knows
  // their hazards: the caller waits for them, and the descriptor has its wait states here.
  RGLRU_DEVICE void request(const IO* base, long long ld, int k_left, int limit, unsigned lds, int wave) const {
    const int lines = limit < ROWS ? limit : ROWS;
    const unsigned long long at = (unsigned long long)base;
    i32x4 r;
    r[0] = __builtin_amdgcn_readfirstlane((int)(unsigned)at);
    r[1] = __builtin_amdgcn_readfirstlane((int)((unsigned)(at >> 32) & 0xffffu));
    r[2] = __builtin_amdgcn_readfirstlane(k_left > 0 ? (int)((unsigned)((long long)lines * ld) * (unsigned)sizeof(IO)) : 0);
    r[3] = 0x00020000;
    asm volatile("s_nop 4" :: "s"(r));
    const unsigned step = 32u * (unsigned)(ld * (int)sizeof(IO));
    const unsigned first = (int)cv * HW < k_left ? off : kOutOfRange;
    const unsigned to = __builtin_amdgcn_readfirstlane(lds + (unsigned)wave * 1024u);
#pragma unroll
    for (int i = 0; i < NV; ++i)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                   :: "s"(to + (unsigned)i * 4096u), "v"(first + (unsigned)i * step), "s"(r) : "memory", "m0");
  }
  RGLRU_DEVICE Frag fragment(const unsigned char* lds, int first, int kg) const {
    return *reinterpret_cast<const Frag*>(lds + first * 128 + place[kg]);
  }
};

// DIRECT: both operands' rows are result indices and go to LDS directly (DirectTile).  STAGES: slices of them in LDS; two and three workgroups
// on a compute unit (64 x 64 with two or four slices: 11.8 and 10.2 us for 10).
template <typename IO, bool TA, bool TB, int BM, int BN, int STAGES = BN == 64 ? 3 : 2, bool DIRECT = !TA && !TB>
struct LinearTile {
  typedef Io<IO> Tr;
  typedef typename Tr::Frag Frag;
  typedef OperandTile<IO, TA, BM, kLinearThreads> TileA;
  typedef OperandTile<IO, TB, BN, kLinearThreads> TileB;
  static constexpr int BK = TileA::BK, KGS = BK / Tr::KG;
  static constexpr int MI = BM / 64, NI = BN / 64;           // 32 x 32 accumulator tiles of a wave (2 x 2 waves)
  static constexpr int kStageRow = BN / 2 + Tr::HW;          // epilogue: the wave's half tile, row by row
  static constexpr int kStage = 4 * (BM / 2) * kStageRow;
  static constexpr int kBuffers = DIRECT ? STAGES * (BM + BN) * BK : 2 * (TileA::kElems + TileB::kElems);
  static constexpr int kElems = kBuffers > kStage ? kBuffers : kStage;         // of the workgroup's LDS

  // The tile of workgroup `block` of the product.
  static RGLRU_DEVICE void run(const LinearArgs& p, unsigned block, IO* lds) {
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, hf = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  // Workgroups go to the eight XCDs round-robin; each XCD gets a contiguous run of tiles (columns fastest), so that
  // the rows they share come from memory once and the weights stay in its L2.
  const int per_xcd = (p.total + 7) >> 3;
  int t = (block & 7) * per_xcd + (block >> 3);
  if ((int)(block >> 3) >= per_xcd || t >= p.total) return;
  const int tn = t % p.tiles_n; t /= p.tiles_n;
  const int problem = t % p.problems; t /= p.problems;
  const int tm = t % p.tiles_m; t /= p.tiles_m;
  const int item = t % p.batch;
  const int split = t / p.batch;
  const int m0 = tm * BM, n0 = tn * BN;
  const int m_left = p.M - m0, n_left = p.N - n0;
  const int k_begin = split * p.k_per_split;
  const int k_end = (k_begin + p.k_per_split) < p.K ? (k_begin + p.k_per_split) : p.K;
  const int slices = (k_end - k_begin + BK - 1) / BK;
  const int total_slices = slices * p.segments;
  // one input, two weights (forward); two gradients, one input (weight gradient); both change with the segment (input gradient)
  const bool masked = TA && p.active != nullptr;

  TileA ta;
  TileB tb;
  ta.setup(tid, p.lda, m_left);
  tb.setup(tid, p.ldb, n_left);
  // the segments' operands, read from the arguments once: inside the loop that would be a scalar load and a wait for it a slice
  const IO* const a_first = (const IO*)p.a[p.segments > 1 ? 0 : (TA ? problem : 0)] + item * p.a_step;
  const IO* const b_first = (const IO*)p.b[p.segments > 1 ? 0 : (TA ? 0 : problem)] + item * p.b_step;
  const IO* const a_second = p.segments > 1 ? (const IO*)p.a[1] + item * p.a_step : a_first;
  const IO* const b_second = p.segments > 1 ? (const IO*)p.b[1] + item * p.b_step : b_first;
  const unsigned char* const active = masked ? p.active : nullptr;
  const long long lda = p.lda, ldb = p.ldb;
  auto request = [&](int q, int s) {
    const bool second = s >= slices;
    const int k = k_begin + (s - (second ? slices : 0)) * BK;
    const IO* a = second ? a_second : a_first;
    const IO* b = second ? b_second : b_first;
    const int left = s < total_slices ? k_end - k : 0;
    const long long ks = s < total_slices ? k : 0;
    ta.request(q, a + (TA ? ks * lda + m0 : m0 * lda + ks), lda, left, m_left, tid, masked ? active + ks : nullptr);
    tb.request(q, b + (TB ? ks * ldb + n0 : n0 * ldb + ks), ldb, left, n_left, tid);
  };
  constexpr int kBuffer = TileA::kElems + TileB::kElems;

  f32x16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  // The weights are the products' first operand, so an accumulator's lane has ONE row of the result (m = r) and runs of four
  // columns (n = 8 (v / 4) + 4 hf + v % 4): what is loaded, staged and stored below are vectors of four.
  typedef IO io4 __attribute__((ext_vector_type(4)));
  if (p.accumulate) {
    const rsrc_t rc = make_rsrc((const IO*)p.c[problem] + item * p.c_step + (long long)m0 * p.ldc + n0, (unsigned)((long long)(m_left < BM ? m_left : BM) * p.ldc) * (unsigned)sizeof(IO));
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int n = wn * (BN / 2) + 32 * j + 8 * g + 4 * hf, m = wm * (BM / 2) + 32 * i + r;
          const io4 c = buf_load_four<IO>(rc, n < n_left ? ((unsigned)m * (unsigned)p.ldc + (unsigned)n) * (unsigned)sizeof(IO) : kOutOfRange);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][j][4 * g + e] = (float)c[e];
        }
  }
  // A bias may start at any element (a view of a longer tensor).  Vectors of it are asked for here, since behind the last slice they
  // would be waited for; one that starts off their boundaries is loaded there, by elements.
  const IO* const bias_from = TA ? nullptr : (const IO*)p.bias[problem];
  const bool bias_vectors = bias_from != nullptr && (unsigned long long)bias_from % sizeof(io4) == 0;
  io4 bias[NI][4];
  if constexpr (!TA) {
    const rsrc_t rb = make_rsrc(bias_from + n0, bias_vectors ? (unsigned)n_left * (unsigned)sizeof(IO) : 0u);
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) bias[j][g] = buf_load_four<IO>(rb, (unsigned)(wn * (BN / 2) + 32 * j + 8 * g + 4 * hf) * (unsigned)sizeof(IO));
  } else {
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) bias[j][g] = io4{};
  }
  float sum[MI];                                             // column sums of A over the lane's share of K
#pragma unroll
  for (int i = 0; i < MI; ++i) sum[i] = 0.f;
  const bool sums = TA && p.colsum && tn == 0 && wn == 0;

  if constexpr (DIRECT) {
    DirectTile<IO, BM> da;
    DirectTile<IO, BN> db;
    da.setup(wave, lane, lda);
    db.setup(wave, lane, ldb);
    constexpr unsigned kBytesA = DirectTile<IO, BM>::kBytes, kStageBytes = kBytesA + DirectTile<IO, BN>::kBytes;
    constexpr int LOADS = DirectTile<IO, BM>::NV + DirectTile<IO, BN>::NV;     // of a wave and slice
    unsigned char* const bytes = reinterpret_cast<unsigned char*>(lds);
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)bytes;
    auto fetch = [&](int s, int stage) {
      const int k = k_begin + s * BK, left = s < total_slices ? k_end - k : 0;
      const long long ks = s < total_slices ? k : 0;
      da.request(a_first + m0 * lda + ks, lda, left, m_left, lds0 + (unsigned)stage * kStageBytes, wave);
      db.request(b_first + n0 * ldb + ks, ldb, left, n_left, lds0 + (unsigned)stage * kStageBytes + kBytesA, wave);
    };
    // a slice has landed when every wave has waited for its own part of it
    auto landed = [&](auto younger) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(decltype(younger)::value) : "memory");
    };
#pragma unroll
    for (int q = 0; q < STAGES - 1; ++q) fetch(q, q);
    landed(std::integral_constant<int, (STAGES - 2) * LOADS>{});
    int stage = 0;
    for (int s = 0; s < total_slices; ++s) {
      const int last = stage == 0 ? STAGES - 1 : stage - 1;                      // read in the pass before
      fetch(s + STAGES - 1, last);
      const unsigned char* cur = bytes + (unsigned)stage * kStageBytes;
      Frag fa[2][MI], fb[2][NI];
      auto read = [&](int kg) {
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[kg & 1][i] = da.fragment(cur, wm * (BM / 2) + 32 * i, kg);
#pragma unroll
        for (int j = 0; j < NI; ++j) fb[kg & 1][j] = db.fragment(cur + kBytesA, wn * (BN / 2) + 32 * j, kg);
      };
      read(0);
#pragma unroll
      for (int kg = 0; kg < KGS; ++kg) {
        if (kg + 1 < KGS) read(kg + 1);
        __builtin_amdgcn_sched_barrier(0);               // or the reads sink to their use, and the products wait for them
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) Tr::mma(acc[i][j], fb[kg & 1][j], fa[kg & 1][i]);
      }
      landed(std::integral_constant<int, (STAGES - 2) * LOADS>{});
      stage = stage + 1 == STAGES ? 0 : stage + 1;
    }
    landed(std::integral_constant<int, 0>{});                                  // nothing may land over the epilogue's staging
  } else {
  request(0, 0);
  request(1, 1);
  ta.deposit(0, lds, tid, masked);
  tb.deposit(0, lds + TileA::kElems, tid);
  __syncthreads();
  // Slice s is multiplied out of one buffer while slice s + 1 goes from registers to the other and slice s + 2 is requested.  The
  // order inside a slice: requests first (left to itself the compiler sinks them to the end, where they cover nothing), then half of
  // the products, whose LDS reads would otherwise queue behind the writes, then the writes, then the other half.
  auto multiply = [&](const IO* cur, int from) {
#pragma unroll
    for (int kg = from; kg < from + KGS / 2; ++kg) {
      Frag fa[MI], fb[NI];
#pragma unroll
      for (int i = 0; i < MI; ++i) fa[i] = TileA::fragment(cur, wm * (BM / 2) + 32 * i, kg, lane);
#pragma unroll
      for (int j = 0; j < NI; ++j) fb[j] = TileB::fragment(cur + TileA::kElems, wn * (BN / 2) + 32 * j, kg, lane);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) Tr::mma(acc[i][j], fb[j], fa[i]);
      if (sums) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int e = 0; e < Tr::HW; ++e) sum[i] += (float)fa[i][e];
      }
    }
  };
  for (int s0 = 0; s0 < total_slices; s0 += 2) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {                            // the parity names buffer and slot
      const int s = s0 + u;
      if (s >= total_slices) break;
      const IO* cur = lds + u * kBuffer;
      IO* nxt = lds + (u ^ 1) * kBuffer;
      request(u, s + 2);
      __builtin_amdgcn_sched_barrier(0);
      multiply(cur, 0);
      ta.deposit(u ^ 1, nxt, tid, masked);
      tb.deposit(u ^ 1, nxt + TileA::kElems, tid);
      multiply(cur, KGS / 2);
      __syncthreads();
    }
  }

  }

  if constexpr (!TA) if (bias_from != nullptr && !bias_vectors) {
    const rsrc_t rb = make_rsrc(bias_from + n0, (unsigned)n_left * (unsigned)sizeof(IO));
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          bias[j][g][e] = (IO)BufIo<IO>::load(rb, (unsigned)(wn * (BN / 2) + 32 * j + 8 * g + 4 * hf + e) * (unsigned)sizeof(IO), 0u);
  }
  if (sums) {
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const float both = sum[i] + xhalf(sum[i], hf);
      const int m = wm * (BM / 2) + 32 * i + r;
      if (hf == 0 && m < m_left) p.colsum[((long long)split * p.problems + problem) * p.M + m0 + m] = both;
    }
  }
  const int col0 = wn * (BN / 2), row0 = wm * (BM / 2);
  if constexpr (TA) if (p.partial) {                         // weight gradients
    const int ld = p.partial_ld ? p.partial_ld : p.N, rows = p.partial_ld ? p.partial_ld : p.M;
    float* part = p.partial + ((((long long)split * p.batch + item) * p.problems + problem) * rows + m0) * ld + n0;
    const rsrc_t rc = make_rsrc(part, (unsigned)((long long)(m_left < BM ? m_left : BM) * ld) * 4u);
    // through LDS like the result: stored from the accumulators, a row of the wave's tile is 32 bytes an instruction (two weight
    // gradients of 2048 x 1024 x 768, when bf16 ran here: 45 us that way, 42 element by element, 41 like this)
    constexpr int kRow = BN / 2 + 4;
    static_assert(4 * (BM / 2) * kRow * 4 <= kElems * (int)sizeof(IO), "the fp32 tile fits where the slices were");
    float* stage = reinterpret_cast<float*>(lds) + wave * (BM / 2) * kRow;
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x4 c;
#pragma unroll
          for (int e = 0; e < 4; ++e) c[e] = acc[i][j][4 * g + e];
          *reinterpret_cast<f32x4*>(stage + (32 * i + r) * kRow + 32 * j + 8 * g + 4 * hf) = c;
        }
    wave_lds_fence();
    constexpr int VPR = (BN / 2) / 4, ROWS = 64 / VPR;
#pragma unroll
    for (int q = 0; q < (BM / 2) / ROWS; ++q) {
      const int m = q * ROWS + lane / VPR, cv = lane % VPR, row = row0 + m, n = col0 + cv * 4;
      const i32x4 c = *reinterpret_cast<const i32x4*>(stage + m * kRow + cv * 4);
      buf_store_b128<kWriteThrough>(c, rc, n < n_left && row < m_left ? ((unsigned)row * (unsigned)ld + (unsigned)n) * 4u : kOutOfRange);
    }
    return;
  }
  // result in the storage type: through LDS (the slices have been read), then 16-byte vectors of rows, written through the L2s
  // (kWriteThrough).  Kernel times: 2331 x 2 x 1024 x 768 in bf16 16.6 -> 15.8 us, fp32
  // gate gradients of B4 T1024 W1024 37.5 -> 34.8; the largest tried, 134 MB, 183 -> 181.
  IO* stage = lds + wave * (BM / 2) * kStageRow;
#pragma unroll
  for (int j = 0; j < NI; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int n = 32 * j + 8 * g + 4 * hf;
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        io4 c;
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] = (IO)(acc[i][j][4 * g + e] + (float)bias[j][g][e]);
        *reinterpret_cast<io4*>(stage + (32 * i + r) * kStageRow + n) = c;
      }
    }
  wave_lds_fence();
  const rsrc_t rc = make_rsrc((IO*)p.c[problem] + item * p.c_step + (long long)m0 * p.ldc + n0, (unsigned)((long long)(m_left < BM ? m_left : BM) * p.ldc) * (unsigned)sizeof(IO));
  constexpr int VPR = (BN / 2) / Tr::HW, ROWS = 64 / VPR;
  static_assert(64 % VPR == 0 && (BM / 2) % ROWS == 0, "whole rows an instruction");
#pragma unroll
  for (int q = 0; q < (BM / 2) / ROWS; ++q) {
    const int m = q * ROWS + lane / VPR, cv = lane % VPR;
    Frag f = *reinterpret_cast<const Frag*>(stage + m * kStageRow + cv * Tr::HW);
    const int row = row0 + m, n = col0 + cv * Tr::HW;
    if (!TA && p.active && row < m_left && !p.active[m0 + row]) f = Tr::zero();
    const unsigned off = n < n_left && row < m_left ? ((unsigned)row * (unsigned)p.ldc + (unsigned)n) * (unsigned)sizeof(IO) : kOutOfRange;
    buf_store_b128<kWriteThrough>(__builtin_bit_cast(i32x4, f), rc, off);
  }
  }
};

template <typename IO, bool TA, bool TB, int BM, int BN>
__global__ __launch_bounds__(kLinearThreads, 2) void linear_kernel(LinearArgs p) {
  typedef LinearTile<IO, TA, TB, BM, BN> Tile;
  __shared__ __attribute__((aligned(16))) IO lds[Tile::kElems];
  if constexpr (!TA && !TB && sizeof(IO) == 2) {
    if (p.positions.B > 0) token_positions(p.positions, (long long)blockIdx.x * kLinearThreads + threadIdx.x, (long long)gridDim.x * kLinearThreads);
  }
  Tile::run(p, blockIdx.x, lds);
}

// The weight and input gradients of the gates' products in fp32, in small tiles, in one launch: neither reads what the other writes.  The
// weight gradients' workgroups have twice the slices and go first.  Steps of the layer in fp32, two launches and one, us, four processes each: B4 T1024
// W1024 (16 gate blocks) 97.1 to 100.1 and 96.7 to 97.5, B8 T2048 333 to 335 and 322; B2 T256 W256 is the host's, whose spread (60 to 100) hides it.
__global__ __launch_bounds__(kLinearThreads, 2) void gate_grads_kernel(LinearArgs weights, LinearArgs input, unsigned first) {
  typedef LinearTile<float, true, true, 64, 64> Weights;
  typedef LinearTile<float, false, true, 64, 64> Input;
  __shared__ __attribute__((aligned(16))) float lds[Weights::kElems > Input::kElems ? Weights::kElems : Input::kElems];
  if (blockIdx.x < first) Weights::run(weights, blockIdx.x, lds);
  else Input::run(input, blockIdx.x - first, lds);
}

// How a product is cut up.  Forward in bf16: the cheapest of four tiles by a model of the time in us, whose constants come from 100 sizes (60 to 16000
// rows, 256 to 2560 columns, 128 to 2560 contraction indices, one and two problems) on 256 compute units, every product behind a kernel that
// writes its input.  A launch takes `launch`; the units run their tiles in rounds of `per_cu`, each of which takes `start` and `slice[n - 1]` for
// 64 contraction indices with n workgroups on a compute unit; and `moved` for every 256,000 operand lines that go to LDS (what the L2s
// give).  It picks within 1 % (at most 10) of the best of the four, and is 3 % (-4 to 44) faster than two tiles (64 x 64 up to three to a compute unit,
// else 128 x 128).  Kernel us, 64 x 64 : 128 x 64 : 128 x 128 : 192 x 128 (* taken, + by the two-tile rule), two problems unless said:
//   600 x 1024 x 768 +9.1 : *9.0 : 14.2 : 15.6, 2331 18.8 : 18.7 : *+15.7 : 16.6, 4096 27.5 : 23.0 : *+17.8 : 21.2, 6216 38.8 : 34.6 : *+29.0 : 32.6;
//   415 x 2048 x 1536 +17.4 : *14.6 : 23.2 : 25.4;  2668 x 768 x 512 14.0 : *10.0 : +11.2 : 12.4;  11981 x 384 x 384 20.2 : 18.4 : +18.7 : *14.5;
//   one of 2331 x 768 x 1024 +11.0 : *10.4 : 15.7 : 18.0, 8704 28.4 : 24.2 : *+20.3 : 24.0;  8704 x 1024 x 768 28.9 : 26.7 : +26.2 : *21.4;
//   7012 x 1280 x 1024 34.9 : 32.0 : +31.2 : *24.8;  4518 x 2560 x 512 29.7 : 24.6 : +22.1 : *17.9;  901 x 1536 x 2560 +21.4 : *19.3 : 34.9 : 37.4
// 64 x 128 is 128 x 64 but for few rows (415 x 2048 x 1536 16.6); 192 x 192, 256 x 128 and 128 x 192 are the better ones nowhere by more than 4 %.
// From six tiles of 128 x 128 to a compute unit on the largest are taken without the model (two of 16384 x 1024 x 768 109.8 : 92 : +75 : *66.7).
// fp32 is bound by its MFMAs, and a small tile takes 1 / 4 of a large one and 6 % more, so the number of steps decides (M x 256 x 256, two
// problems; steps small : large x 4):  8183 (4 : 4) 22.1 : 22.2, 8439 (5 : 8) 26.3 : 36.0, 14071 (7 : 8) 35.8 : 36.9, 15991 (8 : 8) 40.3 : 37.8, 16631
// (9 : 12) 44.2 : 54.9, 24567 (12 : 12) 58.9 : 56.3;  input gradient 8183 (2 : 4) 24.6 : 40.8, 16375 (4 : 4)
// 39.9 : 42.5.
// A weight gradient contracts over the tokens, so its tiles are few and its contraction long: it is split over workgroups (every split
// costs a pass over the result in fp32).  In fp32 until there are about two to a compute unit, at least four slices each and at most
// eight splits (two of 1024 x 768 at 2331 tokens 83 us in small tiles, 108 in large ones).
struct ForwardCost { int rows, columns; unsigned per_cu; float launch, start, slice[3], moved; };
static LinearPlan forward16_plan(int64_t M, int64_t N, int64_t K, int problems) {
  static const ForwardCost costs[] = {{64, 64, 3, 2.23f, 2.12f, {0.219f, 0.329f, 0.398f}, 0.49f}, {128, 64, 2, 2.31f, 2.38f, {0.304f, 0.435f, 0.0f}, 0.48f},
                                      {128, 128, 2, 1.68f, 3.30f, {0.644f, 0.789f, 0.0f}, 0.41f}, {192, 128, 2, 0.63f, 4.93f, {0.726f, 1.030f, 0.0f}, 0.67f}};
  const float slices = (float)((K + 63) / 64);
  const unsigned units = (unsigned)num_compute_units();
  if (M * N * problems >= (int64_t)units * 6 * 128 * 128) return {192, 1, 128};
  LinearPlan best = {64, 1, 64};
  float least = 1e30f;
  for (const ForwardCost& c : costs) {
    const unsigned tiles = (unsigned)((M + c.rows - 1) / c.rows) * (unsigned)((N + c.columns - 1) / c.columns) * (unsigned)problems;
    const unsigned each = (tiles + units - 1) / units, rounds = each / c.per_cu, rest = each - rounds * c.per_cu;
    const float t = c.launch + (float)rounds * (c.start + c.slice[c.per_cu - 1] * slices) + (rest ? c.start + c.slice[rest - 1] * slices : 0.0f) +
                    c.moved * (float)(c.rows + c.columns) * (1.0f / 256e3f) * (float)tiles * slices;
    if (t < least) { least = t; best = {c.rows, 1, c.columns}; }
  }
  return best;
}
struct TileCost { int edge; unsigned per_cu; double start, slice[3]; };
// Gradients in bf16: the cheapest by a model of the time in us.  A workgroup of a tile size takes `start` and `slice[n - 1]` for 64 contraction
// indices with n of them on a compute unit; the units run their tiles in rounds of `per_cu`.  Constants from 64, 128 and 256 on
// 1000 to 16384 tokens of 768 and 1024 channels.  What it picks, us in calls behind each other, weight gradients with the launch that adds up their sets and the
// column sums, sizes 64 : 128 : 256 (* taken; splits of that size behind the slash):
//   input, two segments of 1024 into 768   1000 *12.5 : 21.0 : 48.9, 2331 *17.3 : 22.1 : 48.9, 4096 23.9 : *22.7 : 49.1, 8704 47.8 : *31.1 : 50.4, 16384 79.6 :
//          *53.6 : 55.5
//   input, 768 into 1024   1000 *6.9 : 10.1 : 22.2, 2331 *10.9 : 10.4 : 22.4, 6000 19.6 : *15.1 : 22.8, 8704 26.9 : *23.0 : 23.3, 16384 46.1 : 29.8 : *29.0
//   weight, two of 1024 x 768   1000 *15.2/1 : 19.1/2 : 27.3/4, 2331 *23.9/2 : 24.9/2 : 30.7/8, 4096 32.4/2 : *29.4/5 : 34.8/8, 8704 57.2/2 : *46.2/5 :
//          47.5/10, 16384 103.9/2 : 76.5/5 : *71.8/10
//   weight, 768 x 1024   1000 *13.2/2 : 16.2/4 : 20.8/4, 2331 *17.9/4 : 19.5/5 : 26.9/8, 4096 *21.2/4 : 20.5/5 : 29.1/16, 8704 32.9/4 : *30.6/5 : 36.5/20, 16384
//          54.3/4 : *43.3/10 : 47.4/20
// Kernels alone at 8704 tokens, in the order above: 30.9, 22.7, 39.1 and 26.1; those they replace, whose slices went through registers, 40.2, 29.8, 64.5 and
// 31.8.
static LinearPlan linear16_plan(bool weight, int64_t M, int64_t N, int64_t K, int problems, int segments) {
  static const TileCost input[] = {{64, 3, 2.5, {0.36, 0.47, 0.69}}, {128, 2, 4.5, {0.58, 0.87, 0.0}}, {256, 1, 10.0, {1.43, 0.0, 0.0}}};
  static const TileCost weights[] = {{64, 3, 3.0, {0.39, 0.52, 0.71}}, {128, 2, 6.0, {0.70, 1.18, 0.0}}, {256, 1, 12.0, {1.74, 0.0, 0.0}}};
  static const unsigned some[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24};
  const unsigned units = (unsigned)num_compute_units(), slices = (unsigned)((K + 63) / 64);
  LinearPlan best = {64, 1};
  double least = 1e30;
  for (const TileCost& c : weight ? weights : input) {
    if (c.edge == 256 && N >= (1 << 20)) continue;           // 256 lines of fp32 within a lane's reach
    const double all = (double)((M + c.edge - 1) / c.edge) * (double)((N + c.edge - 1) / c.edge) * problems;
    if (all > 1e6) {                                         // far more tiles than units: by their throughput
      const double t = all / units * c.slice[c.per_cu - 1] / c.per_cu * slices * segments;
      if (t < least) { least = t; best = {c.edge, 1}; }
      continue;
    }
    const unsigned tiles = (unsigned)all;
    for (unsigned splits : some) {
      if (splits > 1 && (!weight || splits * 4 > slices)) break;
      const unsigned each = (tiles * splits + units - 1) / units, rounds = each / c.per_cu, rest = each - rounds * c.per_cu;
      const double part = (double)((slices + splits - 1) / splits) * segments;
      double t = rounds * (c.start + c.slice[c.per_cu - 1] * part) + (rest ? c.start + c.slice[rest - 1] * part : 0.0);
      if (splits > 1) t += (double)splits * problems * M * N * (4.0 / 4.5e6);        // the sets are read again
      if (t < least) { least = t; best = {c.edge, (int)splits}; }
    }
  }
  return best;
}
static LinearPlan linear_plan(int kind, int64_t M, int64_t N, int64_t K, int problems, int segments, int dtype) {
  if (dtype == RGLRU_BF16 && kind == RGLRU_LINEAR_FORWARD) return forward16_plan(M, N, K, problems);
  if (dtype == RGLRU_BF16) return linear16_plan(kind == RGLRU_LINEAR_WEIGHT_GRAD, M, N, K, problems, segments);
  auto tiles = [&](int64_t edge) { return ((M + edge - 1) / edge) * ((N + edge - 1) / edge) * problems; };
  const int64_t units = num_compute_units();
  auto steps = [&](int64_t edge) { return (tiles(edge) + units - 1) / units; };
  LinearPlan p = {tiles(128) > units && 106 * steps(64) >= 400 * steps(128) ? 128 : 64, 1};
  if (kind != RGLRU_LINEAR_WEIGHT_GRAD) return p;
  const int64_t slices = (K + 31) / 32;
  auto splits = [&](int64_t t) {
    int64_t s = (2 * units + t - 1) / t;
    if (s > slices / 4) s = slices / 4;
    return s > 8 ? (int64_t)8 : s < 1 ? (int64_t)1 : s;
  };
  p.edge = tiles(128) * splits(tiles(128)) >= units ? 128 : 64;
  p.splits = (int)splits(tiles(p.edge));
  return p;
}

template <int BM, int BN>
static unsigned linear_grid(LinearArgs& a) {
  a.tiles_m = (a.M + BM - 1) / BM;
  a.tiles_n = (a.N + BN - 1) / BN;
  a.total = a.tiles_m * a.tiles_n * a.problems * a.batch * a.splits;
  return (unsigned)(8 * ((a.total + 7) / 8));
}
template <typename IO, bool TA, bool TB, int BM, int BN>
static void linear_launch(LinearArgs& a, hipStream_t s) {
  const unsigned grid = linear_grid<BM, BN>(a);
  hipLaunchKernelGGL((linear_kernel<IO, TA, TB, BM, BN>), dim3(grid), dim3(kLinearThreads), 0, s, a);
}
template <bool TA, bool TB>
static void linear32_launch(LinearArgs& a, int edge, hipStream_t s) {
  edge > 64 ? linear_launch<float, TA, TB, 128, 128>(a, s) : linear_launch<float, TA, TB, 64, 64>(a, s);
}

static void linear_launch(LinearArgs& a, int kind, LinearPlan plan, int dtype, hipStream_t s) {
  if (dtype == RGLRU_BF16) {
    if (kind != RGLRU_LINEAR_FORWARD) linear16_launch(a, kind, plan.edge, s);
    else if (plan.edge == 192) linear_launch<__bf16, false, false, 192, 128>(a, s);
    else if (plan.edge == 64) linear_launch<__bf16, false, false, 64, 64>(a, s);
    else if (plan.columns == 64) linear_launch<__bf16, false, false, 128, 64>(a, s);
    else linear_launch<__bf16, false, false, 128, 128>(a, s);
  } else {
    if (kind == RGLRU_LINEAR_FORWARD) linear32_launch<false, false>(a, plan.edge, s);
    else if (kind == RGLRU_LINEAR_INPUT_GRAD) linear32_launch<false, true>(a, plan.edge, s);
    else linear32_launch<true, true>(a, plan.edge, s);
  }
}

// ---- the gate blocks' products (griffin/griffin.py:149-154 and their reverse mode) as batches ----------------------
// For the configurations whose scan kernels leave the gradients at the gate pre-activations in memory.  Tiles of 128 where
// the block is wider than 64 channels and there are enough of them.
static bool batch_large(const Geometry& g, long long tokens_or_width, int problems) {
  return g.bw > 64 && ((tokens_or_width + 127) / 128) * ((g.bw + 127) / 128) * g.nb * problems >= num_compute_units();
}

bool gate_products_cover(const Geometry& g, int dtype, std::initializer_list<const void*> tensors, std::initializer_list<long long> strides) {
  const int vec = dtype == RGLRU_BF16 ? 8 : 4;
  if (g.bw % vec || g.W % vec) return false;
  for (const void* q : tensors) if ((uintptr_t)q % 16) return false;
  for (long long v : strides) if (v % vec || v >= (1 << 22)) return false;
  return true;
}

int gate_pre_product(const void* x, const void* wg, void* pre, long long N, const Geometry& g, hipStream_t s) {
  LinearArgs a;
  memset(&a, 0, sizeof(a));
  const long long gate = g.nb * g.bwp * g.bwp;
  a.a[0] = x; a.b[0] = wg; a.b[1] = (const __bf16*)wg + gate; a.c[0] = pre; a.c[1] = (__bf16*)pre + g.bw;
  a.lda = g.W; a.ldb = g.bwp; a.ldc = 2 * g.bw; a.a_step = g.bw; a.b_step = g.bwp * g.bwp; a.c_step = N * 2 * g.bw;
  a.batch = (int)g.nb; a.problems = 2; a.segments = 1; a.splits = 1;
  a.M = (int)N; a.N = a.K = a.k_per_split = (int)g.bw;
  linear_launch(a, RGLRU_LINEAR_FORWARD, {batch_large(g, N, 2) ? 128 : 64, 1}, RGLRU_BF16, s);
  return check_launch("gate pre-activations");
}

int gate_grads(const void* x, const void* du_a, const void* du_x, long long du_ld, long long du_blk, const void* wg, void* dx, float* partial, int splits,
               long long N, const Geometry& g, int dtype, hipStream_t s) {
  LinearArgs in, w;
  memset(&in, 0, sizeof(in));
  const long long gate = g.nb * g.bwp * g.bwp;
  in.a[0] = du_a; in.a[1] = du_x; in.b[0] = wg; in.b[1] = (const char*)wg + gate * (dtype == RGLRU_BF16 ? 2 : 4); in.c[0] = dx;
  in.lda = du_ld; in.ldb = g.bwp; in.ldc = g.W; in.a_step = du_blk; in.b_step = g.bwp * g.bwp; in.c_step = g.bw;
  in.batch = (int)g.nb; in.problems = 1; in.segments = 2; in.splits = 1; in.accumulate = 1;
  in.M = (int)N; in.N = in.K = in.k_per_split = (int)g.bw;
  memset(&w, 0, sizeof(w));
  w.a[0] = du_a; w.a[1] = du_x; w.b[0] = x; w.partial = partial; w.partial_ld = (int)g.bwp;
  w.lda = du_ld; w.ldb = g.W; w.a_step = du_blk; w.b_step = g.bw;
  w.batch = (int)g.nb; w.problems = 2; w.segments = 1; w.splits = splits;
  w.M = w.N = (int)g.bw; w.K = (int)N;
  const long long bk = dtype == RGLRU_BF16 ? 64 : 32;
  w.k_per_split = (int)(((N + splits - 1) / splits + bk - 1) / bk * bk);
  const bool large_in = batch_large(g, N, 1), large_w = batch_large(g, g.bw, 2 * splits);
  if (dtype == RGLRU_F32 && !large_in && !large_w) {
    const unsigned first = linear_grid<64, 64>(w), second = linear_grid<64, 64>(in);
    hipLaunchKernelGGL(gate_grads_kernel, dim3(first + second), dim3(kLinearThreads), 0, s, w, in, first);
    return check_launch("gate gradients");
  }
  linear_launch(in, RGLRU_LINEAR_INPUT_GRAD, {large_in ? 128 : 64, 1}, dtype, s);
  linear_launch(w, RGLRU_LINEAR_WEIGHT_GRAD, {large_w ? 128 : 64, 1}, dtype, s);
  return check_launch("gate gradients");
}

}  // namespace rglru

using namespace rglru;

static int linear_product(int kind, const void* a0, const void* a1, int64_t lda, const void* b0, const void* b1, int64_t ldb,
                          const void* bias0, const void* bias1, const uint8_t* active, void* c0, void* c1, int64_t ldc,
                          float* partial, float* colsum, int64_t M, int64_t N, int64_t K, int dtype, void* stream, const PositionArgs* positions) {
  if (dtype != RGLRU_F32 && dtype != RGLRU_BF16) return fail(RGLRU_E_ARG, "linear: dtype must be RGLRU_F32 or RGLRU_BF16, got %d", dtype);
  if (kind < RGLRU_LINEAR_FORWARD || kind > RGLRU_LINEAR_WEIGHT_GRAD) return fail(RGLRU_E_ARG, "linear: unknown kind %d", kind);
  if (M <= 0 || N <= 0 || K <= 0) return fail(RGLRU_E_ARG, "linear: empty product %lld x %lld x %lld", (long long)M, (long long)N, (long long)K);
  LinearArgs a;
  memset(&a, 0, sizeof(a));
  a.a[0] = a0; a.a[1] = a1; a.b[0] = b0; a.b[1] = b1; a.bias[0] = bias0; a.bias[1] = bias1; a.c[0] = c0; a.c[1] = c1;
  a.batch = 1; a.active = active; a.colsum = colsum; a.lda = lda; a.ldb = ldb; a.ldc = ldc;
  a.problems = kind == RGLRU_LINEAR_FORWARD ? (b1 ? 2 : 1) : kind == RGLRU_LINEAR_WEIGHT_GRAD ? (a1 ? 2 : 1) : 1;
  a.segments = kind == RGLRU_LINEAR_INPUT_GRAD && a1 ? 2 : 1;
  LinearPlan plan = linear_plan(kind, M, N, K, a.problems, a.segments, dtype);
  if (plan.edge == 256 && (lda >= (1 << 21) || ldc >= (1 << 21))) plan.edge = 128;        // 256 lines within a lane's reach
  a.splits = plan.splits;
  if (plan.splits > 1) a.partial = partial;
  if (!a0 || !b0 || (a.segments == 2 && !b1) || (plan.splits > 1 ? !partial : (!c0 || (a.problems == 2 && !c1)))) return fail(RGLRU_E_ARG, "linear: null pointer");
  const int64_t es = dtype == RGLRU_BF16 ? 2 : 4, vec = 16 / es;
  const bool ta = kind == RGLRU_LINEAR_WEIGHT_GRAD, tb = kind != RGLRU_LINEAR_FORWARD;
  // rows of whole 16-byte vectors on a 16-byte boundary: what every load and store of the kernel is
  const void* ptrs[] = {a0, a1, b0, b1, a.partial ? nullptr : c0, a.partial ? nullptr : c1};
  for (const void* q : ptrs) if ((uintptr_t)q % 16) return fail(RGLRU_E_UNSUPPORTED, "linear: operands must be 16-byte aligned");
  if ((lda % vec) || (ldb % vec) || (!a.partial && ldc % vec) || (ta ? M : K) % vec || N % vec || (!tb && K % vec))
    return fail(RGLRU_E_UNSUPPORTED, "linear: rows must be whole 16-byte vectors");
  if (lda < (ta ? M : K) || ldb < (tb ? N : K) || (!a.partial && ldc < N)) return fail(RGLRU_E_ARG, "linear: a row stride is smaller than the row");
  if (M >= (1ll << 30) || N >= (1ll << 24) || K >= (1ll << 30) || lda >= (1 << 22) || ldb >= (1 << 22) || ldc >= (1 << 22) ||
      ((M + 63) / 64) * ((N + 63) / 64) * a.problems * a.splits >= (1ll << 30))
    return fail(RGLRU_E_UNSUPPORTED, "linear: product too large");
  a.M = (int)M; a.N = (int)N; a.K = (int)K;
  const int64_t bk = dtype == RGLRU_BF16 ? 64 : 32;
  a.k_per_split = (int)(((K + a.splits - 1) / a.splits + bk - 1) / bk * bk);
  if (positions) a.positions = *positions;
  hipStream_t s = (hipStream_t)stream;
  linear_launch(a, kind, plan, dtype, s);
  return check_launch("linear");
}

namespace rglru {
int linear_pair_with_positions(const void* x, const void* w0, const void* w1, const void* bias0, const void* bias1, void* u, void* v, int64_t M,
                               int64_t N, int64_t K, int dtype, const PositionArgs& positions, void* stream) {
  if (dtype != RGLRU_BF16) return fail(RGLRU_E_UNSUPPORTED, "block_project: needs bf16 storage");
  if (!w1 || !v) return fail(RGLRU_E_ARG, "block_project: null pointer");
  return linear_product(RGLRU_LINEAR_FORWARD, x, nullptr, K, w0, w1, K, bias0, bias1, nullptr, u, v, N, nullptr, nullptr, M, N, K, dtype, stream, &positions);
}
}  // namespace rglru

extern "C" {

int64_t rglru_hip_linear_splits(int kind, int64_t M, int64_t N, int64_t K, int problems, int dtype) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return linear_plan(kind, M, N, K, problems, 1, dtype).splits;
}

int rglru_hip_linear(int kind, const void* a0, const void* a1, int64_t lda, const void* b0, const void* b1, int64_t ldb,
                     const void* bias0, const void* bias1, const uint8_t* active, void* c0, void* c1, int64_t ldc,
                     float* partial, float* colsum, int64_t M, int64_t N, int64_t K, int dtype, void* stream) {
  return linear_product(kind, a0, a1, lda, b0, b1, ldb, bias0, bias1, active, c0, c1, ldc, partial, colsum, M, N, K, dtype, stream, nullptr);
}

}  // extern "C"

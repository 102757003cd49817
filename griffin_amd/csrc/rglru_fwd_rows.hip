// Forward of large batches: a workgroup owns whole sequences, so its tiles need nothing from any other workgroup.
#include "rglru_fused.h"

namespace rglru {

// Tiles of a sequence run one after the other in one workgroup, the state stays in a register: no tickets, no records, no look-back,
// nothing to clear, and the order of the sums is fixed.  A workgroup of four waves holds the unit's 128 channels (or its
// blocks side by side) like the tiled kernel; x is double-buffered in LDS, so a tile costs one barrier, and the next tile is requested
// as soon as this one is in LDS.  Calls with flags have a variant of their own: they come as one byte a lane and become two words by
// ballot, and a tile without any takes the plain gate math.  Two versions of that math in one kernel cost 40 registers and the
// scheduler its freedom, so calls without flags do not have them (128-wide: 243 -> 208 registers with 64-token tiles, 142 with 32).
// Bound by power: 24.8 vector instructions an element, six of them transcendental, and the matrix products beside them draw the
// clock down to 2.0-2.1 GHz.  In a series where the kernel took 650 us (B256 T2048 W1024; 628 in the one below) it took 500 without its
// loads and stores, 530 without its gate math, and 650 to 660 in every arrangement tried: tiles requested two ahead, x or y brought into
// their layout by products with the identity instead of two-byte LDS accesses.
// Forward of B256 W1024 in calls behind each other (the clock follows the load: a launch between lighter ones says little), us, tiled with
// the clearing of its records : two workgroups a compute unit with 64-token tiles and both versions of the math : three with 32-token
// tiles and one: T2048 in 128-wide blocks 708 : 672 : 628, T512 185 : 175 : 162.  With flags 829 : 686, the three-workgroup form
// spills (11 % more).  64-wide blocks, three workgroups and 32-token tiles: T512 171 : 150 : 146, with flags T2048 750 : 583.
// Where no more than two workgroups a compute unit have a sequence, the tiles of 96- and 128-wide blocks have 64 tokens without flags, too
// (B64 T2048 W1024 176.7 -> 172).
constexpr int rows_occ(int nkg, bool flags) { return nkg <= 4 || !flags ? 3 : 2; }
static bool rows_long_tiles(int nkg, bool flags, int64_t workgroups) { return nkg > 4 && (flags || workgroups <= 2 * (int64_t)num_compute_units()); }

// Gate outputs of 16 consecutive tokens (bits at .. at + 15 of the reset and padding words belong to them; without MASKED, bit 0 of
// `resets` to the first of them).
template <bool MASKED>
RGLRU_DEVICE void rows_gates(const f32x16& ua, const f32x16& ux, const float (&xv)[16], float sp, float nba, float nbx,
                             unsigned resets, unsigned pads, int at, float* a, float* z) {
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const float r = sigmoid_fast(ua[v], nba), i = sigmoid_fast(ux[v], nbx);
    float l2 = r * sp;
    if constexpr (MASKED) {
      const unsigned m_reset = (unsigned)__builtin_amdgcn_sbfe((int)resets, at + v, 1), m_pad = (unsigned)__builtin_amdgcn_sbfe((int)pads, at + v, 1);
      unsigned u = __builtin_bit_cast(unsigned, l2);
      u = (u & ~m_reset) | (__builtin_bit_cast(unsigned, kResetLog2) & m_reset);
      l2 = __builtin_bit_cast(float, u & ~m_pad);
    } else if (v == 0) {
      l2 = resets & 1u ? kResetLog2 : l2;
    }
    const GateOut o = gate_outputs<false>(r, i, xv[v], l2);
    a[v] = o.a; z[v] = o.z;
  }
}

// FLAGS: the call has an array of them; else only a sequence's first token may carry one (p.first_reset).
template <int NKG, bool PAD, bool FLAGS, int MT>
__global__ __launch_bounds__(kThreads, MT == 1 ? 3 : 2) void fwd_rows_kernel(FusedArgs p) {
  typedef __bf16 IO;
  typedef Io<IO> Tr;
  typedef Tr::Frag Frag;
  constexpr int TR = 32 * MT, EL = 16 * MT;
  constexpr int KC = kPackedWidth, LDSROW = KC + Tr::HW;
  constexpr int VPR = KC / Tr::HW, RP = kThreads / VPR, NV = TR / RP;      // a pass of the workgroup loads RP rows
  __shared__ __attribute__((aligned(16))) IO lds[2][TR * LDSROW];
  __shared__ __attribute__((aligned(16))) unsigned char stage_all[kWaves * WaveStage<TR>::kBytes];

  const WaveId w = wave_identity(p, blockIdx.x, true);
  const int hf = w.hf, tid = threadIdx.x;
  unsigned char* stage = stage_all + w.wave * WaveStage<TR>::kBytes;
  // nothing of the workspace is needed but a failure word that starts out zero (no kernel of this pass sets it)
  if (blockIdx.x == 0 && tid == 0) __hip_atomic_store(p.fail, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const IO* wg = (const IO*)p.wg;
  const int o_safe = w.slab_ok ? w.o : 0;
  HeldWeights<IO, NKG> hw;
  hw.load(wg + ((long long)(0 * p.nb + w.k) * p.bwp + o_safe) * p.bwp + hf * Tr::HW, wg + ((long long)(1 * p.nb + w.k) * p.bwp + o_safe) * p.bwp + hf * Tr::HW);
  const float nba = -kLog2e * p.bias[w.kp], nbx = -kLog2e * p.bias[p.Wp + w.kp];   // biases as the sigmoids take them
  const float sp = w.ch_ok ? p.sp[w.kp] : 0.f;
  const long long W = p.W;
  const unsigned uW = (unsigned)p.W, row_bytes = uW * 2u, ch = (unsigned)w.ch;
  const int nT = p.nCf;

  const int x_row = tid / VPR, x_cv = tid - x_row * VPR;
  const int x_ch = tile_channel<PAD>(p, w.unit, w.tile_col, x_cv * Tr::HW);
  const unsigned x_off = x_ch >= 0 && x_ch < p.W ? (unsigned)x_row * row_bytes + (unsigned)x_ch * 2u : kOutOfRange;
  IO* const x_at = &lds[0][0] + x_row * LDSROW + x_cv * Tr::HW;
  const rsrc_t rh0 = make_rsrc(p.h0, p.h0 ? (unsigned)p.B * uW * 4u : 0u), rhl = make_rsrc(p.h_last, p.h_last ? (unsigned)p.B * uW * 4u : 0u);
  Frag pre[NV];
  unsigned pre_fl = 0;
  float pre_h0;
  // a tile past the last sequence keeps valid addresses but an empty extent: nothing is fetched
  auto issue = [&](int b, int c) {
    const bool live = b < p.B;
    const int bb = live ? b : 0, rows = !live ? 0 : ((p.T - c * TR) < TR ? (p.T - c * TR) : TR);
    const long long row0 = (long long)bb * p.T + (long long)c * TR;
    const rsrc_t rx = make_rsrc((const IO*)p.x + row0 * W, (unsigned)rows * row_bytes);
    unsigned xo = x_off;
    asm volatile("" : "+v"(xo));
#pragma unroll
    for (int i = 0; i < NV; ++i) pre[i] = buf_load_frag<Frag>(rx, xo + (unsigned)(i * RP) * row_bytes);
    if constexpr (FLAGS) {
      const rsrc_t rf = make_rsrc(p.flags + row0, (unsigned)rows);
      pre_fl = (unsigned)__builtin_amdgcn_raw_buffer_load_b8(rf, (unsigned)(w.lane & (TR - 1)), 0, 0);
    }
    pre_h0 = BufIo<float>::load(rh0, live && c == 0 ? ((unsigned)b * uW + ch) * 4u : kOutOfRange, 0u);
  };
  int b = w.wg_in_unit, c = 0;
  issue(b, c);
  {
    // The loop is entered with as many stores behind its loads as its back edge has: the wait for a tile then leaves the stores of
    // the tile before in flight.
    const rsrc_t nowhere = make_rsrc(p.y, 0u);
    const i32x4 nothing = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < TR / 16 + MT + 1; ++i) buf_store_b128(nothing, nowhere, kOutOfRange - 16u * (unsigned)i);
  }
  float h_in = 0.f;
  int buf = 0;
  while (b < p.B) {
    const int t0 = c * TR;
#pragma unroll
    for (int i = 0; i < NV; ++i) *reinterpret_cast<Frag*>(x_at + buf * (TR * LDSROW) + i * RP * LDSROW) = pre[i];
    // one bit per token; tokens past the end read as padding
    unsigned long long resets = 0ull, pads = 0ull;
    if constexpr (FLAGS) { resets = __ballot(pre_fl & RGLRU_FLAG_RESET); pads = __ballot(pre_fl & RGLRU_FLAG_INACTIVE); }
    if (p.T - t0 < TR) pads |= ~0ull << (p.T - t0);
    if (p.first_reset && c == 0) resets |= 1ull;
    if (c == 0) h_in = pre_h0;
    const int bn = c + 1 < nT ? b : b + p.wg_per_unit, cn = c + 1 < nT ? c + 1 : 0;
    issue(bn, cn);
    lds_barrier();
    const IO* tile = &lds[buf][0];
    float a[EL], z[EL];
    const bool plain = TR == 64 ? (resets | pads) == 0ull : ((unsigned)resets | (unsigned)pads) == 0u;
    const unsigned my_resets = hf ? (unsigned)(resets >> (TR / 2)) : (unsigned)resets, my_pads = hf ? (unsigned)(pads >> (TR / 2)) : (unsigned)pads;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      f32x16 ua, ux;
      float xv[16];
      gate_mfma_held<IO, MT, NKG, KC>(tile, hw, mt, w.slab, w.r, hf, 0.0f, 0.0f, ua, ux, xv, NKG >= 8 ? 0 : w.kb);
      if (!FLAGS) rows_gates<false>(ua, ux, xv, sp, nba, nbx, mt == 0 ? my_resets : 0u, 0u, 0, a + 16 * mt, z + 16 * mt);
      else if (plain) rows_gates<false>(ua, ux, xv, sp, nba, nbx, 0u, 0u, 0, a + 16 * mt, z + 16 * mt);
      else rows_gates<true>(ua, ux, xv, sp, nba, nbx, my_resets, my_pads, 16 * mt, a + 16 * mt, z + 16 * mt);
    }
    if constexpr (!FLAGS) {
      // tokens past the end leave the state alone
      if (p.T - t0 < TR) {
#pragma unroll
        for (int e = 0; e < EL; ++e) {
          const bool past = (my_pads >> e) & 1u;
          a[e] = past ? 1.0f : a[e];
          z[e] = past ? 0.0f : z[e];
        }
      }
    }
    // the carry is known, so the lower half-wave's run is walked for its end, then both for their states
    float h = h_in;
#pragma unroll
    for (int e = 0; e < EL; ++e) h = fmaf(a[e], h, z[e]);
    const float h_mid = xhalf(h, hf);
    h = hf ? h_mid : h_in;
    unsigned char* my = stage + WaveStage<TR>::row_offset(hf * EL) + w.r * 2;
    const rsrc_t rck = make_rsrc(p.ckpt + (long long)b * p.ckpt_nC * W, (unsigned)p.ckpt_nC * uW * 4u);
    const unsigned ck_off = w.ch_ok ? ((unsigned)((t0 + hf * EL) >> 4) * uW + ch) * 4u : kOutOfRange;
#pragma unroll
    for (int e = 0; e < EL; ++e) {
      h = fmaf(a[e], h, z[e]);
      *reinterpret_cast<IO*>(my + e * WaveStage<TR>::kRowBytes) = (IO)h;
      if ((e & 15) == 15) BufIo<float>::store(h, rck, w.ch_ok ? ck_off + (unsigned)(e >> 4) * uW * 4u : kOutOfRange, 0u);   // state after every 16 tokens
    }
    const float h_hi = xhalf(h, hf);
    h_in = hf ? h : h_hi;
    BufIo<float>::store(h_in, rhl, w.ch_ok && hf == 0 && c == nT - 1 ? ((unsigned)b * uW + ch) * 4u : kOutOfRange, 0u);
    wave_lds_fence();
    const int rows = (p.T - t0) < TR ? (p.T - t0) : TR;
    const rsrc_t ry = make_rsrc((const IO*)p.y + ((long long)b * p.T + t0) * W, (unsigned)rows * row_bytes);
    stage_flush<TR>(stage, ry, row_bytes, (unsigned)(w.k * p.bw + w.slab * 32) * 2u, w.lane, w.slab_ok && (!PAD || w.slab * 32 + (w.lane & 3) * 8 < p.bw));
    wave_lds_fence();
    buf ^= 1;
    b = bn; c = cn;
  }
}

int fwd_rows_tile(int nkg, bool flags, int64_t workgroups) { return rows_long_tiles(nkg, flags, workgroups) ? 64 : 32; }
int fwd_rows_per_cu(int nkg, bool flags) { return rows_occ(nkg, flags); }

int launch_fwd_rows(const FusedArgs& a, int nkg, bool pad, hipStream_t s) {
  const dim3 grid((unsigned)(a.wg_per_unit * a.units));
  const bool flags = a.flags != nullptr;
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, s, a); };
#define RGLRU_ROWS_CASE(N, F, MT) pad ? launch(fwd_rows_kernel<N, true, F, MT>) : launch(fwd_rows_kernel<N, false, F, MT>)
  if (nkg == 2) flags ? (RGLRU_ROWS_CASE(2, true, 1)) : (RGLRU_ROWS_CASE(2, false, 1));
  else if (nkg == 4) flags ? (RGLRU_ROWS_CASE(4, true, 1)) : (RGLRU_ROWS_CASE(4, false, 1));
  else {
    const bool long_tiles = rows_long_tiles(nkg, flags, (int64_t)a.wg_per_unit * a.units);
    if (nkg == 6) flags ? (RGLRU_ROWS_CASE(6, true, 2)) : long_tiles ? (RGLRU_ROWS_CASE(6, false, 2)) : (RGLRU_ROWS_CASE(6, false, 1));
    else flags ? (RGLRU_ROWS_CASE(8, true, 2)) : long_tiles ? (RGLRU_ROWS_CASE(8, false, 2)) : (RGLRU_ROWS_CASE(8, false, 1));
  }
#undef RGLRU_ROWS_CASE
  return check_launch("fwd");
}

}  // namespace rglru

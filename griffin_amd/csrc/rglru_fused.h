// Shared by the translation units of the fused RG-LRU kernels (forward, backward, decode): kernel
// arguments, the wave/tile helpers the kernels have in common, and the host-side checks and launch
// helpers of their entry points.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "rglru_device.h"
#include "rglru_host.h"
#include "rglru_layout.h"

namespace rglru {

// ------------------------------------------------------------------------------------------
// Parameter preparation
// ------------------------------------------------------------------------------------------
struct PrepArgs {
  const void* w_a; const void* w_x; const void* b_a; const void* b_x; const void* lambda;
  void* wg; float* bias; float* sp; float* cs; float* dsp; void* w2t;
  int W, nb, bw, bwp, Wp, vec_dtype;
  int vec_ok;                          // 16-bit weights, blocks of a multiple of 8 channels, 16-byte aligned: eight elements per thread
  int rows_ok;                         // 16-bit weights whose rows are whole 16-byte vectors (blocks of a multiple of 8 channels)
  float c;
  uint4* clear; long long clear_n;     // optional: a workspace region to zero in the same launch
  // optional: two arrays of `stack_n` 16-byte vectors each to lay one behind the other in the same launch
  const uint4* stack_from[2]; uint4* stack_to; long long stack_n;
};

// Element i of a vector stored as fp32 or bf16 (RGLRU_F32 / RGLRU_BF16).
RGLRU_DEVICE float load_vec(const void* p, long long i, int dtype) {
  return dtype == RGLRU_BF16 ? (float)((const __bf16*)p)[i] : ((const float*)p)[i];
}
RGLRU_DEVICE void store_vec(void* p, long long i, float v, int dtype) {
  if (dtype == RGLRU_BF16) ((__bf16*)p)[i] = (__bf16)v; else ((float*)p)[i] = v;
}

RGLRU_DEVICE float log_sigmoid(float v) {
  return v >= 0.f ? -log1pf(expf(-v)) : v - log1pf(expf(v));
}

// Per-channel constants of padded channel kp: the two biases, c log sigmoid(Lambda) in natural and
// binary logarithm, and the factor of the Lambda gradient.
RGLRU_DEVICE void prepare_channel(const PrepArgs& p, int kp) {
  const int k = kp / p.bwp, o = kp - k * p.bwp;
  float ba = 0.f, bx = 0.f, sp = 0.f, cs = 0.f, dsp = 0.f;
  if (o < p.bw) {
    const int ch = k * p.bw + o;
    ba = load_vec(p.b_a, ch, p.vec_dtype); bx = load_vec(p.b_x, ch, p.vec_dtype);
    const float lam = load_vec(p.lambda, ch, p.vec_dtype);
    const float ls = log_sigmoid(lam);
    cs = p.c * ls;
    sp = cs * kLog2e;
    dsp = p.c / (1.0f + expf(lam));          // c * d/dLambda log sigmoid(Lambda) = c * sigmoid(-Lambda)
  }
  p.bias[kp] = ba; p.bias[p.Wp + kp] = bx; p.sp[kp] = sp; p.cs[kp] = cs; p.dsp[kp] = dsp;
}

template <typename IO>
__global__ void prepare_kernel(PrepArgs p) {
  const long long per_gate = (long long)p.nb * p.bwp * p.bwp;
  const long long n_w = 2 * per_gate;
  const long long total = 2 * n_w + p.Wp;
  long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long z = i; z < p.clear_n; z += stride) p.clear[z] = make_uint4(0u, 0u, 0u, 0u);
  for (long long z = i; z < 2 * p.stack_n; z += stride) p.stack_to[z] = z < p.stack_n ? p.stack_from[0][z] : p.stack_from[1][z - p.stack_n];
  if (sizeof(IO) == 2 && p.vec_ok) {
    // wg is a copy of [w_a ; w_x], 16 bytes a thread; the padding is zero in both.  w2t[k][j][2 o + gate] is the transpose of both: a thread turns eight j of four o, and the
    // lanes of a wave cover 64 j x 32 o, so that both sides move in runs of 128 bytes.  With a thread a vector of w2t, its eight elements gathered
    // one by one, W2560 in 8 gate blocks took 15.5 us with the clearing for B1 T32768, so 10.9; a training step of B2 T2048 W2560 167 and 160.
    const int row8 = p.bwp / 8, tiles_j = (p.bwp + 63) / 64, tiles_o = p.bwp / 32;             // row8: vectors per row of wg
    const long long per_gate8 = per_gate / 8, n_w8 = 2 * per_gate8;
    const long long turned = (long long)p.nb * tiles_j * tiles_o * 64;
    const bf16x8 zero = Io<__bf16>::zero();
    for (; i < turned + n_w8 + p.Wp; i += stride) {
      if (i < turned) {
        const int lane = (int)i & 63;
        long long tile = i >> 6;
        const int to = (int)(tile % tiles_o); tile /= tiles_o;
        const int tj = (int)(tile % tiles_j), k = (int)(tile / tiles_j);
        const int j = tj * 64 + (lane >> 3) * 8, o = to * 32 + (lane & 7) * 4;
        if (j >= p.bwp) continue;
        const bool there = j < p.bw && o < p.bw;                                      // whole vectors: bw is a multiple of 8
        const long long at = there ? ((long long)k * p.bw + o) * p.bw + j : 0;        // W[k][o][j]
        const int next = there ? p.bw : 0;
        bf16x8 a[4], x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          a[u] = *(const bf16x8*)((const __bf16*)p.w_a + at + (long long)u * next);
          x[u] = *(const bf16x8*)((const __bf16*)p.w_x + at + (long long)u * next);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const bf16x8 v = {a[0][e], x[0][e], a[1][e], x[1][e], a[2][e], x[2][e], a[3][e], x[3][e]};
          ((bf16x8*)p.w2t)[((long long)k * p.bwp + j + e) * (2 * row8) + o / 4] = there ? v : zero;
        }
      } else if (i < turned + n_w8) {
        const long long e8 = i - turned;
        const int gate = e8 >= per_gate8;
        const unsigned rem = (unsigned)(e8 - gate * per_gate8), row = rem / (unsigned)row8, j = (rem - row * (unsigned)row8) * 8u;
        const unsigned k = row / (unsigned)p.bwp, o = row - k * (unsigned)p.bwp;
        const bool there = (int)o < p.bw && (int)j < p.bw;
        const bf16x8 v = *(const bf16x8*)((const __bf16*)(gate ? p.w_x : p.w_a) + (there ? ((long long)k * p.bw + o) * p.bw + j : 0));
        ((bf16x8*)p.wg)[e8] = there ? v : zero;
      } else {
        prepare_channel(p, (int)(i - turned - n_w8));
      }
    }
    return;
  }
  for (; i < total; i += stride) {
    if (i < n_w) {
      int gate = (int)(i / per_gate);
      long long rem = i - gate * per_gate;
      int k = (int)(rem / ((long long)p.bwp * p.bwp));
      int oj = (int)(rem - (long long)k * p.bwp * p.bwp);
      int o = oj / p.bwp, j = oj - o * p.bwp;
      float v = 0.f;
      if (o < p.bw && j < p.bw) {
        const IO* src = (const IO*)(gate ? p.w_x : p.w_a);
        v = (float)src[((long long)k * p.bw + o) * p.bw + j];
      }
      ((IO*)p.wg)[i] = (IO)v;
    } else if (i >= n_w + p.Wp) {
      // w2t[k][j][2 * o + gate]
      long long e = i - n_w - p.Wp;
      const long long per_block = 2ll * p.bwp * p.bwp;
      int k = (int)(e / per_block);
      int rem = (int)(e - (long long)k * per_block);
      int j = rem / (2 * p.bwp), kap = rem - j * 2 * p.bwp;
      int o = kap >> 1, gate = kap & 1;
      float v = 0.f;
      if (o < p.bw && j < p.bw) {
        const IO* src = (const IO*)(gate ? p.w_x : p.w_a);
        v = (float)src[((long long)k * p.bw + o) * p.bw + j];
      }
      ((IO*)p.w2t)[e] = (IO)v;
    } else {
      prepare_channel(p, (int)(i - n_w));
    }
  }
}


// ------------------------------------------------------------------------------------------
// Arguments common to the fused kernels
// ------------------------------------------------------------------------------------------
struct FusedArgs {
  // tensors
  const void* x; const void* pre; const void* wg; const float* bias; const float* sp; const float* cs; const void* w2t;
  const float* h0; const uint8_t* flags;
  void* y; float* h_last;                                 // forward
  const void* dy; const float* dh_last;                   // backward in
  void* dx; void* du_a; void* du_x; float* dh0;           // backward out
  float* h_state; const float* h_prev;                    // decode step: state out, state in (may be the same)
  const void* gate_v;                                     // decode step: y = h * gelu_tanh(gate_v) when set
  long long ld_gate;                                      // ... elements between rows of gate_v (>= W)
  // reverse scan behind an output gate (GATED): dy is the gradient at y * gelu_tanh(gate_v), the gradient at gate_v goes to dv
  // (rows ld_dv apart) and its column sums to dv_partial[sequence or workgroup of the unit][W]
  void* dv; long long ld_dv; float* dv_partial;
  // block forward: x = causal depthwise conv of the rows at `x` (taps by lag, carried rows in conv_state),
  // out `gated` = y * gelu_tanh(gate_v); x_out, y and conv_new_state are optional outputs
  const void* conv_state; const void* conv_taps; const void* conv_bias;
  void* x_out; void* conv_new_state; void* gated;
  long long ld_x;                                         // elements between rows of x (>= W)
  int conv_k, conv_vec_dtype;
  // chain forward that also prepares (rglru_hip_prepare_fwd): the caller's parameters, the image to build from
  // them and the workspace region to zero, all in the forward launch
  PrepArgs prep;
  // workspace
  float* ckpt; rec_t* rec_a; unsigned* ticket;
  unsigned* fail; float* partial; float* dw_partial;
  // geometry
  int B, T, W, nb, bw, bwp, S, Wp, groups, units;
  int bpu;                                                // gate blocks per unit (packed narrow blocks), else 1
  long long rows_total;                                   // B * T, the row count of one block of `pre`
  int nC, nCf, ckpt_nC, wg_per_unit, aligned, full_slabs, queues, flags_vec;
  int dw_bf16;                                            // fast backward: per-workgroup weight-gradient sums stored as bf16 (unpadded blocks)
  int xcd_map;                                            // wide blocks: the workgroups that share a block's x tiles sit on one XCD
  int first_reset;                                        // token 0 of every sequence carries RGLRU_FLAG_RESET (and flags is null)
  unsigned bw_magic;                                      // decode step: ceil(2^32 / bw), channel / bw as a multiply-high (channel < 2^16)
  long long limit;
};

// Ticket queues.  A unit's (chunk, sequence) tiles are dealt to `queues` counters: queue j owns the
// sequences b = j, j + queues, ...; its tickets enumerate them chunk-major, i.e. in chain order.  A
// workgroup serves queue wg_in_unit % queues.  Spreading the tickets keeps same-address atomics rare.
struct Queue {
  unsigned* counter; int first_b, n_b; long long tiles;
};
RGLRU_DEVICE Queue make_queue(const FusedArgs& p, int unit, int wg_in_unit, int chunks) {
  Queue q;
  const int j = wg_in_unit % p.queues;
  q.counter = p.ticket + unit * kMaxQueues + j;
  q.first_b = j;
  q.n_b = (p.B - j + p.queues - 1) / p.queues;
  q.tiles = (long long)q.n_b * chunks;
  return q;
}

// Identity of the wave inside its unit; shared by the kernels below.
struct WaveId {
  int lane, r, hf, wave, unit, wg_in_unit, k, slab, o, ch, kp;
  int tile_col, kb;          // first channel of the unit's x tile; offset of the wave's block inside it
  bool slab_ok, ch_ok;
};

// Width of the x tile of the kernels with register-held weights.  Blocks of 64 or 32 channels are
// packed two or four to a unit, so the four waves of a workgroup always have a slab each.
constexpr int kPackedWidth = 128;

// Waves of a chain kernel's workgroup (fwd_chain_kernel, bwd_delta_chain_kernel: one workgroup per chain).
constexpr int kChainWaves = 16;

RGLRU_DEVICE WaveId wave_identity(const FusedArgs& p, int block, bool scalar_wave = false) {
  WaveId w;
  w.lane = threadIdx.x & 63; w.r = w.lane & 31; w.hf = w.lane >> 5;
  // scalar_wave: the wave index is made known to be wave-uniform, so what derives from it (slab, block, buffer
  // descriptors) stays in scalar registers; where registers are short that costs more than it saves
  w.wave = scalar_wave ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : (int)(threadIdx.x >> 6);
  w.unit = block % p.units; w.wg_in_unit = block / p.units;
  if (p.xcd_map) {
    // Workgroups go to the eight XCDs round-robin by index and each XCD has its own L2.  The `groups` units
    // of a wide block stage the same x tiles: index = xcd + 8 * slot keeps the members of a (block,
    // workgroup number) pair in consecutive slots of one XCD, so the tile comes from memory once.  The grid
    // is rounded up to whole rounds of eight pairs; a workgroup number past the end means "nothing to do".
    const int xcd = block & 7, slot = block >> 3;
    const int pair = xcd + 8 * (slot / p.groups);
    w.unit = (pair % p.nb) * p.groups + slot % p.groups;
    w.wg_in_unit = pair / p.nb;
  }
  if (p.bpu > 1) {
    // packed: the unit covers bpu consecutive blocks of S slabs each (bpu * S = waves per workgroup)
    const int blk = w.wave / p.S, k = w.unit * p.bpu + blk;
    w.slab = w.wave - blk * p.S;
    w.slab_ok = k < p.nb;
    w.k = w.slab_ok ? k : p.nb - 1;
    w.tile_col = w.unit * p.bpu * p.bw; w.kb = blk * p.bwp;
  } else {
    w.k = w.unit / p.groups;
    w.slab = (w.unit % p.groups) * kWaves + w.wave;
    w.slab_ok = w.slab < p.S;
    w.tile_col = w.k * p.bw; w.kb = 0;
  }
  w.o = w.slab * 32 + w.r;
  w.ch_ok = w.slab_ok && w.o < p.bw;
  w.ch = w.k * p.bw + (w.ch_ok ? w.o : 0);
  w.kp = w.k * p.bwp + (w.slab_ok ? w.o : 0);
  return w;
}

// Channel behind column `col` of a unit's 128-wide tile, or -1.  Blocks take bwp columns of it each (their width rounded up
// to whole 32-channel slabs); the columns a block does not fill hold zeros, and nothing is stored for them.
template <bool PAD, bool WIDE = false>
RGLRU_DEVICE int tile_channel(const FusedArgs& p, int unit, int tile_col, int col) {
  if constexpr (!PAD) return tile_col + col;
  if constexpr (WIDE) return col < p.bw ? tile_col + col : -1;       // the tile is one block
  const int blk = col / p.bwp, c = col - blk * p.bwp, k = unit * p.bpu + blk;
  return c < p.bw && blk < p.bpu && k < p.nb ? k * p.bw + c : -1;
}

// ------------------------------------------------------------------------------------------
// x tile staging.  A tile is TR consecutive rows (tokens, or sequences for the decode step) of one
// gate block, kept in LDS with row stride KS + HW elements.
// ------------------------------------------------------------------------------------------
template <typename IO>
RGLRU_DEVICE typename Io<IO>::Frag load_x_frag(const FusedArgs& p, const IO* xmat, long long grow,
                                               long long rows_total, int k, int col) {
  typedef Io<IO> Tr;
  typename Tr::Frag v = Tr::zero();
  if (grow < rows_total) {
    const IO* src = xmat + grow * (long long)p.W + (long long)k * p.bw + col;
    if (p.aligned && col + Tr::HW <= p.bw) {
      v = *reinterpret_cast<const typename Tr::Frag*>(src);
    } else {
#pragma unroll
      for (int e = 0; e < Tr::HW; ++e) if (col + e < p.bw) v[e] = src[e];
    }
  }
  return v;
}

// Gate pre-activations of one tile, generic variant (any block width, weights streamed from
// memory, K staged through LDS in slices of KCMAX).  On return ua/ux hold W x + b for the wave's
// slab (register v of tile mt <-> local row hf*16*MT + 16*mt + v) and xv the matching x values.
// Every thread of the workgroup must call this (it contains barriers).
// Narrow blocks are packed like those of the kernels with register-held weights (p.bpu > 1: the tile holds the unit's blocks side
// by side, `first_k` the first of them, and the wave's block starts at column kb), so that all four waves have a slab.
// Bound by the latency of its loads: all vectors of a slice are requested before the first is used (through a descriptor that
// ends with the rows, so no load sits in a branch), and the weights of 32 input channels while the 32 before them are
// multiplied.
template <typename IO, int MT>
RGLRU_DEVICE void gate_tile_generic(const FusedArgs& p, const IO* xmat, long long row0, long long rows_total,
                                    int first_k, int kb, int slab, bool slab_ok, const IO* w_a_row, const IO* w_x_row,
                                    float bias_a, float bias_x, IO* lds,
                                    f32x16 (&ua)[MT], f32x16 (&ux)[MT], float (&xv)[16 * MT]) {
  typedef Io<IO> Tr;
  typedef typename Tr::Frag Frag;
  constexpr int TR = 32 * MT;
  constexpr int KG = Tr::KG, HW = Tr::HW, KCMAX = Tr::KCMAX;
  constexpr int LDSROW = KCMAX + HW;
  constexpr int NV = TR * (KCMAX / HW) / kThreads;         // vectors a thread loads of a slice, at most
  constexpr int GK = 32 / KG;                              // K groups of 32 input channels
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, hf = lane >> 5;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int v = 0; v < 16; ++v) { ua[mt][v] = bias_a; ux[mt][v] = bias_x; }
#pragma unroll
  for (int e = 0; e < 16 * MT; ++e) xv[e] = 0.f;

  const unsigned row_bytes = (unsigned)p.W * (unsigned)sizeof(IO);
  const long long left = rows_total - row0;
  const rsrc_t rx = make_rsrc(xmat + row0 * p.W, left <= 0 ? 0u : (unsigned)(left < TR ? left : TR) * row_bytes);
  Frag xin[NV];
  auto request = [&](int kc0) {
    const int kcw = (p.bwp - kc0) < KCMAX ? (p.bwp - kc0) : KCMAX;
    const int vecs = kcw / HW, per_row = vecs * p.bpu;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + i * kThreads;
      const int row = idx / per_row, at = idx - row * per_row, blk = at / vecs, col = kc0 + (at - blk * vecs) * HW;
      const bool there = row < TR && first_k + blk < p.nb;
      const unsigned off = (unsigned)row * row_bytes + (unsigned)((first_k + blk) * p.bw + col) * (unsigned)sizeof(IO);
      if (p.aligned) {                                     // a vector lies wholly inside or outside its block
        xin[i] = buf_load_frag<Frag>(rx, there && col < p.bw ? off : kOutOfRange);
      } else {
#pragma unroll
        for (int e = 0; e < HW; ++e)
          xin[i][e] = (IO)BufIo<IO>::load(rx, there && col + e < p.bw ? off + (unsigned)(e * sizeof(IO)) : kOutOfRange, 0u);
      }
    }
  };
  Frag fa[2][GK], fx[2][GK];
  auto weights = [&](int set, int col) {                   // past the end: the last 32 channels again
    const int c = col < p.bwp ? col : p.bwp - 32;
#pragma unroll
    for (int g = 0; g < GK; ++g) {
      fa[set][g] = *reinterpret_cast<const Frag*>(w_a_row + c + g * KG);
      fx[set][g] = *reinterpret_cast<const Frag*>(w_x_row + c + g * KG);
    }
  };
  weights(0, 0);
  for (int kc0 = 0; kc0 < p.bwp; kc0 += KCMAX) {           // one slice when blocks are packed: they are narrow
    const int kcw = (p.bwp - kc0) < KCMAX ? (p.bwp - kc0) : KCMAX;
    const int per_row = kcw / HW * p.bpu;
    request(kc0);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + i * kThreads;
      const int row = idx / per_row, at = idx - row * per_row;   // the packed blocks' columns lie side by side
      if (row < TR) *reinterpret_cast<Frag*>(lds + row * LDSROW + at * HW) = xin[i];
    }
    __syncthreads();
    if (slab_ok) {
      auto multiply = [&](int set, int kk) {
#pragma unroll
        for (int g = 0; g < GK; ++g)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            const Frag xa = *reinterpret_cast<const Frag*>(lds + tile_row<MT>(mt, r) * LDSROW + kb + kk + g * KG + hf * HW);
            Tr::mma(ua[mt], xa, fa[set][g]);
            Tr::mma(ux[mt], xa, fx[set][g]);
          }
      };
      for (int kk = 0; kk < kcw; kk += 64) {               // a slice but the last is a multiple of 64 wide: set 0 starts each
        weights(1, kc0 + kk + 32);
        multiply(0, kk);
        if (kk + 32 < kcw) {
          weights(0, kc0 + kk + 64);
          multiply(1, kk + 32);
        }
      }
      const int own = slab * 32 - kc0;                    // first column of this wave's slab in the slice
      if (own >= 0 && own < kcw) {
#pragma unroll
        for (int e = 0; e < 16 * MT; ++e) xv[e] = (float)lds[(hf * 16 * MT + e) * LDSROW + kb + own + r];
      }
    }
    __syncthreads();
  }
}

// Register-resident weights: the wave's 32 rows of both gate matrices, NKG K groups each.  The last LDSG K
// groups can live in LDS instead (`spill`: [group][gate][lane] fragments private to the wave): where the registers
// run out, the compiler's own spill goes to scratch memory, whose reloads count as vector memory operations and
// make the wave wait for every load it has in flight.
template <typename IO, int NKG, int LDSG = 0>
struct HeldWeights {
  static constexpr int kRegs = NKG > 0 ? NKG - LDSG : 1;
  typename Io<IO>::Frag a[kRegs], x[kRegs];
  RGLRU_DEVICE void load(const IO* w_a_row, const IO* w_x_row, typename Io<IO>::Frag* spill = nullptr, int lane = 0) {
    if constexpr (NKG > 0) {
#pragma unroll
      for (int kg = 0; kg < NKG - LDSG; ++kg) {
        a[kg] = *reinterpret_cast<const typename Io<IO>::Frag*>(w_a_row + kg * Io<IO>::KG);
        x[kg] = *reinterpret_cast<const typename Io<IO>::Frag*>(w_x_row + kg * Io<IO>::KG);
      }
#pragma unroll
      for (int g = 0; g < LDSG; ++g) {
        spill[(2 * g) * 64 + lane] = *reinterpret_cast<const typename Io<IO>::Frag*>(w_a_row + (NKG - LDSG + g) * Io<IO>::KG);
        spill[(2 * g + 1) * 64 + lane] = *reinterpret_cast<const typename Io<IO>::Frag*>(w_x_row + (NKG - LDSG + g) * Io<IO>::KG);
      }
    }
  }
};

// MFMA phase for register-held weights, one accumulator tile: the whole block width (NKG * KG
// columns) is in LDS with row stride NKG * KG + HW.  Also returns the 16 x values of the tile in
// accumulator layout.
template <typename IO, int MT, int NKG, int TW = NKG * Io<IO>::KG, int LDSG = 0>
RGLRU_DEVICE void gate_mfma_held(const IO* lds, const HeldWeights<IO, NKG, LDSG>& hw, int mt, int slab, int r, int hf,
                                 float bias_a, float bias_x, f32x16& ua, f32x16& ux, float (&xv)[16], int kb = 0,
                                 const typename Io<IO>::Frag* spill = nullptr, int lane = 0) {
  typedef Io<IO> Tr;
  typedef typename Tr::Frag Frag;
  constexpr int KG = Tr::KG, HW = Tr::HW;
  constexpr int LDSROW = TW + HW;                          // the tile is TW columns wide; the block starts at kb
#pragma unroll
  for (int v = 0; v < 16; ++v) { ua[v] = bias_a; ux[v] = bias_x; }
  const IO* row = lds + tile_row<MT>(mt, r) * LDSROW + kb + hf * HW;
#pragma unroll
  for (int kg = 0; kg < NKG - LDSG; ++kg) {
    Frag xa = *reinterpret_cast<const Frag*>(row + kg * KG);
    Tr::mma(ua, xa, hw.a[kg]);
    Tr::mma(ux, xa, hw.x[kg]);
  }
#pragma unroll
  for (int g = 0; g < LDSG; ++g) {
    Frag xa = *reinterpret_cast<const Frag*>(row + (NKG - LDSG + g) * KG);
    Tr::mma(ua, xa, spill[(2 * g) * 64 + lane]);
    Tr::mma(ux, xa, spill[(2 * g + 1) * 64 + lane]);
  }
#pragma unroll
  for (int e = 0; e < 16; ++e) xv[e] = (float)lds[(hf * 16 * MT + 16 * mt + e) * LDSROW + kb + slab * 32 + r];
}

// Flags of a lane's run of 16 consecutive tokens, two bits per token (token e at bits 2e, 2e + 1);
// tokens past the end of the sequence read as inactive.  When the sequence length is a multiple of
// 16 and the flag array is 16-byte aligned (flags_vec), a run is wholly inside or outside the
// sequence and its flags are one 16-byte load.
RGLRU_DEVICE unsigned pack_flag_bytes(unsigned d) {
  unsigned t = d & 0x03030303u;
  t = (t | (t >> 6)) & 0x000F000Fu;
  return (t | (t >> 12)) & 0xFFu;
}
RGLRU_DEVICE unsigned flag_run(const FusedArgs& p, long long token_row, int t_first) {
  // first_reset: "every sequence starts a document" without a flag array (the run that holds token 0)
  const unsigned first = (p.first_reset && t_first == 0) ? RGLRU_FLAG_RESET : 0u;
  if (p.flags_vec) {
    if (t_first >= p.T) return 0xAAAAAAAAu;
    if (!p.flags) return first;
    const uint4 w = *reinterpret_cast<const uint4*>(p.flags + token_row);
    return pack_flag_bytes(w.x) | (pack_flag_bytes(w.y) << 8) | (pack_flag_bytes(w.z) << 16) | (pack_flag_bytes(w.w) << 24) | first;
  }
  // any length and alignment: sixteen byte loads in flight together, those past the end dropped by their offset
  const int n = p.T - t_first;
  unsigned bits = first | (n >= 16 ? 0u : n <= 0 ? 0xAAAAAAAAu : 0xAAAAAAAAu << (2 * n));
  if (p.flags) {
    const rsrc_t rf = make_rsrc(p.flags, (unsigned)p.B * (unsigned)p.T);
    unsigned f[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) f[e] = (unsigned)__builtin_amdgcn_raw_buffer_load_b8(rf, e < n ? (unsigned)token_row + (unsigned)e : kOutOfRange, 0, 0);
#pragma unroll
    for (int e = 0; e < 16; ++e) bits |= (f[e] & 3u) << (2 * e);   // bits 2-3 belong to the block forward's convolution
  }
  return bits;
}

// ------------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------------
inline int check_geometry(const char* who, int64_t W, int64_t nb, int dtype) {
  if (dtype != RGLRU_F32 && dtype != RGLRU_BF16) return fail(RGLRU_E_ARG, "%s: dtype must be RGLRU_F32 or RGLRU_BF16, got %d", who, dtype);
  if (W <= 0 || nb <= 0 || W % nb != 0) return fail(RGLRU_E_ARG, "%s: width %lld is not divisible into %lld gate blocks", who, (long long)W, (long long)nb);
  if (W / nb > 512) return fail(RGLRU_E_UNSUPPORTED, "%s: gate block width %lld exceeds the supported maximum of 512", who, (long long)(W / nb));
  if (W >= (1 << 24)) return fail(RGLRU_E_UNSUPPORTED, "%s: width too large", who);
  return RGLRU_OK;
}

// Sizes the kernels address with 32-bit offsets.  Tiles and per-sequence slices of the workspace are
// reached through buffer descriptors whose lane offsets are 32-bit and whose "dropped access" offset
// is 0x7ffffff0, so every such extent has to stay below 2^31 bytes: the checkpoints of one sequence
// (the fp32 state after every 16 tokens, 4 W bytes each; the carry records of a sequence are no larger)
// and the [B, W] fp32 state tensors.
inline int check_extents(const char* who, int64_t B, int64_t T, int64_t W) {
  if (B * T * W >= (1ll << 40) || B * T >= (1ll << 31)) return fail(RGLRU_E_UNSUPPORTED, "%s: tensor too large", who);
  const int64_t slots = 4 * ((T + 63) / 64);              // checkpoint slots per sequence
  if (slots * W * 4 >= (1ll << 31))
    return fail(RGLRU_E_UNSUPPORTED, "%s: one sequence of %lld tokens x %lld channels exceeds the 2 GiB per-sequence workspace limit; split the sequence and carry the state", who, (long long)T, (long long)W);
  if (B * W * 4 >= (1ll << 31)) return fail(RGLRU_E_UNSUPPORTED, "%s: state tensor [%lld, %lld] too large", who, (long long)B, (long long)W);
  return RGLRU_OK;
}

inline size_t elem_size(int dtype) { return dtype == RGLRU_BF16 ? 2 : 4; }

inline void fill_common(FusedArgs& a, const Geometry& g, const void* prep, int dtype) {
  PrepLayout pl = make_prep_layout(g, elem_size(dtype));
  const char* pb = (const char*)prep;
  a.wg = pb + pl.wg; a.bias = (const float*)(pb + pl.bias); a.sp = (const float*)(pb + pl.sp); a.cs = (const float*)(pb + pl.cs);
  a.w2t = pb + pl.w2t;
  a.W = (int)g.W; a.nb = (int)g.nb; a.bw = (int)g.bw; a.bwp = (int)g.bwp; a.S = (int)g.S; a.Wp = (int)g.Wp;
  a.groups = (int)g.groups; a.units = (int)g.units; a.bpu = 1;
  a.limit = spin_limit();
  a.full_slabs = (g.bw % 32 == 0) ? 1 : 0;
}

inline const float* finish_dsp(const Geometry& g, const void* prep, int dtype) {
  return (const float*)((const char*)prep + make_prep_layout(g, elem_size(dtype)).dsp);
}

inline int is_aligned(const void* ptr, int64_t W, int64_t bw, size_t es) {
  return ((uintptr_t)ptr % 16 == 0) && ((W * (int64_t)es) % 16 == 0) && ((bw * (int64_t)es) % 16 == 0);
}

// K groups of the kernels for narrow blocks with register-held weights (2, 4, 6, 8: slabs of 32 channels), or 0.  A block
// of any multiple of 8 channels up to 128 takes them, padded to whole slabs in LDS and registers (narrow_padded), although an
// 8-wide block then computes on four times its channels: the portable kernels stream the weights and finish the gradients in
// GEMM kernels of their own.  Forward + backward (forward alone) in us, portable -> padded, width 768:
//   B8 T2048   8-wide blocks 531 -> 310 (100 -> 69), 16: 273 -> 168 (57 -> 46), 40: 222 -> 155, 48: 183 -> 119, 96: 217 -> 115, 120: 173 -> 111
//   B1 T8192   8: 292 -> 180 (62 -> 50), 16: 165 -> 112 (37 -> 33), 40: 142 -> 111, 48: 118 -> 90, 72: 142 -> 110
//   B2 T256    forward alone 12.6-18.0 -> 7.9-8.6 (forward + backward is bound by the host)
inline int narrow_groups(const Geometry& g, int dtype, int aligned) {
  if (narrow_padded(g) && g.W >= (1 << 22)) return 0;     // 64 rows of fp32 past the reach of a lane's offset
  return dtype == RGLRU_BF16 && aligned && g.bw % 8 == 0 && g.bwp <= 128 ? (int)(g.bwp / 16) : 0;
}

// K steps of 32 channels of the decode kernels on 16 x 16 tiles (gate blocks of 16 .. 384 channels in steps
// of 16, 16-bit storage, aligned rows), or 0 for the portable decode kernels
inline int step16_groups(const Geometry& g, int dtype, int aligned) {
  if (dtype != RGLRU_BF16 || !aligned || g.bw % 16 || g.bw > 384) return 0;
  return (int)(g.bwp / 32);
}

// ... and for the blocks wider than a workgroup's four slabs whose weights the forward and the
// gate-gradient kernels hold in registers: K groups of the padded width (whole 32-channel slabs), or 0.  A block of any multiple
// of 8 channels takes them (`padded` as above): at B8 T1000 W1216 (152 channels) the portable kernels took 274 us, forward and
// backward, these 187.
inline int wide_groups(const Geometry& g, int dtype, int aligned) {
  return dtype == RGLRU_BF16 && aligned && g.bw % 8 == 0 && g.bwp > 128 && g.bwp <= 384 ? (int)(g.bwp / 16) : 0;
}
inline bool wide_padded(const Geometry& g) { return g.bw != g.bwp; }

#define RGLRU_DISPATCH(KERNEL, grid, stream, args, dtype, nkg)                                         \
  do {                                                                                                 \
    if ((dtype) == RGLRU_BF16) {                                                                       \
      if ((nkg) == 8) hipLaunchKernelGGL((KERNEL<__bf16, 8>), grid, dim3(kThreads), 0, stream, args);  \
      else if ((nkg) == 4) hipLaunchKernelGGL((KERNEL<__bf16, 4>), grid, dim3(kThreads), 0, stream, args); \
      else if ((nkg) == 2) hipLaunchKernelGGL((KERNEL<__bf16, 2>), grid, dim3(kThreads), 0, stream, args); \
      else hipLaunchKernelGGL((KERNEL<__bf16, 0>), grid, dim3(kThreads), 0, stream, args);             \
    } else {                                                                                           \
      hipLaunchKernelGGL((KERNEL<float, 0>), grid, dim3(kThreads), 0, stream, args);                   \
    }                                                                                                  \
  } while (0)

inline int launch_clear(char* base, size_t begin, size_t end, hipStream_t s) {
  long long words = (long long)(end - begin) / 4;
  int cb = (int)((words + 1023) / 1024); if (cb > 2048) cb = 2048; if (cb < 1) cb = 1;
  hipLaunchKernelGGL(clear_words_kernel, dim3(cb), dim3(256), 0, s, (unsigned*)(base + begin), words);
  return check_launch("workspace clear");
}

// Optional event bracket around the main kernel of an entry point (measurement hook).
inline std::atomic<int> g_timing{0};
struct TimingSlot { hipEvent_t start = nullptr, stop = nullptr; bool armed = false; };
inline TimingSlot& timing_slot(int which) {
  static TimingSlot slots[4];       // process-wide: backward runs on PyTorch's autograd thread
  return slots[which];
}
struct KernelTimer {
  TimingSlot* slot = nullptr; hipStream_t stream;
  KernelTimer(int which, hipStream_t s) : stream(s) {
    if (!g_timing.load(std::memory_order_relaxed)) return;
    slot = &timing_slot(which);
    if (!slot->start && (hipEventCreate(&slot->start) != hipSuccess || hipEventCreate(&slot->stop) != hipSuccess)) { slot = nullptr; return; }
    (void)hipEventRecord(slot->start, stream);
  }
  ~KernelTimer() { if (slot) { (void)hipEventRecord(slot->stop, stream); slot->armed = true; } }
};

// Narrow blocks share a unit (see kPackedWidth), in the kernels with register-held weights and in the portable ones (nkg 0):
// without that a 64-wide block leaves two of a workgroup's four waves without a slab.
inline void pack_units(FusedArgs& a, const Geometry& g, int nkg) {
  if (nkg == 4 || nkg == 2 || (nkg == 0 && g.S <= 2)) {
    a.bpu = kPackedWidth / (int)g.bwp;
    a.units = (int)((g.nb + a.bpu - 1) / a.bpu);
  }
}

inline int pick_wg_per_unit(int units, long long tiles_per_unit, int per_cu, long long cap) {
  long long target = (long long)num_compute_units() * per_cu;
  long long n = (target + units - 1) / units;
  if (n > tiles_per_unit) n = tiles_per_unit;
  if (n > cap) n = cap;
  if (n < 1) n = 1;
  return (int)n;
}

// How many ticket queues a unit's workgroups share.  Queue j owns the sequences j, j + q, ... and is served by
// the workgroups j, j + q, ...; the launch ends with the queue that has the most sequences per workgroup, so
// take the q that makes that ratio smallest (9 sequences on 16 workgroups: one queue, not nine of which seven
// have two workgroups and two have one).  Among equals the largest q, which spreads the ticket atomics.
inline int pick_queues(long long B, int wg) {
  long long qmax = B < wg ? B : wg;
  if (qmax > kMaxQueues) qmax = kMaxQueues;
  int best = 1;
  long long best_num = B, best_den = wg;                  // one queue: B sequences on wg workgroups
  for (int q = 2; q <= qmax; ++q) {
    long long num = 0, den = 1;
    for (int j = 0; j < q; ++j) {
      const long long n = (B - j + q - 1) / q, w = (wg - j + q - 1) / q;
      if (n * den > num * w) { num = n; den = w; }
    }
    if (num * best_den <= best_num * den) { best = q; best_num = num; best_den = den; }
  }
  return best;
}


// rglru_fwd_rows.hip: the forward of batches large enough that every workgroup can own whole sequences (16-bit storage, blocks of
// up to 128 channels).
int fwd_rows_tile(int nkg, bool flags, int64_t workgroups);
int fwd_rows_per_cu(int nkg, bool flags);
int launch_fwd_rows(const FusedArgs& a, int nkg, bool pad, hipStream_t s);

// Whether the forward runs one workgroup per chain (fwd_chain_kernel) instead of tiles with look-back:
// 0 = by shape, 1 = never, 2 = whenever that kernel covers the shape (tests).
inline std::atomic<int> g_chain_forward{0};
inline bool fwd_chain_pays(int64_t B, int64_t T, int64_t W) {    // W: channels with the padding of their blocks
  const int mode = g_chain_forward.load(std::memory_order_relaxed);
  if (mode == 1) return false;
  if (mode == 2) return true;
  // Two time models, in microseconds for the forward and the reverse scan together, fitted to both kernel
  // pairs timed on 358 shapes (widths 512 to 4096, blocks of 32 to 128 channels, 16 to 8192 chains, 128 to 8192
  // tokens); the faster model wins.  A chain workgroup fills a compute unit, so the chains run in
  // ceil(chains / units) rounds, each as long as its sequence (a start-up cost, then a time per token that
  // grows with the share of the units that are busy, since they share the memory system); the tiled kernels
  // spread any shape over the whole chip, pay two longer launches plus one for the parameters, and their time
  // per token is 1.1 to 1.2 times the chain kernels' when those fill their rounds.
  static const int units = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) n = 0;
    return n;
  }();
  if (units <= 0) return false;
  const double chains = (double)B * (double)(W / 32), tokens = (double)T;
  const double rounds = std::ceil(chains / units), last = (chains - (rounds - 1) * units) / units;
  const double full_round = 4.7 + tokens * (0.01465 + 0.01208), last_round = 4.7 + tokens * (0.01465 + 0.01208 * last);
  const double t_chain = 6.6 + (rounds - 1) * full_round + last_round;
  const double work = chains * tokens * (256.0 / units);
  const double t_tiled = std::max(31.4, 24.2 + 1.025e-4 * work + 0.0030 * tokens);
  return t_chain < t_tiled;
}

}  // namespace rglru

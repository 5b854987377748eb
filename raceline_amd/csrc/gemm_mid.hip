// The prefill GEMM for calls whose output has too few 128 x 256 tiles to fill the chip
// (gemm.hip's workgroup tile): batched decode, short prompts, the last chunk of a prompt,
// the output head. The same products as gemm4_kernel, one output element at a time: every
// value is the same chain of 32x32x16 MFMA steps, per-group scale FMAs and bias steps in the
// same order, so a row has gemm4_kernel's bits whichever of the two runs it.
//
// Each wave owns 32 features over 32 MT token rows and all of (its split's) K; a workgroup
// is four waves side by side over the same rows.
//  - The codes and scales go straight from memory to registers, R group pairs ahead: a wave
//    is the only reader of its features, so they gain nothing from the LDS, and R pairs of
//    loads (2.3 KB each) per wave keep the weight stream in flight with few waves on a CU.
//  - The activation rows (prepped as for gemm4_kernel) go through an R-stage LDS ring filled
//    by LDS-DMA, shared by the workgroup's waves, chunks XOR-swizzled by the row.
//  - One hand-over per group pair: in the middle of pair q, once its fragments are all in
//    registers, every wave waits for its own loads of pair q + 1 and passes one barrier,
//    after which pair q's LDS stage is free and pair q + R is issued into it.
//  - The MFMAs of a group run beside the scale FMAs of the group (or row tile) before it and
//    the code conversion of the group after it.
#include "gemm.h"
#include "gemm_bias.h"
#include "q4_tile.h"
#include "../../include/rlq.h"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>

namespace rlq {

constexpr int kMidWaves = 4;             // (two per workgroup measured the same on small grids, up to 1.6 times slower on full ones)
constexpr int kMidCols = 32 * kMidWaves; // features of a workgroup
constexpr int kMidRow = 256;             // LDS bytes of one row of a stage: one pair of groups, 128 fp16
constexpr int kMidBiasChunk = 8;         // bias steps loaded at a time after it

template <int MT> constexpr int mid_stage_bytes() { return 32 * MT * kMidRow; }

// Where one lane's loads of a pair come from.
template <int DMA>
struct MidSrc {
  const u32x4 *w, *s;
  const _Float16 *x;
  uint32_t wrange, srange, xrange, wvoff, svoff;
  uint32_t aoff[DMA];           // the lane's activation chunk of DMA i
  int K, pb, n, wave, c0;       // the split's first pair and its pairs; the logical chunk of DMA 0
};

// One load of pair q (counted from the split's first): part 0 or 1 of its codes, part 2 its
// scale words, into registers (mid_weights), or one of the wave's DMAs of its activation
// rows into stage s of the ring (mid_rows). Every pair makes the same number of loads, so that
// the waits count them: past the last
// pair the descriptors are empty, and the loads touch no memory. The pair's offset goes in
// the scalar operand, which the range check does not see: it stays inside a tile (p < 2 G4)
// and, for inputs below K, inside a row; where the last pair holds one group (an odd number
// of groups), the chunks of the other take an offset past every range and read zeros.
template <int DMA>
__device__ __forceinline__ void mid_weights(const MidSrc<DMA> &src, int part, int q, u32x4 (&wq)[2], uint64_t &sp) {
  const bool live = q < src.n;
  const int p = live ? src.pb + q : 0;
  if (part < 2) {
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(src.w, live ? src.wrange : 0u);
    wq[part] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, src.wvoff + 512u * part, p * 1024, 0));
  } else {
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(src.s, live ? src.srange : 0u);
    sp = __builtin_bit_cast(uint64_t,
                            __builtin_amdgcn_raw_buffer_load_b64(rs, src.svoff, (p >> 1) * 256 + 8 * (p & 1), 0));
  }
}

template <int MT, int DMA>
__device__ __forceinline__ void mid_rows(const MidSrc<DMA> &src, unsigned char *lds, int s, int q, int i) {
  const bool live = q < src.n;
  const int p = live ? src.pb + q : 0;
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(src.x, live ? src.xrange : 0u);
  const bool tail = 128 * (p + 1) > src.K;
  // the rows of DMA i are 16 i past DMA 0's: the same logical chunk
  dma16(rx, lds, s * mid_stage_bytes<MT>() + (src.wave + kMidWaves * i) * 1024,
        tail && (src.c0 & 8) ? kFarOffset : src.aoff[i], 256 * p);
}

template <int BOOK, int SD, int MT, int R>
__global__ __launch_bounds__(64 * kMidWaves, 2) void gemm_mid_kernel(GemmArgs a, int accum) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int kStage = mid_stage_bytes<MT>();
  constexpr int kDma = 8 * MT / kMidWaves;                        // activation LDS-DMAs per wave and pair
  constexpr int kParts = BOOK == kAffine ? 3 : 2;         // weight loads per wave and pair
  constexpr int kLoads = kDma + kParts;                   // vector memory loads per wave and pair
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.K / kGroup, G4 = quads_of(a.K), GP = 2 * G4;
  const int NP = (G + 1) / 2;
  const int T = tiles_of(a.N);
  const int split = blockIdx.y, S = gridDim.y;            // split K as gemm4_kernel splits it
  const int pb = split * a.np_split;
  const int NPs = min(NP, pb + a.np_split) - pb;

  // each XCD takes a contiguous range of the tiles, token blocks fastest, so that the
  // workgroups that read the same weights share an L2
  const int mblocks = (a.M + 32 * MT - 1) / (32 * MT);
  const int nwg = gridDim.x, wid = blockIdx.x, xcd = wid & 7, xq = nwg >> 3, xr = nwg & 7;
  const int lin = (xcd < xr ? xcd * (xq + 1) : xr * (xq + 1) + (xcd - xr) * xq) + (wid >> 3);
  const int nb = lin / mblocks, mb = lin - nb * mblocks;
  const int m0 = mb * 32 * MT;
  const int tw = 2 * (nb * kMidWaves + wave);                     // the wave's first 16-row weight tile

  // lane l: column c32 of the wave's 32 features (row cr of tile tt), half h (see gemm4_kernel)
  const int h = lane >> 5, c32 = lane & 31, tt = c32 >> 4, cr = c32 & 15;
  const int tiles = max(0, min(T, tw + 2) - tw);
  MidSrc<kDma> src;
  src.w = a.codes + (size_t)min(tw, T) * GP * 64;
  src.s = a.sb + (size_t)min(tw, T) * G4 * 16;
  src.x = a.x;
  src.wrange = (uint32_t)tiles * GP * 1024u;
  src.srange = BOOK == kAffine ? (uint32_t)tiles * G4 * 256u : 0u;
  src.xrange = (uint32_t)((size_t)a.M * a.x_stride * 2);
  src.wvoff = (uint32_t)tt * GP * 1024u + 256u * h + 16u * cr;
  src.svoff = (uint32_t)tt * G4 * 256u + 16u * cr;
  src.K = a.K; src.pb = pb; src.n = NPs; src.wave = wave;
  src.c0 = (lane & 15) ^ ((4 * wave + (lane >> 4)) & 15);
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int r = 4 * (wave + kMidWaves * i) + (lane >> 4), c = (lane & 15) ^ (r & 15);
    src.aoff[i] = m0 + r < a.M ? (uint32_t)(((size_t)(m0 + r) * a.x_stride + 8 * c) * 2) : kFarOffset;
  }
  uint32_t aoff[2][4];                                    // A fragment offsets within a row tile of a stage
#pragma unroll
  for (int gg = 0; gg < 2; ++gg)
#pragma unroll
    for (int i = 0; i < 4; ++i) aoff[gg][i] = (uint32_t)(c32 * kMidRow + (((8 * gg + 2 * i + h) ^ cr) << 4));

  u32x4 wq[R][2];
  uint64_t sp[R];   // one 64-bit value: as two words the loop carried copies of the second, waiting for the load

  // the A fragment of step i of group gg, row tile mt, from stage s
  auto frag = [&](int s, int gg, int mt, int i) -> half8 {
    return *reinterpret_cast<const half8 *>(lds + s * kStage + mt * 32 * kMidRow + aoff[gg][i]);
  };
  // codes of step i, group gg: word 2i + h, i.e. read (i & 1), element 2 gg + (i >> 1)
  auto conv = [&](int s, int gg, int i) -> half8 {
    const uint32_t u = wq[s][i & 1][2 * gg + (i >> 1)];
    if constexpr (BOOK == kAffine) return nib8_to_half8_oddx16(u);
    else return native8_to_half8<BOOK>(u);
  };

  f32x16 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x16{};

  // Affine: the bias product, an MFMA over the group sums' pieces (see gemm4_kernel, whose
  // steps and order these are): st_lo .. st_pro before the K loop, the rest after it. Each
  // wave reads its rows' pieces and its features' scale quads from memory (L2); steps past
  // the range load zeros and add nothing.
  const int bsteps = a.gs_stride / 16;
  const int st_lo = split * bsteps / S, st_hi = (split + 1) * bsteps / S;
  const int st_pro = BOOK == kAffine ? min(st_hi, st_lo + kBiasProSteps) : st_lo;
  BiasSrc bias;
  bias.rgs = make_rsrc(a.gs, BOOK == kAffine ? (uint32_t)((size_t)a.M * a.gs_stride * 2) : 0u);
  bias.rsb = make_rsrc(src.s, src.srange);
  bias.svoff = src.svoff;
  bias.M = a.M; bias.gs_stride = a.gs_stride; bias.G4 = G4; bias.m0 = m0; bias.c32 = c32; bias.h = h;
  // the first R pairs; the weights of the last of them follow in the first round
  auto fill = [&]() {
#pragma unroll
    for (int s = 0; s < R; ++s) {
#pragma unroll
      for (int i = 0; i < kDma; ++i) mid_rows<MT>(src, lds, s, s, i);
      if (s + 1 < R) {
#pragma unroll
        for (int i = 0; i < kParts; ++i) mid_weights(src, i, s, wq[s], sp[s]);
      }
      __builtin_amdgcn_sched_barrier(0);      // in the order they are used
    }
  };
  if constexpr (BOOK == kAffine) {
    u32x4 bv[kBiasProSteps], ba[kBiasProSteps][MT];
    bias_load<SD, MT>(bias, bv, ba, st_lo, st_pro);
    __builtin_amdgcn_sched_barrier(0);        // requested before the ring: they complete first
    fill();
    __builtin_amdgcn_sched_barrier(0);
    bias_mul<SD, MT>(bv, ba, h, acc);
  } else {
    fill();
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vmcnt((R - 1) * kLoads));   // pair 0 has landed for this wave
  asm volatile("s_barrier" ::: "memory");   // and for every wave

  // A round is eight MFMAs: both groups of a pair (MT = 1) or one group (MT = 2), as two
  // chains of four (the two groups, the two row tiles), taken in turn so that no MFMA waits
  // for the one before it. (Native books chain all of K: with one row tile that is a single
  // chain, in group order.) Beside them run the 32 scale FMAs of the round before, the code
  // conversion of the next step and, in the first four steps, the reads of the next round's
  // fragments; by the next hand-over those have long returned.
  constexpr bool kOneChain = BOOK != kAffine && MT == 1;
  half8 fr[2][8], bf[2];
  f32x16 pp[2][2];
  float sc[2] = {0.0f, 0.0f};           // the scales of the round before's two chains
  pp[0][0] = pp[0][1] = pp[1][0] = pp[1][1] = f32x16{};
  // step j of a round of pair slot s (MT = 2: group gg): its fragment and its code word
  auto step_frag = [&](int s, int gg, int j) -> half8 {
    if constexpr (kOneChain) return frag(s, j >> 2, 0, j & 3);
    else if constexpr (MT == 1) return frag(s, j & 1, 0, j >> 1);
    else return frag(s, gg, j & 1, j >> 1);
  };
  auto step_codes = [&](int s, int gg, int j) -> half8 {
    if constexpr (kOneChain) return conv(s, j >> 2, j & 3);
    else if constexpr (MT == 1) return conv(s, j & 1, j >> 1);
    else return conv(s, gg, j >> 1);
  };
#pragma unroll
  for (int j = 0; j < 8; ++j) fr[0][j] = step_frag(0, 0, j);
  bf[0] = step_codes(0, 0, 0);

  // PAR: which half of the double buffers the round uses; gg: its group (MT = 2)
  auto round = [&](auto slot_c, auto par_c, int gg, int q) {
    constexpr int SL = decltype(slot_c)::value, NX = (SL + 1) % R, PV = (SL + R - 1) % R, PAR = decltype(par_c)::value;
    const bool last = MT == 1 || gg == 1;             // the pair's last round: the next one reads the next stage
    float scn[2] = {0.0f, 0.0f};
    if constexpr (BOOK == kAffine) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        scn[c] = scale_f32<SD>((uint16_t)(sp[SL] >> (32 * (MT == 1 ? c : gg)))) * kTwo24;
        asm volatile("" : "+v"(scn[c]));              // taken now: the slot's next load is issued in the next round
      }
    }
    if (last) {
      // the pair's fragments are all in registers: its stage is free once every wave is
      // here, and pair q + 1's rows have landed when each wave's own part has
      // (MT = 2: the weights of this pair's first round have gone out since)
      __builtin_amdgcn_s_waitcnt(0x0070 | (waitcnt_vmcnt((R - 2) * kLoads + (MT == 1 ? 0 : kParts)) & 0xC00F));   // and lgkmcnt(0)
      asm volatile("s_barrier" ::: "memory");
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int c = j & 1, i = j >> 1;
      if (j < 4) {
        // (past the last pair: zeros, or stale rows nobody uses)
#pragma unroll
        for (int e = 2 * j; e < 2 * j + 2; ++e) fr[PAR ^ 1][e] = last ? step_frag(NX, 0, e) : step_frag(SL, 1, e);
      }
      // The loads go out a step or two apart: all of a pair's at once, right after the
      // barrier, queued behind those of the workgroup's other waves (about 60 cycles each).
      // Weights: the slot of the pair before, whose codes are all used; rows: this pair's
      // stage. The last load of a pair is a DMA (the wait above counts on it).
      if (MT == 1 || gg == 0) {
        if ((j & 1) && j / 2 < kParts) mid_weights(src, j / 2, q - 1 + R, wq[PV], sp[PV]);
      }
      if (last && (MT == 1 ? j == 2 || j == 6 : (j & 1) == 0)) mid_rows<MT>(src, lds, SL, q + R, MT == 1 ? j / 4 : j / 2);
      const half8 b = bf[(MT == 1 ? j : i) & 1];
      if (MT == 1 || c == 1) {                        // the next step's codes (MT = 2: both chains share them)
        const int nj = j + 1, slot = ((MT == 1 ? nj : i + 1)) & 1;
        bf[slot] = nj < 8 ? step_codes(SL, gg, nj) : last ? step_codes(NX, 0, 0) : step_codes(SL, 1, 0);
      }
      if constexpr (BOOK == kAffine) {
        pp[PAR][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[PAR][j], b, i == 0 ? f32x16{} : pp[PAR][c], 0, 0, 0);
        const int fc = j >> 2, fm = MT == 1 ? 0 : fc; // the FMAs' chain and row tile
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int v = 4 * (j & 3) + e;
          acc[fm][v] = __builtin_fmaf(sc[fc], pp[PAR ^ 1][fc][v], acc[fm][v]);
        }
        asm volatile("" : "+v"(acc[fm]));             // these FMAs stay beside this MFMA
      } else {
        const int mt = MT == 1 ? 0 : c;
        acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[PAR][j], b, acc[mt], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    sc[0] = scn[0];
    sc[1] = scn[1];
  };
  auto pair = [&](auto slot_c, int q) {
    if constexpr (MT == 1) {
      round(slot_c, std::integral_constant<int, decltype(slot_c)::value & 1>{}, 0, q);
    } else {
      round(slot_c, std::integral_constant<int, 0>{}, 0, q);
      round(slot_c, std::integral_constant<int, 1>{}, 1, q);
    }
  };
  static_assert(R % 2 == 0, "rounds alternate between the two halves of the buffers");
  // R pairs per iteration, one per stage, so that every register and LDS offset is known at
  // compile time. The pairs past the last one, up to a multiple of R, multiply zeros. (One
  // exit only: with an exit per pair the compiler copied the accumulators at each.)
  for (int q = 0; q < NPs; q += R) {
    [&]<int... SL>(std::integer_sequence<int, SL...>) {
      (pair(std::integral_constant<int, SL>{}, q + SL), ...);
    }(std::make_integer_sequence<int, R>{});
  }
  if constexpr (BOOK == kAffine) {
#pragma unroll
    for (int c = 0; c < 2; ++c)                // the last round's products: an even number of rounds, so pp[1]
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int fm = MT == 1 ? 0 : c;
        acc[fm][v] = __builtin_fmaf(sc[c], pp[1][c][v], acc[fm][v]);
      }
    for (int st0 = st_pro; st0 < st_hi; st0 += kMidBiasChunk) {
      u32x4 bv[kMidBiasChunk], ba[kMidBiasChunk][MT];
      bias_load<SD, MT>(bias, bv, ba, st0, st_hi);
      bias_mul<SD, MT>(bv, ba, h, acc);
    }
  }
  __builtin_amdgcn_s_waitcnt(0);              // no LDS-DMA outlives the workgroup's LDS

  // D of a 32x32 tile: lane l holds column l%32, rows 8 (v/4) + 4 (l/32) + v%4. Every value
  // the results still need (row factors, and y where it is added to) is loaded at once, from
  // an address clamped into the matrix, and only the stores look at the edges: a load inside
  // a per-element branch waited for memory once per element.
  const int n = 16 * tw + c32, nc = min(n, a.N - 1);
  const bool col = n < a.N;
  const bool acc_here = accum && split == 0;
  auto row_of = [&](int mt, int v) { return m0 + mt * 32 + 8 * (v >> 2) + 4 * h + (v & 3); };
  if constexpr (BOOK == kAffine) {
    float rs[MT][16];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) rs[mt][v] = a.rscale[min(row_of(mt, v), a.M - 1)];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mt][v] = mul_rounded(acc[mt][v], rs[mt][v]);   // undoes the prep's 2^e, exactly
  } else {
    const float rs_n = a.srow ? a.srow[nc] : 1.0f;                            // no row scales: the raw product
    if constexpr (BOOK == kInt16) {
      if (split == 0) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            acc[mt][v] = __builtin_fmaf(0.5f, a.asum[min(row_of(mt, v), a.M - 1)], acc[mt][v]);
      }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mt][v] = mul_rounded(acc[mt][v], rs_n);
  }
  if (acc_here) {
    float yv[MT][16];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) yv[mt][v] = a.y[(size_t)min(row_of(mt, v), a.M - 1) * a.y_stride + nc];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mt][v] = yv[mt][v] + acc[mt][v];
  }
  if (S == 1) {
    if (!col) return;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = row_of(mt, v);
        if (m < a.M) a.y[(size_t)m * a.y_stride + n] = acc[mt][v];
      }
    return;
  }

  // Split K (S = 2), as gemm4_kernel ends: both splits store their values (split 0 in y),
  // wait for them and count the arrival; the second to arrive adds the two in split order.
  float *const mine = split == 0 ? a.y : a.y_part + (size_t)(split - 1) * a.M * a.N;
  const int mstride = split == 0 ? a.y_stride : a.N;
  if (col) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = row_of(mt, v);
        if (m < a.M)
          __hip_atomic_store(mine + (size_t)m * mstride + n, acc[mt][v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
  }
  __builtin_amdgcn_s_waitcnt(0);                     // this wave's values are stored
  __syncthreads();                                   // and every wave's
  int *const arrival = reinterpret_cast<int *>(lds);   // the ring is done with
  if (threadIdx.x == 0) arrival[0] = __hip_atomic_fetch_add(a.cnt + lin, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (arrival[0] != S - 1) return;                   // uniform: the tile's last split goes on
  if (threadIdx.x == 0) __hip_atomic_store(a.cnt + lin, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (!col) return;
  const float *const other = split == 0 ? a.y_part : a.y;
  const int ostride = split == 0 ? a.N : a.y_stride;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    float p[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = min(row_of(mt, v), a.M - 1);
      p[v] = __hip_atomic_load(other + (size_t)m * ostride + n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = row_of(mt, v);
      if (m < a.M) a.y[(size_t)m * a.y_stride + n] = split == 0 ? acc[mt][v] + p[v] : p[v] + acc[mt][v];
    }
  }
}

// ------------------------------------------------------------------ host

template <int MT> constexpr int mid_ring() { return MT == 1 ? 8 : 4; }   // 64 KB of LDS

template <int BOOK, int SD, int MT>
static int launch_mid(const GemmArgs &a, int S, int accum, hipStream_t st) {
  static LdsOptIn opt;
  constexpr int R = mid_ring<MT>();
  auto kernel = gemm_mid_kernel<BOOK, SD, MT, R>;
  if (int rc = allow_large_lds(reinterpret_cast<const void *>(kernel), opt)) return rc;
  const int mblocks = (a.M + 32 * MT - 1) / (32 * MT), nblocks = (a.N + kMidCols - 1) / kMidCols;
  kernel<<<dim3(mblocks * nblocks, S), 64 * kMidWaves, (size_t)R * mid_stage_bytes<MT>(), st>>>(a, accum);
  RLQ_HIP(hipGetLastError());
  return 0;
}

template <int BOOK, int SD>
static int launch_mid_rows(int mt, const GemmArgs &a, int S, int accum, hipStream_t st) {
  return mt == 1 ? launch_mid<BOOK, SD, 1>(a, S, accum, st) : launch_mid<BOOK, SD, 2>(a, S, accum, st);
}

// Which kernel and tile take a call: the one of three estimated fastest (32 or 64 rows x 128
// features here, gemm4_kernel's 128 x 256), each as, in us,
//   once + pairs x (per_round x rounds of the chip + per_fill x fill) + (per_tile + split (S - 1)) x fill
// with fill = workgroups / CUs, rounds = fill rounded up, and the group pairs of a workgroup
// rounded up to the ones its loop runs (3, 8 or 4 LDS stages). A wave here is bound by its own
// instruction issue, and two workgroups on a CU take about as long as one after the other, so
// the rounds count; how full they are costs memory time and clock. Past three rounds the CUs
// drift apart, and a partial round counts half its empty part.
// The tiles here have one more term. Each 128 features read all rows, which an XCD's L2 (4 MB)
// holds for small calls; rows beyond it come from memory once per 128 features, at row_mb us per
// MB (from 2 MB of rows on, in full from 12 MB). The native books' waves have little to do
// beside those loads and pay the sum, the affine ones' scale FMAs hide most of the shorter of
// the two (the cube root of the sum of cubes). gemm4_kernel orders its tiles in blocks of 512
// rows and shows no such term.
// The books differ in what a code costs to convert (4 operations for eight fp4 codes, 13 for
// eight integer ones, shared by two row tiles at 64 rows), the affine ones in their scale FMAs
// and bias steps (twice as many for bf16), int16 in the launch that sums its rows first. Fitted
// to launches timed with their prep pass: K 128 .. 17408 (odd numbers of groups and split
// weights among them), N 16 .. 34816, 9 .. 4096 rows (to 16384 where N < 256), 600 to 734 calls
// a book. Against the fastest of the three the choice loses 0.2% (affine), 0.1% (integer books)
// and 0.3% (fp4) on average, and 4%, 5% and 6% at 99 of 100 calls. Without the rows' term, the
// rounding of the pairs and the split it took the 64-row tiles for large calls and was slower
// than gemm4_kernel alone: bf16 K = 16512, N = 2187 at 2762 rows 383 us for 266, fp4 K = 2240,
// N = 3877 at 1600 rows 46.1 for 36.5.
struct MidCost { double once, per_round, per_fill, per_tile, split, row_mb; };
constexpr MidCost kCost[5][3] = {   // affine with fp16 scales, int15, int16, fp4, affine with bf16 scales: gemm4, 32 rows, 64 rows
    {{10.4, 1.353, 0.537, 1.9, 20.2, 0}, {9.3, 0.359, 0.022, 1.1, 2.2, 0.0997}, {12.5, 0.511, 0.003, 3, 3.8, 0.1117}},
    {{4.4, 1.161, 0.477, 5.9, 8.6, 0}, {4.7, 0.358, 0.009, 0.4, 0.6, 0.001}, {4.3, 0.47, 0.004, 1.7, 0, 0.0193}},
    {{9.6, 1.207, 0.55, 5, 15.2, 0}, {7.9, 0.368, 0, 0.4, 2.7, 0.0073}, {7.6, 0.476, 0.008, 1.5, 3.4, 0.0171}},
    {{4, 1.016, 0.521, 5.9, 5.8, 0}, {4.3, 0.216, 0.023, 1.1, 1.5, 0.0229}, {4, 0.335, 0.046, 2, 0.2, 0.0206}},
    {{8.4, 1.447, 0.482, 5.6, 11.1, 0}, {8.5, 0.372, 0.029, 1.4, 0.9, 0.1222}, {12.3, 0.561, 0.003, 2.6, 0.7, 0.0953}}};
static_assert(kAffine == 0 && kInt15 == 1 && kInt16 == 2 && kFp4 == 3, "kCost's rows");
// Ties: what gemm4_kernel may be estimated slower by and still take a call, the margin that left
// the fewest calls slower than on the kernel they ran before (between boxes the two differ by
// 5% either way, as the clock does).
constexpr double mid_margin(int book) { return book == kInt15 || book == kInt16 ? 0.99 : 1.02; }

// a split call's tiles count their arrivals in the workspace's counters
bool gemm_mid_counters_fit(int mt, int M, int N, int S) {
  return S == 1 || (long long)((M + 32 * mt - 1) / (32 * mt)) * ((N + kMidCols - 1) / kMidCols) <= kGemmMaxCounters;
}

int gemm_mid_tiles(int book, int sd, int M, int K, int N, int S) {
  const int pairs = ((K / kGroup + 1) / 2 + S - 1) / S;
  const double rows_mb = 2e-6 * M * K, beyond = std::clamp((rows_mb - 2.0) / 10.0, 0.0, 1.0);
  const double read = rows_mb * ((N + kMidCols - 1) / kMidCols) * beyond;
  const MidCost *cost = kCost[book == kAffine && sd == RLQ_BF16 ? 4 : book];
  // the kernel of cost[i]: workgroups of rows x cols, and the pairs of one turn of its loop
  auto time = [&](int i, int rows, int cols, int stages) {
    const MidCost &c = cost[i];
    const long long wgs = (long long)((N + cols - 1) / cols) * ((M + rows - 1) / rows) * S;
    const double fill = wgs / 256.0, whole = (double)((wgs + 255) / 256);
    const double rounds = i > 0 && fill > 3.0 ? 0.5 * (whole + fill) : whole;
    const double run = (double)((pairs + stages - 1) / stages * stages);
    const double work = run * (c.per_round * rounds + c.per_fill * fill) + (c.per_tile + c.split * (S - 1)) * fill;
    const double mem = c.row_mb * read;
    return c.once + (book == kAffine ? std::cbrt(work * work * work + mem * mem * mem) : work + mem);
  };
  const double t4 = time(0, 128, 256, 3);
  const double t1 = mid_margin(book) * time(1, 32, kMidCols, mid_ring<1>());
  const double t2 = mid_margin(book) * time(2, 64, kMidCols, mid_ring<2>());
  if (t1 <= t2 && t1 < t4 && gemm_mid_counters_fit(1, M, N, S)) return 1;
  return t2 < t4 && gemm_mid_counters_fit(2, M, N, S) ? 2 : 0;
}

int launch_gemm_mid(int book, int sd, int mt, const GemmArgs &a, int S, int accum, hipStream_t st) {
  switch (book) {
    case kInt15: return launch_mid_rows<kInt15, 0>(mt, a, S, accum, st);
    case kInt16: return launch_mid_rows<kInt16, 0>(mt, a, S, accum, st);
    case kFp4: return launch_mid_rows<kFp4, 0>(mt, a, S, accum, st);
    default:
      return sd == RLQ_BF16 ? launch_mid_rows<kAffine, 1>(mt, a, S, accum, st)
                            : launch_mid_rows<kAffine, 0>(mt, a, S, accum, st);
  }
}

}  // namespace rlq

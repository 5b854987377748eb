// The affine prefill GEMM for calls of a few rows: batched decode, a draft's verification,
// very short prompts. The same products as gemm4_kernel (gemm.hip), in the same order per
// output element, so a row has its bits.
//
// gemm4's order is serial in K: group after group, acc = fma(s_g, x_g . q_g, acc). A wave that
// does everything for its 32 x 32 outputs (gemm_mid.hip) is bound by its own instruction
// issue, about 950 cycles per group pair, and with one row tile a weight of 4096 features has
// only 128 such waves. But the group products x_g . q_g do not depend on each other, so here
// twelve waves, the whole of a CU, share one 32 x 32 tile:
//  - eight producer waves take the group pairs in turn (wave w: pairs w, w + 8, ...), convert
//    the codes, form the two groups' products (eight MFMAs) and write them, with the scale
//    words, to the LDS;
//  - four accumulator waves, each with a quarter of the tile's rows, run the scale FMAs over
//    the groups in order, eight pairs behind. They also form the bias product (before the K
//    loop, while the first loads are in flight), and store the results.
// One barrier per eight pairs; the LDS holds two sets of products.
//
// The activations come straight to registers in operand order: the prep pass writes them
// here by 16-byte chunk, then row ([K / 8][M][8 halves]), so a fragment is two contiguous
// runs of rows and a wave needs no LDS stage to transpose through. Rows past M load as
// zeros; products of rows that do not exist are not written to the LDS (8 rows at a time).
//
// What bounds it: the CU's vector memory path (TA 77%, TD 89% busy at K = 12288, 27 rows), of
// which the activations are four fifths (8 KB a pair, the codes 2.3 KB). So where the chip has
// CUs to spare a workgroup takes 16 or 8 rows and others the rest. Measured with the prep pass,
// against gemm_mid_kernel: 4096 x 4096 at 9 / 32 / 64 rows 11.5 / 12.4 / 14.8 us (18.7, 19.4,
// 20.1); K = 12288, N = 4096 20.6 / 23.2 / 28.9 (40.5, 43.0, 43.7). Two workgroups of four
// producers and two accumulators per CU: 11.7 / 13.2 / 14.2 and 21.1 / 26.8 / 28.5.
#include "gemm.h"
#include "gemm_bias.h"
#include "q4_tile.h"
#include "../../include/rlq.h"

#include <type_traits>

namespace rlq {

constexpr int kFewProducers = 8, kFewAccs = 4;
constexpr int kFewThreads = 64 * (kFewProducers + kFewAccs);
constexpr int kFewBiasChunk = 8;
constexpr int kFewPairBytes = 2 * 4 * 1024;           // a pair's products: [group][quarter of the rows][lane] 16 bytes
constexpr int kFewScaleBytes = 512;                   // and its scale words: [lane] 8 bytes
constexpr int kFewSetBytes = kFewProducers * (kFewPairBytes + kFewScaleBytes);
constexpr int kFewMaxTiles = 256;                     // a workgroup per CU
constexpr int kFewMaxRows = 2048, kFewShortK = 320;   // see gemm_few_fits
constexpr int kFewLds = 2 * kFewSetBytes;             // 136 KB: one workgroup per CU

// What a producer wave reads (see few_codes, few_frag).
struct FewSrc {
  const u32x4 *w, *s;
  const _Float16 *x;
  uint32_t wrange, srange, xrange, wvoff, svoff, avoff;
  int K, M, pb, n, wave;
};

// Codes and scale words of the wave's pair of phase ph (pair 8 ph + wave of the split). Past
// the last pair the descriptors are empty and the loads read zeros. The pair's offset, in
// the scalar operand, stays inside a tile (p < 2 G4).
__device__ __forceinline__ void few_codes(const FewSrc &f, int ph, u32x4 (&wq)[2], uint64_t &sp) {
  const int q = kFewProducers * ph + f.wave;
  const bool live = q < f.n;
  const int p = live ? f.pb + q : 0;
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(f.w, live ? f.wrange : 0u), rs = make_rsrc(f.s, live ? f.srange : 0u);
  wq[0] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, f.wvoff, p * 1024, kNonTemporal));
  wq[1] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, f.wvoff + 512u, p * 1024, kNonTemporal));
  sp = __builtin_bit_cast(uint64_t,
                          __builtin_amdgcn_raw_buffer_load_b64(rs, f.svoff, (p >> 1) * 256 + 8 * (p & 1), 0));
}

// Where the A fragments of that pair start: chunk 16 p + 8 gg + 2 i + h of the lane's row for
// step i of group gg. The chunk's offset, in the scalar operand, stays inside the chunks
// below K except in the second group of an odd number of groups' last pair, which gets an
// empty descriptor and reads zeros.
struct FewRows {
  __amdgpu_buffer_rsrc_t r[2];   // per group
  int base;
};
__device__ __forceinline__ FewRows few_rows(const FewSrc &f, int ph) {
  const int q = kFewProducers * ph + f.wave;
  const bool live = q < f.n;
  const int p = live ? f.pb + q : 0;
  FewRows r;
  r.r[0] = make_rsrc(f.x, live ? f.xrange : 0u);
  r.r[1] = make_rsrc(f.x, live && 128 * p + 64 < f.K ? f.xrange : 0u);
  r.base = p * 256 * f.M;
  return r;
}
__device__ __forceinline__ half8 few_frag(const FewSrc &f, const FewRows &r, int gg, int i) {
  return __builtin_bit_cast(
      half8, __builtin_amdgcn_raw_buffer_load_b128(r.r[gg], f.avoff, r.base + (8 * gg + 2 * i) * 16 * f.M, 0));
}

template <int SD>
__global__ __launch_bounds__(kFewThreads, 3) void gemm_few_kernel(GemmArgs a, int rb, int accum) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.K / kGroup, G4 = quads_of(a.K), GP = 2 * G4;
  const int NP = (G + 1) / 2;
  const int T = tiles_of(a.N);
  const int split = blockIdx.y, S = gridDim.y;            // split K as gemm4_kernel splits it
  const int pb = split * a.np_split;
  const int NPs = min(NP, pb + a.np_split) - pb;
  const int F = (NPs + 2 * kFewProducers - 1) / (2 * kFewProducers) * 2;   // phases

  // row blocks fastest, a contiguous range per XCD: the workgroups that read the same weights
  // share an L2
  const int mblocks = (a.M + rb - 1) / rb;
  const int nwg = gridDim.x, wid = blockIdx.x, xcd = wid & 7, xq = nwg >> 3, xr = nwg & 7;
  const int lin = (xcd < xr ? xcd * (xq + 1) : xr * (xq + 1) + (xcd - xr) * xq) + (wid >> 3);
  const int nb = lin / mblocks, m0 = rb * (lin - nb * mblocks);
  const int rows_here = min(rb, a.M - m0), quarters = (rows_here + 7) / 8;   // of the tile's rows

  // lane l: column c32 of the 32 features (row cr of 16-row weight tile tt), half h
  const int h = lane >> 5, c32 = lane & 31, tt = c32 >> 4, cr = c32 & 15;
  const int tiles = max(0, min(T, 2 * nb + 2) - 2 * nb);
  FewSrc f;
  f.w = a.codes + (size_t)min(2 * nb, T) * GP * 64;
  f.s = a.sb + (size_t)min(2 * nb, T) * G4 * 16;
  f.x = a.x;
  f.wrange = (uint32_t)tiles * GP * 1024u;
  f.srange = (uint32_t)tiles * G4 * 256u;
  f.xrange = (uint32_t)((size_t)a.M * a.K * 2);
  f.wvoff = (uint32_t)tt * GP * 1024u + 256u * h + 16u * cr;
  f.svoff = (uint32_t)tt * G4 * 256u + 16u * cr;
  f.avoff = c32 < rows_here ? (uint32_t)(h * a.M + m0 + c32) * 16u : kFarOffset;
  f.K = a.K; f.M = a.M; f.pb = pb; f.n = NPs; f.wave = wave;

  float acc[4];                                           // accumulator waves: their quarters' values
  if (wave < kFewProducers) {
    u32x4 wq[2][2];
    uint64_t sp[2];
    half8 fr[2][8];                                       // fragment of step j of phase ph: fr[ph & 1][j]
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      few_codes(f, s, wq[s], sp[s]);
#pragma unroll
      for (int j = 0; j < 8; ++j) fr[s][j] = few_frag(f, few_rows(f, s), j & 1, j >> 1);
      __builtin_amdgcn_sched_barrier(0);                  // in the order they are used
    }
    // Step j: chain (group) j & 1, its MFMA step j >> 1, so that no MFMA waits for the one
    // before it. A fragment's register is refilled for the phase after next once its
    // MFMA is issued, the codes' once they are converted.
    auto phase = [&](auto slot_c, int ph) {
      constexpr int SL = decltype(slot_c)::value;
      f32x16 pp[2];
      const FewRows next = few_rows(f, ph + 2);
      half8 b = nib8_to_half8_oddx16(wq[SL][0][0]);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int c = j & 1, i = j >> 1;
        pp[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[SL][j], b, i == 0 ? f32x16{} : pp[c], 0, 0, 0);
        // codes of step i', group c': word 2i' + h, i.e. read (i' & 1), element 2 c' + (i' >> 1)
        if (j < 7) {
          const int c1 = (j + 1) & 1, i1 = (j + 1) >> 1;
          b = nib8_to_half8_oddx16(wq[SL][i1 & 1][2 * c1 + (i1 >> 1)]);
        }
        if (j > 0) fr[SL][j - 1] = few_frag(f, next, (j - 1) & 1, (j - 1) >> 1);
        if (j == 3) {
          // the phase before is complete: its products left for the LDS half a phase ago
          __builtin_amdgcn_s_waitcnt(0xC07F);             // lgkmcnt(0): this wave's are there
          asm volatile("s_barrier" ::: "memory");
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      fr[SL][7] = few_frag(f, next, 1, 3);
      uint64_t sw = sp[SL];
      asm volatile("" : "+v"(sw));                        // taken before the slot's next load
      unsigned char *set = lds + (ph & 1) * kFewSetBytes;
      *reinterpret_cast<uint64_t *>(set + kFewProducers * kFewPairBytes + wave * kFewScaleBytes + 8 * lane) = sw;
      few_codes(f, ph + 2, wq[SL], sp[SL]);
      unsigned char *out = set + wave * kFewPairBytes + 16 * lane;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (k < quarters)                               // uniform
            *reinterpret_cast<f32x4 *>(out + (4 * c + k) * 1024) =
                f32x4{pp[c][4 * k], pp[c][4 * k + 1], pp[c][4 * k + 2], pp[c][4 * k + 3]};
    };
    // one exit only (with an exit per phase the compiler carried copies of every fragment);
    // a phase past the last pair multiplies zeros
    for (int ph = 0; ph < F; ph += 2) {
      phase(std::integral_constant<int, 0>{}, ph);
      phase(std::integral_constant<int, 1>{}, ph + 1);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    asm volatile("s_barrier" ::: "memory");               // the last phase is complete
    if (S == 1) return;
  }
  const int quarter = wave - kFewProducers;               // accumulator wave: rows 8 quarter .. + 7 of the tile
  const int bsteps = a.gs_stride / 16;
  const int st_lo = split * bsteps / S, st_hi = (split + 1) * bsteps / S;
  const int st_pro = min(st_hi, st_lo + kBiasProSteps);
  const int n = 32 * nb + c32, nc = min(n, a.N - 1);
  const bool col = n < a.N;
  const int mrow = m0 + 8 * quarter + 4 * h;              // the lane's first row; registers 4 quarter + 0 .. 3 of the tile
  const bool acc_here = accum && split == 0;
  if (wave >= kFewProducers) {
    BiasSrc bias;
    bias.rgs = make_rsrc(a.gs, (uint32_t)((size_t)a.M * a.gs_stride * 2));
    bias.rsb = make_rsrc(f.s, f.srange);
    bias.svoff = f.svoff;
    bias.M = a.M; bias.gs_stride = a.gs_stride; bias.G4 = G4; bias.m0 = m0; bias.c32 = c32; bias.h = h;
    const bool rows = quarter < quarters;                 // uniform: the wave has rows to sum
    f32x16 full[1] = {f32x16{}};
    if (rows) {
      u32x4 bv[kBiasProSteps], ba[kBiasProSteps][1];
      bias_load<SD, 1>(bias, bv, ba, st_lo, st_pro);
      bias_mul<SD, 1>(bv, ba, h, full);
    }
    // the wave's four of the tile's 16 registers, and back (the MFMA rows are independent:
    // what the others hold is not used)
    f32x4 av = f32x4{full[0][0], full[0][1], full[0][2], full[0][3]};
#pragma unroll
    for (int q = 1; q < 4; ++q)
      if (quarter == q) av = f32x4{full[0][4 * q], full[0][4 * q + 1], full[0][4 * q + 2], full[0][4 * q + 3]};
    asm volatile("s_barrier" ::: "memory");               // the producers' barrier inside phase 0
    for (int ph = 0; ph < F; ++ph) {
      asm volatile("s_barrier" ::: "memory");             // phase ph is in the LDS
      if (!rows) continue;
      const unsigned char *set = lds + (ph & 1) * kFewSetBytes;
      const int pairs = min(kFewProducers, NPs - kFewProducers * ph);
      const unsigned char *in = set + quarter * 1024 + 16 * lane;
      // everything is requested at once (one LDS round trip per phase; what no producer wrote
      // is read and not used)
      uint64_t sw[kFewProducers];
      f32x4 p[kFewProducers][2];
#pragma unroll
      for (int w = 0; w < kFewProducers; ++w) {
        sw[w] = *reinterpret_cast<const uint64_t *>(set + kFewProducers * kFewPairBytes + w * kFewScaleBytes + 8 * lane);
#pragma unroll
        for (int c = 0; c < 2; ++c) p[w][c] = *reinterpret_cast<const f32x4 *>(in + w * kFewPairBytes + 4 * c * 1024);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int w = 0; w < kFewProducers; ++w) {
        if (w < pairs) {                                  // uniform
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const float sc = scale_f32<SD>((uint16_t)(sw[w] >> (32 * c))) * kTwo24;
#pragma unroll
            for (int e = 0; e < 4; ++e) av[e] = __builtin_fmaf(sc, p[w][c][e], av[e]);
          }
        }
      }
      __builtin_amdgcn_s_waitcnt(0xC07F);                 // lgkmcnt(0): the set may be overwritten after the next barrier
    }
    if (!rows && S == 1) return;
    // the bias steps the prologue left (long K, bf16 biases)
#pragma unroll
    for (int v = 0; v < 16; ++v) full[0][v] = quarter == v >> 2 ? av[v & 3] : 0.0f;
    for (int st0 = st_pro; st0 < st_hi; st0 += kFewBiasChunk) {
      u32x4 bv[kFewBiasChunk], ba[kFewBiasChunk][1];
      bias_load<SD, 1>(bias, bv, ba, st0, st_hi);
      bias_mul<SD, 1>(bv, ba, h, full);
    }
    float rs[4], yv[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = min(mrow + e, a.M - 1);
      rs[e] = a.rscale[m];
      if (acc_here) yv[e] = a.y[(size_t)m * a.y_stride + nc];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float val = full[0][e];
#pragma unroll
      for (int q = 1; q < 4; ++q) val = quarter == q ? full[0][4 * q + e] : val;
      val = mul_rounded(val, rs[e]);                      // undoes the prep's 2^e, exactly
      if (acc_here) val = yv[e] + val;
      acc[e] = val;
    }
    if (S == 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col && 4 * h + 8 * quarter + e < rows_here) a.y[(size_t)(mrow + e) * a.y_stride + n] = acc[e];
      return;
    }
    // Split K (S = 2), as gemm4_kernel ends: both splits store their values (split 0 in y),
    // wait for them and count the arrival; the second to arrive adds the two in split order.
    float *const mine = split == 0 ? a.y : a.y_part + (size_t)(split - 1) * a.M * a.N;
    const int mstride = split == 0 ? a.y_stride : a.N;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col && 4 * h + 8 * quarter + e < rows_here)
        __hip_atomic_store(mine + (size_t)(mrow + e) * mstride + n, acc[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);                        // this wave's values are stored
  }
  __syncthreads();                                        // and every wave's; the sets are done with
  int *const arrival = reinterpret_cast<int *>(lds);
  if (threadIdx.x == 0) arrival[0] = __hip_atomic_fetch_add(a.cnt + lin, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (arrival[0] != S - 1) return;                        // uniform: the tile's last split goes on
  if (threadIdx.x == 0) __hip_atomic_store(a.cnt + lin, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (wave < kFewProducers || !col) return;
  const float *const other = split == 0 ? a.y_part : a.y;
  const int ostride = split == 0 ? a.N : a.y_stride;
  float p[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    p[e] = __hip_atomic_load(other + (size_t)min(mrow + e, a.M - 1) * ostride + n, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (4 * h + 8 * quarter + e < rows_here) a.y[(size_t)(mrow + e) * a.y_stride + n] = split == 0 ? acc[e] + p[e] : p[e] + acc[e];
}

// ------------------------------------------------------------------ host

// Taken where the call's tiles fill the CUs once at most (a workgroup is a CU's worth of waves
// and LDS): a second round costs a whole workgroup's time again, which the streaming kernels
// do not pay (4096 x 4096 at 96 rows, 384 tiles: 23.5 us against gemm_mid_kernel's 20.3; at
// 64 rows, 256 tiles: 14.8 against 20.1). Tall, narrow calls stay with those too: the prep
// pass writes each row's chunks 16 M bytes apart, eight rows to a cache line, which costs more
// than the GEMM gains past about 2000 rows (f16 K = 2752 .. 13504, N = 21 .. 39: 3043 rows 35.1
// us against 29.0, 3905 135.8 against 61.2, 8191 60.2 against 33.0; 1929 rows 27.1 against 28.0).
// With a short K there is little to prepare (K = 192 .. 320: 3114 rows 12.8 against 14.2, 7915
// 18.1 against 19.0; K = 512: 2843 rows 14.7 against 14.3).
static long long few_tiles(int M, int N, int S, int rb) {
  return (long long)((N + 31) / 32) * ((M + rb - 1) / rb) * S;
}
bool gemm_few_fits(int M, int K, int N, int S) {
  return (M <= kFewMaxRows || K <= kFewShortK) && few_tiles(M, N, S, 32) <= kFewMaxTiles;
}
bool gemm_few_counters_fit(int M, int N, int S) { return S == 1 || few_tiles(M, N, 1, 32) <= kGemmMaxCounters; }

int launch_gemm_few(int sd, const GemmArgs &a, int S, int accum, hipStream_t st) {
  static LdsOptIn o0, o1;
  const int nt = (a.N + 31) / 32;
  int rb = 32;
  while (rb > 8 && few_tiles(a.M, a.N, S, rb / 2) <= kFewMaxTiles) rb /= 2;
  const dim3 grid((a.M + rb - 1) / rb * nt, S);
  if (sd == RLQ_BF16) {
    if (int rc = allow_large_lds(reinterpret_cast<const void *>(&gemm_few_kernel<1>), o1)) return rc;
    gemm_few_kernel<1><<<grid, kFewThreads, kFewLds, st>>>(a, rb, accum);
  } else {
    if (int rc = allow_large_lds(reinterpret_cast<const void *>(&gemm_few_kernel<0>), o0)) return rc;
    gemm_few_kernel<0><<<grid, kFewThreads, kFewLds, st>>>(a, rb, accum);
  }
  RLQ_HIP(hipGetLastError());
  return 0;
}

}  // namespace rlq

// The prefill GEMM of the 4-bit formats (gemm.hip), called by the entry points of
// linear.hip, and the small activation-sum kernels it shares with them.
#pragma once

#include "rlq_common.h"

namespace rlq {

struct GemmArgs {
  const _Float16 *x;    // affine: the prepped activations [M][K]; native: x [M][x_stride]
  const u32x4 *codes;
  const u32x4 *sb;      // affine: scale/bias quads
  const uint16_t *gs;   // affine: the group sums' pieces, fp16 or bf16 bits [M][gs_stride]
  const float *srow;    // native books: row scales [N]
  const float *asum;    // kInt16: activation row sums [M]
  const float *rscale;  // affine: 2^-e per row, undoing the prep pass's prescale [M]
  float *y;
  float *y_part;        // split K: splits 1 .. S-1's partial products [S-1][M][N]
  int *cnt;             // split K: arrivals per output tile (zero between calls)
  int x_stride, M, K, N, y_stride, gs_stride;
  int np_split;         // group pairs per split (all of them when not split)
};

// Output tiles of one prefill launch whose K is split can count their arrivals in the
// workspace's counter bytes (see rlq_linear_workspace_bytes); larger calls launch in row
// chunks.
constexpr int kGemmMaxCounters = 1024;

// Bytes of workspace run_gemm4 needs (affine: the prepped activations and the split group
// sums; kInt16: row sums; a shape whose K is split: the partial products).
size_t gemm4_workspace(int book, int M, int K, int N);

// Affine: steps of the bias product that run before the K loop, the rest after it. A row's bits
// depend on the number, so all prefill kernels share it (it is what fits gemm4_kernel's stage 2).
constexpr int kBiasProSteps = 11;

// The prefill kernels and their tiles, with the same bits for every row; kRouteAuto takes the
// one estimated fastest (run_gemm4, gemm_mid_tiles).
enum PrefillRoute { kRouteAuto = 0, kRouteFull = 1, kRouteMid32 = 2, kRouteMid64 = 3, kRouteFew = 4 };

// The route a call of these sizes takes (its first launch: a split weight's rows go in chunks).
int prefill_route(int book, int sd, int M, int K, int N);

// route: kRouteAuto, or the kernel to run (an error where it cannot take the call).
// codes, sbq: the two sections of a packed matrix (q4_tile.h), or of rows [r0, r0 + N) of a
// larger one (r0 a multiple of 16: see packed_tile_offsets in linear.h). cnt: the
// kGemmMaxCounters arrival counters at the start of the linear workspace (zero).
int run_gemm4(int route, int book, const _Float16 *x, int x_stride, int M, int K, int N, const void *codes,
              const void *sbq, int sd, const float *srow, float *y, int y_stride, int accum, int *cnt, void *ws,
              size_t ws_bytes, hipStream_t st);

// The kernel for calls with too few 128 x 256 tiles (gemm_mid.hip): gemm_mid_tiles gives the
// 32-row tiles (1 or 2) of its workgroups' rows, or 0 where gemm4_kernel takes the call. Both
// kernels give the same bits.
int gemm_mid_tiles(int book, int sd, int M, int K, int N, int S);
bool gemm_mid_counters_fit(int mt, int M, int N, int S);   // a split launch's tiles have counters
int launch_gemm_mid(int book, int sd, int mt, const GemmArgs &a, int S, int accum, hipStream_t st);

// The affine kernel for a few rows (gemm_few.hip), the same bits again, and whether it takes a
// call; a.x: the prepped activations by chunk, then row ([K / 8][M][8 halves]).
bool gemm_few_fits(int M, int K, int N, int S);
bool gemm_few_counters_fit(int M, int N, int S);
int launch_gemm_few(int sd, const GemmArgs &a, int S, int accum, hipStream_t st);

// defined in linear.hip
void launch_row_sums(const _Float16 *x, int x_stride, int M, int K, float *asum, hipStream_t st);

}  // namespace rlq

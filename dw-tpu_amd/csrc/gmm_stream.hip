// Ragged grouped matmul for few rows per expert (decode batches): the same
// product, layouts and results as gmm_fp4.hip, built for streaming weights.
//
// What bounds it: HBM (6.6 TB/s reached at 198 rows over 256 experts, K = N =
// 4096: 188 us, the tiles 256; one token over 32 experts 49 -> 23).  With at most 32 rows per expert each weight byte
// feeds at most 64 FLOPs, so the packed weights' stream sets the time.
// The 512-column tiles of gmm_fp4.hip leave CUs idle when few experts hold
// rows (one token with top-8: 64 tiles for 256 CUs) and pay their start and
// epilogue once per tile with nothing else on the CU.
//
// Design: a wave owns 64 columns of one (expert, <= 32 rows) row tile over
// all of K, and shares nothing with other waves: no LDS stages, no barrier.
// Everything a K block of 128 reads -- 4 KiB of weights and 512 bytes of
// scales (each lane two dwords), the lhs fragments -- travels in a D-deep
// register ring, loaded in K order, so the wait for one block leaves the
// loads of the next D - 1 in flight (13.5 KiB of weights per wave at D = 3).
// A lane's 16 weight bytes are the 32 codes of one column (fp4.hip); the
// 16x16x32 operand of column block u wants, in lane row q, K chunk
// 2 v + q % 2 of the slot of lane row (2 (q / 2) + u % 2): one
// v_permlane16_swap per two dwords moves the pieces, 8 per K block and half.
// Every accumulator takes the MFMAs of gmm_fp4.hip's consumers in the same
// order, so a row's bits do not depend on which kernel computed it.
#include <algorithm>

#include "gmm_tiles.h"

namespace dwm {

constexpr int kStreamRows = 32;  // rows of a row tile

// The wave's tile: row tile rt of group g (row tiles of kStreamRows rows,
// innermost in the order so that the row tiles of one column tile run side
// by side on one XCD and share its L2's copy of the weights), column tile ct
// of n_ct.  The tile list is cut into 8 contiguous runs, one per XCD (blocks
// whose index is equal mod 8).  Every wave finds its tile alone: lane l holds
// the sizes of groups l PL .. + PL - 1, and prefix sums over the lanes give
// row starts, then row-tile counts.  Returns false when there is no tile.
//
// Group sizes are not checked by the host: negative ones count as empty, and
// every group is cut to the rows left below M before its tiles are counted,
// so the list holds the tiles of rows [0, M) and no others, and fits the grid
// (stream_grid) whatever the sizes sum to.
template <int PL>
__device__ __forceinline__ bool stream_tile(const int32_t *__restrict__ group_sizes, int num_groups, int go,
                                            int64_t e_local, int64_t M, int n_ct, int &g, int64_t &row0, int &rows,
                                            int &ct) {
  const int lane = threadIdx.x & 63;
  const int m32 = (int)min(M, (int64_t)0x7FFFFFFF);
  int sz[PL], rows_in = 0, tiles = 0;
#pragma unroll
  for (int i = 0; i < PL; ++i) sz[i] = group_sizes[min(lane * PL + i, num_groups - 1)];  // loads side by side
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    sz[i] = lane * PL + i < num_groups ? min(max(sz[i], 0), m32) : 0;
    rows_in += sz[i];
  }
  const int start = wave_inclusive_scan(rows_in) - rows_in;  // first row of the lane's first group
  int left = start >= 0 ? max(m32 - start, 0) : 0;           // (a sum past int32 is past M too)
  auto tiles_of = [&](int gi, int s) {
    return gi >= go && (int64_t)gi < (int64_t)go + e_local ? s / kStreamRows + (s % kStreamRows != 0 ? 1 : 0) : 0;
  };
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    sz[i] = min(sz[i], left);
    left -= sz[i];
    tiles += tiles_of(lane * PL + i, sz[i]);
  }
  const int upto = wave_inclusive_scan(tiles), before = upto - tiles;  // row tiles before the lane's groups
  const int64_t total = (int64_t)wave_last(upto) * n_ct;
  const int64_t run = (total + 7) >> 3;
  const int64_t j = blockIdx.x >> 3;
  const int64_t entry = (int64_t)(blockIdx.x & 7) * run + j;
  if (j >= run || entry >= total || entry > 0x7FFFFFFFll) return false;
  const int trow = (int)((uint32_t)entry / (uint32_t)n_ct);
  const uint64_t hit = __ballot(before <= trow && trow < upto);
  if (!hit) return false;
  const int sel = __ffsll((unsigned long long)hit) - 1;
  int rs = __builtin_amdgcn_readlane(start, sel);
  int tc = __builtin_amdgcn_readlane(before, sel);
  g = -1;
  int szg = 0;
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    if (g < 0) {
      const int s = __builtin_amdgcn_readlane(sz[i], sel);
      const int n = tiles_of(sel * PL + i, s);
      if (trow < tc + n) {
        g = sel * PL + i;
        szg = s;
      } else {
        rs += s;
        tc += n;
      }
    }
  }
  if (g < 0) return false;
  const uint32_t n = (uint32_t)tiles_of(g, szg), local = (uint32_t)entry - (uint32_t)tc * (uint32_t)n_ct;
  const int rt = (int)(local % n);
  ct = (int)(local / n);
  row0 = (int64_t)rs + (int64_t)rt * kStreamRows;
  rows = min(szg - rt * kStreamRows, kStreamRows);
  return true;
}

__device__ __forceinline__ bool find_stream_tile(const int32_t *__restrict__ group_sizes, int num_groups, int go,
                                                 int64_t e_local, int64_t M, int n_ct, int &g, int64_t &row0,
                                                 int &rows, int &ct) {
  if (num_groups <= 64) return stream_tile<1>(group_sizes, num_groups, go, e_local, M, n_ct, g, row0, rows, ct);
  if (num_groups <= 256) return stream_tile<4>(group_sizes, num_groups, go, e_local, M, n_ct, g, row0, rows, ct);
  return stream_tile<kMaxGroups / 64>(group_sizes, num_groups, go, e_local, M, n_ct, g, row0, rows, ct);
}

// One row tile of NH 16-row blocks x the wave's 64 columns.
template <int NH, int D, bool ACT>
__device__ __forceinline__ void stream_columns(const uint16_t *__restrict__ lhs, const int32_t *__restrict__ row_idx,
                                               int64_t lhs_rows, int64_t row0, int rows, int K,
                                               const uint8_t *__restrict__ w, const uint8_t *__restrict__ s,
                                               int64_t col0, int N, void *__restrict__ out, int out_f32,
                                               const void *bias, const GmmEpilogue &ep, float *ep_lds) {
  const int lane = threadIdx.x & 63, c16 = lane & 15, q = lane >> 4;
  const int KB = K >> 7;
  // lhs fragment of MFMA step v of 64-deep half f: row c16 of the block, K
  // chunk 4 (q / 2) + q % 2 + 2 v of the half's 8 (16 bytes each).
  uint32_t aoff[NH];
  const uint8_t *const abase = (const uint8_t *)(row_idx ? lhs : lhs + row0 * K);
#pragma unroll
  for (int hb = 0; hb < NH; ++hb) {
    const int r = min(16 * hb + c16, rows - 1);  // rows past the tile repeat its last row
    const int64_t src = row_idx ? gather_index(row_idx[row0 + r], lhs_rows) : r;
    aoff[hb] = (uint32_t)(src * K * 2) + 16u * (4 * (q >> 1) + (q & 1));
  }
  const uint32_t woff = lane * 16u, soff = (c16 + 32 * (q >> 1)) * 4u;
  u32x4_t wr[D][4], ar[D][NH][4];
  uint32_t sr[D][2];
  auto load = [&](int d, int kb) {
    const uint8_t *const wb = w + (int64_t)kb * 4096;
    const uint8_t *const sb = s + (int64_t)kb * 256;
    const uint8_t *const ab = abase + (int64_t)kb * 256;
#pragma unroll
    for (int i = 0; i < 4; ++i) wr[d][i] = __builtin_nontemporal_load((const u32x4_t *)(wb + 1024 * i + woff));
#pragma unroll
    for (int i = 0; i < 2; ++i) sr[d][i] = *(const uint32_t *)(sb + 64 * i + soff);
#pragma unroll
    for (int hb = 0; hb < NH; ++hb)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        ar[d][hb][i] = *(const u32x4_t *)(ab + 128 * (i >> 1) + 32 * (i & 1) + aoff[hb]);
  };
  f32x4_t acc[NH][4];
#pragma unroll
  for (int hb = 0; hb < NH; ++hb)
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[hb][u] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  auto consume = [&](int d) {
#pragma unroll
    for (int f = 0; f < 2; ++f) {
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        u32x4_t bop[4];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const auto p = __builtin_amdgcn_permlane16_swap(wr[d][2 * f + j][2 * v], wr[d][2 * f + j][2 * v + 1], false, false);
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const float sc = __builtin_bit_cast(float, __builtin_amdgcn_ubfe(sr[d][u], 16 * f + 8 * j, 8) << 23);
            const uint32_t c = p[u];
            bop[2 * j + u] = u32x4_t{cvt_fp4x2_bf16<0>(c, sc), cvt_fp4x2_bf16<1>(c, sc), cvt_fp4x2_bf16<2>(c, sc),
                                     cvt_fp4x2_bf16<3>(c, sc)};
          }
        }
#pragma unroll
        for (int hb = 0; hb < NH; ++hb)
#pragma unroll
          for (int u = 0; u < 4; ++u)
            acc[hb][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8_t, ar[d][hb][2 * f + v]), __builtin_bit_cast(bf16x8_t, bop[u]), acc[hb][u],
                0, 0, 0);
      }
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d) {
    load(d, min(d, KB - 1));
    __builtin_amdgcn_sched_barrier(0);  // the waits below count the loads in this order
  }
  int kb = 0;
  for (; kb + 2 * D <= KB; kb += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      consume(d);
      load(d, kb + D + d);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // The last KB - kb < 2 D blocks.
#pragma unroll
  for (int i = 0; i < 2 * D - 1; ++i) {
    if (kb + i < KB) {
      consume(i % D);
      if (i + D < 2 * D - 1 && kb + i + D < KB) load(i % D, kb + i + D);
    }
  }
  store_halves<NH, ACT, 72>(acc, ep_lds, row0, rows, col0, N, out, out_f32, bias, ep.bias_bf16, ep.act);
}

template <int WPB, bool ACT>
__global__ __launch_bounds__(64 * WPB) __attribute__((amdgpu_waves_per_eu(2))) void gmm_fp4_stream_kernel(
    const uint16_t *__restrict__ lhs, const int32_t *__restrict__ row_idx, int64_t lhs_rows, int64_t M, int K,
    const uint8_t *__restrict__ wpk, const uint8_t *__restrict__ spk, const int32_t *__restrict__ group_sizes,
    int num_groups, const int32_t *__restrict__ group_offset, int64_t e_local, int N, void *__restrict__ out,
    int out_f32, GmmEpilogue ep) {
  __shared__ __attribute__((aligned(16))) float s_ep[WPB][16 * 72];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = (N + 63) >> 6, n_ct = (G + WPB - 1) / WPB;
  const int go = group_offset ? group_offset[0] : 0;
  int g, rows, ct;
  int64_t row0;
  if (!find_stream_tile(group_sizes, num_groups, go, e_local, M, n_ct, g, row0, rows, ct)) return;
  const int cg = ct * WPB + wave;  // the wave's 64-column group
  if (cg >= G) return;
  const int64_t e = g - go;
  const uint8_t *const w = wpk + (e * G + cg) * (int64_t)(K >> 6) * 2048;
  const uint8_t *const s = spk + (e * G + cg) * (int64_t)(K >> 7) * 256;
  const void *const bias = expert_bias(ep, e, N);
  if (rows <= 16)
    stream_columns<1, 4, ACT>(lhs, row_idx, lhs_rows, row0, rows, K, w, s, (int64_t)cg * 64, N, out, out_f32, bias,
                              ep, s_ep[wave]);
  else
    stream_columns<2, 3, ACT>(lhs, row_idx, lhs_rows, row0, rows, K, w, s, (int64_t)cg * 64, N, out, out_f32, bias,
                              ep, s_ep[wave]);
}

// Grid of a streaming launch: four waves (256 columns) per block, or one
// where the waves are few, so that every CU gets a block.
struct StreamGrid {
  unsigned blocks;
  int wpb;
};

static int stream_grid(int64_t M, int64_t N, int64_t E_local, int num_groups, const char *what, StreamGrid &sg) {
  const int64_t G = (N + 63) / 64;
  // Row tiles: every group that holds rows has at most one partial one.
  const int64_t max_rt = M / kStreamRows + std::min(std::min(E_local, (int64_t)num_groups), M);
  sg.wpb = max_rt * G >= 4096 ? 4 : 1;
  const int64_t grid = (max_rt * ((G + sg.wpb - 1) / sg.wpb) + 7) / 8 * 8;
  DWM_UNSUPPORTED_IF(grid > (1ll << 31) - 1, "%s: too many tiles (%lld)", what, (long long)grid);
  sg.blocks = (unsigned)grid;
  return DWM_OK;
}

int launch_gmm_stream(const uint16_t *lhs, const int32_t *row_idx, int64_t lhs_rows, int64_t M, int64_t K,
                      const uint8_t *weight, const uint8_t *scale, const int32_t *group_sizes, int num_groups,
                      const int32_t *group_offset, int64_t E_local, int64_t N, void *out, int out_f32, bool gated,
                      const GmmEpilogue &ep, hipStream_t st) {
  StreamGrid sg;
  int rc = stream_grid(M, N, E_local, num_groups, "gmm_fp4", sg);
  if (rc != DWM_OK) return rc;
#define DWM_STREAM(WPB, ACT)                                                                                     \
  hipLaunchKernelGGL((gmm_fp4_stream_kernel<WPB, ACT>), dim3(sg.blocks), dim3(64 * WPB), 0, st, lhs,            \
                     row_idx, lhs_rows, M, (int)K, weight, scale, group_sizes, num_groups, group_offset, E_local, \
                     (int)N, out, out_f32, ep)
  if (gated) {
    if (sg.wpb == 4) DWM_STREAM(4, true);
    else DWM_STREAM(1, true);
  } else {
    if (sg.wpb == 4) DWM_STREAM(4, false);
    else DWM_STREAM(1, false);
  }
#undef DWM_STREAM
  return launch_status("gmm_fp4");
}

// The MX form: e4m3 (or, F4, e2m1) lhs codes with e8m0 block-32 row scales on
// the scaled 32x32x64 MFMA, which takes a lane's 16 weight bytes as they are.
// One wave: <= 32 rows x 64 columns, over K in the order of the MX tiles
// (gmm_mx.hip), so the results are theirs bit for bit.
typedef __attribute__((ext_vector_type(8))) int i32x8_t;

template <int D, bool ACT, bool F4>
__device__ __forceinline__ void mx_stream_columns(const uint8_t *__restrict__ lhs, const uint8_t *__restrict__ lsc,
                                                  const int32_t *__restrict__ row_idx, int64_t lhs_rows, int64_t row0,
                                                  int rows, int K, const uint8_t *__restrict__ w,
                                                  const uint8_t *__restrict__ s, int64_t col0, int N,
                                                  void *__restrict__ out, int out_f32, const void *bias,
                                                  const GmmEpilogue &ep, float *ep_lds) {
  constexpr int AB = F4 ? 64 : 128, AV = F4 ? 2 : 4;  // lhs bytes per row and K block; 16-byte loads per lane
  const int lane = threadIdx.x & 63, c32 = lane & 31, h = lane >> 5;
  const int KB = K >> 7;
  const int64_t r = row0 + min(c32, rows - 1);  // rows past the tile repeat its last row
  const int64_t src = row_idx ? gather_index(row_idx[r], lhs_rows) : r;
  const uint32_t aoff = (uint32_t)(src * (F4 ? K / 2 : K)) + 16u * h;
  const uint32_t asoff = (uint32_t)(src * (K / 32));
  const uint32_t woff = lane * 16u, soff = lane * 4u;
  u32x4_t wr[D][4], ar[D][AV];
  uint32_t sr[D], as[D];
  // lhs chunks of 64-deep half f: e4m3 4 f + h and 4 f + 2 + h, e2m1 2 f + h.
  auto load = [&](int d, int kb) {
    const uint8_t *const wb = w + (int64_t)kb * 4096;
#pragma unroll
    for (int i = 0; i < 4; ++i) wr[d][i] = __builtin_nontemporal_load((const u32x4_t *)(wb + 1024 * i + woff));
    sr[d] = *(const uint32_t *)(s + (int64_t)kb * 256 + soff);
    as[d] = *(const uint32_t *)(lsc + (int64_t)kb * 4 + asoff);
#pragma unroll
    for (int i = 0; i < AV; ++i) ar[d][i] = *(const u32x4_t *)(lhs + (int64_t)kb * AB + 32 * i + aoff);
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x16_t acc[1][2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[0][j][e] = 0.0f;
  auto consume = [&](int d) {
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      const u32x4_t lo = ar[d][F4 ? f : 2 * f], hi = ar[d][F4 ? 0 : 2 * f + 1];
      const i32x8_t a = F4 ? i32x8_t{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], 0, 0, 0, 0}
                           : i32x8_t{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3],
                                     (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
      const u32x4_t w0 = wr[d][2 * f], w1 = wr[d][2 * f + 1];
      const i32x8_t b0 = {(int)w0[0], (int)w0[1], (int)w0[2], (int)w0[3], 0, 0, 0, 0};
      const i32x8_t b1 = {(int)w1[0], (int)w1[1], (int)w1[2], (int)w1[3], 0, 0, 0, 0};
      const int sb = (int)(sr[d] >> (16 * f));
      const int sa = (int)((as[d] >> (16 * f + 8 * h)) & 0xFFu);
      constexpr int AFMT = F4 ? 4 : 0;  // A operand format: e2m1 or e4m3 (B: e2m1)
      acc[0][0] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b0, acc[0][0], AFMT, 4, 0, sa, 0, sb);
      acc[0][1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b1, acc[0][1], AFMT, 4, 0, sa, 1, sb);
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, min(d, KB - 1));
  int kb = 0;
  for (; kb + 2 * D <= KB; kb += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      consume(d);
      load(d, kb + D + d);
    }
  }
#pragma unroll
  for (int i = 0; i < 2 * D - 1; ++i) {
    if (kb + i < KB) {
      consume(i % D);
      if (i + D < 2 * D - 1 && kb + i + D < KB) load(i % D, kb + i + D);
    }
  }
  store_tile<1, ACT, 72>(acc, ep_lds, row0, rows, col0, N, out, out_f32, bias, ep.bias_bf16, ep.act);
}

template <int WPB, bool ACT, bool F4>
__global__ __launch_bounds__(64 * WPB) __attribute__((amdgpu_waves_per_eu(2))) void gmm_mx_stream_kernel(
    const uint8_t *__restrict__ lhs, const uint8_t *__restrict__ lsc, const int32_t *__restrict__ row_idx,
    int64_t lhs_rows, int64_t M, int K, const uint8_t *__restrict__ wpk, const uint8_t *__restrict__ spk,
    const int32_t *__restrict__ group_sizes, int num_groups, const int32_t *__restrict__ group_offset,
    int64_t e_local, int N, void *__restrict__ out, int out_f32, GmmEpilogue ep) {
  __shared__ __attribute__((aligned(16))) float s_ep[WPB][32 * 72];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = (N + 63) >> 6, n_ct = (G + WPB - 1) / WPB;
  const int go = group_offset ? group_offset[0] : 0;
  int g, rows, ct;
  int64_t row0;
  if (!find_stream_tile(group_sizes, num_groups, go, e_local, M, n_ct, g, row0, rows, ct)) return;
  const int cg = ct * WPB + wave;
  if (cg >= G) return;
  const int64_t e = g - go;
  const uint8_t *const w = wpk + (e * G + cg) * (int64_t)(K >> 6) * 2048;
  const uint8_t *const s = spk + (e * G + cg) * (int64_t)(K >> 7) * 256;
  mx_stream_columns<4, ACT, F4>(lhs, lsc, row_idx, lhs_rows, row0, rows, K, w, s, (int64_t)cg * 64, N, out, out_f32,
                                expert_bias(ep, e, N), ep, s_ep[wave]);
}

int launch_gmm_mx_stream(const uint8_t *lhs, const uint8_t *lhs_scale, const int32_t *row_idx, int64_t lhs_rows,
                         int64_t M, int64_t K, const uint8_t *weight, const uint8_t *scale,
                         const int32_t *group_sizes, int num_groups, const int32_t *group_offset, int64_t E_local,
                         int64_t N, void *out, int out_f32, bool gated, const GmmEpilogue &ep, hipStream_t st,
                         bool lhs_fp4) {
  StreamGrid sg;
  int rc = stream_grid(M, N, E_local, num_groups, "gmm_fp4_mx", sg);
  if (rc != DWM_OK) return rc;
#define DWM_STREAM(WPB, ACT, F4)                                                                                    \
  hipLaunchKernelGGL((gmm_mx_stream_kernel<WPB, ACT, F4>), dim3(sg.blocks), dim3(64 * WPB), 0, st, lhs, lhs_scale, \
                     row_idx, lhs_rows, M, (int)K, weight, scale, group_sizes, num_groups, group_offset, E_local,   \
                     (int)N, out, out_f32, ep)
#define DWM_STREAM_W(ACT, F4) \
  do {                        \
    if (sg.wpb == 4) DWM_STREAM(4, ACT, F4); \
    else DWM_STREAM(1, ACT, F4);             \
  } while (0)
  if (lhs_fp4) {
    if (gated) DWM_STREAM_W(true, true);
    else DWM_STREAM_W(false, true);
  } else {
    if (gated) DWM_STREAM_W(true, false);
    else DWM_STREAM_W(false, false);
  }
#undef DWM_STREAM_W
#undef DWM_STREAM
  return launch_status("gmm_fp4_mx");
}

}  // namespace dwm

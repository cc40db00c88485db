// Ragged grouped matmul for few rows per expert (decode batches): the same
// product, layouts and results as gmm_fp4.hip, built for streaming weights.
//
// What bounds it: HBM (6.6 TB/s reached at 198 rows over 256 experts, K = N =
// 4096: 188 us, the tiles 256; one token over 32 experts 49 -> 23).  Up to 32
// rows of an expert a weight byte (two codes) feeds at most 128 FLOPs, so the
// packed weights' stream sets the time.
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

// The wave's tile: `rows` rows from row0 of group g, 64-column group cg;
// stream: its weights are loaded with the streaming policy.
struct StreamRef {
  int64_t row0;
  int g, rows, cg;
  bool stream;
};

// A block's first w waves take w adjacent 64-column groups of one row tile.
// The list runs (group, column tile, row tile) with the row tile innermost,
// so that the row tiles of one column tile run side by side on one XCD and
// share its L2's copy of the weights; it is cut into 8 contiguous runs, one
// per XCD (blocks whose index is equal mod 8).  Every wave finds its tile
// alone: lane l holds the sizes of groups l PL .. + PL - 1, and prefix sums
// over the lanes give row starts and row-tile counts.  Returns false when
// the wave has no tile.
//
// Group sizes are not checked by the host: negative ones count as empty, and
// sizes that sum past M are cut to the rows left below M before their tiles
// are counted, so the list holds the tiles of rows [0, M) and no others, and
// fits the grid (stream_grid) whatever the sizes sum to.
//
// Row tiles hold 16 rows (MX: 32, its MFMA's) or 32.  With 16 the waves are
// alike: while weights stream from HBM, a wave with twice the rows falls
// behind and ends alone.  32 are taken in launches of at most half a round of
// waves (64 Zipf rows over 8 experts, K = 3072, N = 4096 14.3 -> 12.8 us), where
// most tiles would share their weights with another one anyway (few groups
// hold all rows: larger tiles read less from L2), where only they fit one
// round, and where 16 would not fit the grid.  Against 32 throughout, us: 384 rows over 64
// experts by a Zipf law (1.1), K = N = 4096 100.5 -> 90.5; 192 such rows over
// 32 experts, K = 2048, N = 7168 50.5 -> 44.0; 32 of 64 rows in one of 32
// experts, K = 7168 101.5 -> 86.2 (but 20 of 40 rows there 55.4 -> 61.2, the
// tiles of gmm_fp4.hip 65.8).  Against 16 throughout: 1536 rows in one
// of 256 experts 121 -> 109; 192 Zipf rows over 32 experts, K = 7168 94 -> 88.
//
// Blocks of four waves share their lhs rows through L1.  A launch of at most
// one round takes one or two waves a block where that leaves fewer waves on
// the fullest CU (128 rows in 4 of 64 experts, K = N = 4096 37.6 -> 15.5).
template <int PL, bool R16, int WPB>
__device__ __forceinline__ bool stream_tile(const int32_t *__restrict__ group_sizes, int num_groups, int go,
                                            int64_t e_local, int64_t M, int G, int max_rt, int ncu, int wave,
                                            StreamRef &ref) {
  const int lane = threadIdx.x & 63;
  const int m32 = (int)min(M, (int64_t)0x7FFFFFFF);
  int sz[PL];
#pragma unroll
  for (int i = 0; i < PL; ++i) sz[i] = group_sizes[min(lane * PL + i, num_groups - 1)];  // loads side by side
  auto tiles_of = [&](int gi, int s, int lg) {
    return gi >= go && (int64_t)gi < (int64_t)go + e_local ? (s >> lg) + ((s & ((1 << lg) - 1)) != 0 ? 1 : 0) : 0;
  };
  int rows_in = 0, v[2] = {0, 0};  // row tiles of 32 rows, of 16
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    sz[i] = lane * PL + i < num_groups ? min(max(sz[i], 0), m32) : 0;
    rows_in += sz[i];
  }
  const int start = wave_inclusive_scan(rows_in) - rows_in;  // first row of the lane's first group
  int left = start >= 0 ? max(m32 - start, 0) : 0;           // (a sum past int32 is past M too)
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    sz[i] = min(sz[i], left);
    left -= sz[i];
    v[0] += tiles_of(lane * PL + i, sz[i], 5);
    if (R16) v[1] += tiles_of(lane * PL + i, sz[i], 4);
  }
  const int own[2] = {v[0], v[1]};
  wave_inclusive_scan_n<2>(v);
  const int64_t cap = 8 * (int64_t)ncu;  // waves of one round: 256 VGPRs each
  const int all32 = wave_last(v[0]), all16 = R16 ? wave_last(v[1]) : 0;
  const bool small = R16 && all16 <= max_rt && 2 * (int64_t)all16 < 3 * (int64_t)all32 &&
                     2 * all32 * (int64_t)G > cap && (all16 * (int64_t)G <= cap || all32 * (int64_t)G > cap);
  const int lg = small ? 4 : 5, all = small ? all16 : all32;
  const int upto = small ? v[1] : v[0], before = upto - (small ? own[1] : own[0]);
  const int j = blockIdx.x >> 3;
  if (j >= (all * (int64_t)G + 7) >> 3) return false;  // past the run of every w
  int w = WPB;
  if (WPB == 4 && all * (int64_t)G <= cap) {
    // Waves on the fullest CU with k a block; the list has to fit the grid.
    auto fullest = [&](int k) {
      const int blocks = all * ((G + k - 1) / k);
      return blocks <= (int)gridDim.x ? (blocks + ncu - 1) / ncu * k : 1 << 30;
    };
    if (fullest(2) < fullest(w)) w = 2;
    if (fullest(1) < fullest(w)) w = 1;
  }
  const int n_ct = w == 1 ? G : w == 2 ? (G + 1) >> 1 : (G + 3) >> 2;
  const int64_t total = (int64_t)all * n_ct;
  const int64_t run = (total + 7) >> 3;
  const int64_t entry = (int64_t)(blockIdx.x & 7) * run + j;
  if (wave >= w || j >= run || entry >= total || entry > 0x7FFFFFFFll) return false;
  const int trow = (int)((uint32_t)entry / (uint32_t)n_ct);
  const uint64_t hit = __ballot(before <= trow && trow < upto);
  if (!hit) return false;
  const int sel = __ffsll((unsigned long long)hit) - 1;
  int rs = __builtin_amdgcn_readlane(start, sel);  // first row of lane sel's first group
  int tc = __builtin_amdgcn_readlane(before, sel);         // row tiles before it
  int g = -1, szg = 0;
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    if (g < 0) {
      const int s = __builtin_amdgcn_readlane(sz[i], sel);
      const int n = tiles_of(sel * PL + i, s, lg);
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
  const uint32_t n = (uint32_t)tiles_of(g, szg, lg), local = (uint32_t)entry - (uint32_t)tc * (uint32_t)n_ct;
  const int rt = (int)(local % n);
  ref.g = g;
  ref.cg = (int)(local / n) * w + wave;
  ref.row0 = (int64_t)rs + ((int64_t)rt << lg);
  ref.rows = min(szg - (rt << lg), 1 << lg);
  ref.stream = n == 1 || all * (int64_t)G <= cap;
  return ref.cg < G;
}

template <bool R16, int WPB>
__device__ __forceinline__ bool find_stream_tile(const int32_t *__restrict__ group_sizes, int num_groups, int go,
                                                 int64_t e_local, int64_t M, int G, int max_rt, int ncu, int wave,
                                                 StreamRef &ref) {
  if (num_groups <= 64) return stream_tile<1, R16, WPB>(group_sizes, num_groups, go, e_local, M, G, max_rt, ncu, wave, ref);
  if (num_groups <= 256) return stream_tile<4, R16, WPB>(group_sizes, num_groups, go, e_local, M, G, max_rt, ncu, wave, ref);
  return stream_tile<kMaxGroups / 64, R16, WPB>(group_sizes, num_groups, go, e_local, M, G, max_rt, ncu, wave, ref);
}

// NT: the weights stream past the caches.  Not where other row tiles of the
// group read them in a later round of waves (plain loads, K = N = 4096: half
// of 1536 rows in one of 256 experts 512 -> 467 us, 384 Zipf rows over 64
// experts 107 -> 100); within one round the tiles run side by side and share
// them anyway, and plain loads lose (64 rows in one of 8 experts, K = 1024, N
// = 2048 6.3 -> 7.1).
template <bool NT>
__device__ __forceinline__ u32x4_t load_weights(const u32x4_t *p) {
  return NT ? __builtin_nontemporal_load(p) : *p;
}

// One row tile of NH 16-row blocks x the wave's 64 columns.
template <int NH, int D, bool NT, bool ACT>
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
    for (int i = 0; i < 4; ++i) wr[d][i] = load_weights<NT>((const u32x4_t *)(wb + 1024 * i + woff));
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

template <int WPB, bool R16, bool ACT>
__global__ __launch_bounds__(64 * WPB) __attribute__((amdgpu_waves_per_eu(2))) void gmm_fp4_stream_kernel(
    const uint16_t *__restrict__ lhs, const int32_t *__restrict__ row_idx, int64_t lhs_rows, int64_t M, int K,
    const uint8_t *__restrict__ wpk, const uint8_t *__restrict__ spk, const int32_t *__restrict__ group_sizes,
    int num_groups, const int32_t *__restrict__ group_offset, int64_t e_local, int N, void *__restrict__ out,
    int out_f32, GmmEpilogue ep, int max_rt, int ncu) {
  __shared__ __attribute__((aligned(16))) float s_ep[WPB][16 * 72];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = (N + 63) >> 6;
  const int go = group_offset ? group_offset[0] : 0;
  StreamRef ref;
  if (!find_stream_tile<R16, WPB>(group_sizes, num_groups, go, e_local, M, G, max_rt, ncu, wave, ref)) return;
  const int rows = ref.rows, cg = ref.cg;
  const int64_t e = ref.g - go;
  const uint8_t *const w = wpk + (e * G + cg) * (int64_t)(K >> 6) * 2048;
  const uint8_t *const s = spk + (e * G + cg) * (int64_t)(K >> 7) * 256;
  const void *const bias = expert_bias(ep, e, N);
#define DWM_COLUMNS(NH, D, NT)                                                                              \
  stream_columns<NH, D, NT, ACT>(lhs, row_idx, lhs_rows, ref.row0, rows, K, w, s, (int64_t)cg * 64, N, out, \
                                 out_f32, bias, ep, s_ep[wave])
  if (rows <= 16) {
    if (!R16 || ref.stream) DWM_COLUMNS(1, 4, true);
    else DWM_COLUMNS(1, 4, false);
  } else {
    if (!R16 || ref.stream) DWM_COLUMNS(2, 3, true);
    else DWM_COLUMNS(2, 3, false);
  }
#undef DWM_COLUMNS
}

// Grid of a streaming launch: four waves (256 columns) per block, or one
// where the waves are few, so that every CU gets a block.
struct StreamGrid {
  unsigned blocks;
  int wpb, max_rt;
};

static int stream_grid(int64_t M, int64_t N, int64_t E_local, int num_groups, const char *what, StreamGrid &sg) {
  const int64_t G = (N + 63) / 64;
  // Row tiles of 32 rows: every group that holds rows has at most one partial one.
  const int64_t max_rt = M / 32 + std::min(std::min(E_local, (int64_t)num_groups), M);
  sg.wpb = max_rt * G >= 4096 ? 4 : 1;
  const int64_t grid = (max_rt * ((G + sg.wpb - 1) / sg.wpb) + 7) / 8 * 8;
  DWM_UNSUPPORTED_IF(grid > (1ll << 31) - 1, "%s: too many tiles (%lld)", what, (long long)grid);
  sg.blocks = (unsigned)grid;
  sg.max_rt = (int)max_rt;
  return DWM_OK;
}

int launch_gmm_stream(const uint16_t *lhs, const int32_t *row_idx, int64_t lhs_rows, int64_t M, int64_t K,
                      const uint8_t *weight, const uint8_t *scale, const int32_t *group_sizes, int num_groups,
                      const int32_t *group_offset, int64_t E_local, int64_t N, void *out, int out_f32, bool gated,
                      const GmmEpilogue &ep, hipStream_t st) {
  StreamGrid sg;
  int rc = stream_grid(M, N, E_local, num_groups, "gmm_fp4", sg);
  if (rc != DWM_OK) return rc;
#define DWM_STREAM(WPB, R16, ACT)                                                                                \
  hipLaunchKernelGGL((gmm_fp4_stream_kernel<WPB, R16, ACT>), dim3(sg.blocks), dim3(64 * WPB), 0, st, lhs,       \
                     row_idx, lhs_rows, M, (int)K, weight, scale, group_sizes, num_groups, group_offset, E_local, \
                     (int)N, out, out_f32, ep, sg.max_rt, ncu)
  // 16-row tiles are taken (stream_tile) past half a round of waves, and make
  // a difference with a group of more than 16 rows: a launch too small for
  // both runs the kernel without that choice (0.2 us less search: 8 rows, K =
  // 2048, N = 7168 12.3 -> 12.0).
  const int ncu = device_cu_count();
  const int64_t half = 4 * (int64_t)ncu / ((N + 63) / 64);  // row tiles in half a round
  const bool r16 = sg.max_rt > half && M > 16 + half;
  if (gated) {
    if (sg.wpb == 4) DWM_STREAM(4, true, true);
    else if (r16) DWM_STREAM(1, true, true);
    else DWM_STREAM(1, false, true);
  } else {
    if (sg.wpb == 4) DWM_STREAM(4, true, false);
    else if (r16) DWM_STREAM(1, true, false);
    else DWM_STREAM(1, false, false);
  }
#undef DWM_STREAM
  note_kernel("gmm_stream");
  return launch_status("gmm_fp4");
}

// The MX form: e4m3 (or, F4, e2m1) lhs codes with e8m0 block-32 row scales on
// the scaled 32x32x64 MFMA, which takes a lane's 16 weight bytes as they are.
// One wave: <= 32 rows x 64 columns, over K in the order of the MX tiles
// (gmm_mx.hip), so the results are theirs bit for bit.
typedef __attribute__((ext_vector_type(8))) int i32x8_t;

template <int D, bool NT, bool ACT, bool F4>
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
    for (int i = 0; i < 4; ++i) wr[d][i] = load_weights<NT>((const u32x4_t *)(wb + 1024 * i + woff));
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
    int64_t e_local, int N, void *__restrict__ out, int out_f32, GmmEpilogue ep, int max_rt, int ncu) {
  __shared__ __attribute__((aligned(16))) float s_ep[WPB][32 * 72];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = (N + 63) >> 6;
  const int go = group_offset ? group_offset[0] : 0;
  StreamRef ref;
  if (!find_stream_tile<false, WPB>(group_sizes, num_groups, go, e_local, M, G, max_rt, ncu, wave, ref)) return;
  const int rows = ref.rows, cg = ref.cg;
  const int64_t e = ref.g - go;
  const uint8_t *const w = wpk + (e * G + cg) * (int64_t)(K >> 6) * 2048;
  const uint8_t *const s = spk + (e * G + cg) * (int64_t)(K >> 7) * 256;
#define DWM_COLUMNS(NT)                                                                                          \
  mx_stream_columns<4, NT, ACT, F4>(lhs, lsc, row_idx, lhs_rows, ref.row0, rows, K, w, s, (int64_t)cg * 64, N, \
                                    out, out_f32, expert_bias(ep, e, N), ep, s_ep[wave])
  if (ref.stream) DWM_COLUMNS(true);
  else DWM_COLUMNS(false);
#undef DWM_COLUMNS
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
                     (int)N, out, out_f32, ep, sg.max_rt, device_cu_count())
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
  note_kernel("gmm_mx_stream");
  return launch_status("gmm_fp4_mx");
}

}  // namespace dwm

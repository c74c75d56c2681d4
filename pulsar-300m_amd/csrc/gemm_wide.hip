// Row-set GEMMs for hundreds to tens of thousands of rows (prefill, the output head of large
// steps, draft blocks at large batches), bf16: C[rows, N] = epi(A[rows, K] . W[N, K]^T) in
// tiles staged through LDS.
#include <algorithm>

#include "gemm_common.h"

namespace pulsar {

namespace {

// A workgroup of WR x WC waves owns a tile of 16 RT WR rows x 16 CT WC output columns (SwiGLU:
// half of them gate columns, half their up-projection twins); wave (wr, wc) computes RT x CT
// MFMA tiles. Per 32-wide k step the workgroup stages the A tile (gathered rows in MFMA lane
// order) and the weight tiles (1 KB each, stored in lane order) in LDS with direct
// global-to-LDS loads (16 bytes per lane, no staging registers): a wave's load instruction
// fills one 1 KB tile, lane l at +16 l, which is the lane's own MFMA operand. A ring of S
// buffers keeps S - 1 k steps in flight while one is computed; one barrier per step both
// publishes the step's tiles to all waves and frees the buffer the next load overwrites. The
// weights go in as the A operand and the rows as B, so a lane ends with 4 consecutive output
// columns of its own row: 8-byte epilogue loads and stores, and the C row is an entry the
// lane loads itself.
//
// Every shape sums an output's K in one chain of 32-wide products in k order, so the shapes
// give identical results and a launch picks one by speed alone (wide_shape).
template <int RT_, int CT_, int WR_, int WC_, int S_, int WPS_>
struct WideShape {
  static constexpr int RT = RT_, CT = CT_, WR = WR_, WC = WC_, S = S_, WPS = WPS_;
  static constexpr int kWaves = WR * WC, kThreads = 64 * kWaves;
  static constexpr int kRowTiles = RT * WR, kColTiles = CT * WC;  // 16-row / 16-column tiles
  static constexpr int kRows = 16 * kRowTiles, kCols = 16 * kColTiles;
  static constexpr int LA = kRowTiles / kWaves, LW = kColTiles / kWaves;  // loads per wave, step
  static_assert(kRowTiles % kWaves == 0 && kColTiles % kWaves == 0, "whole loads per wave");
  static_assert((S - 2) * (LA + LW) <= 63, "vmcnt range");
};
using WideLarge = WideShape<4, 8, 2, 2, 3, 2>;  // 128 x 256
using WideMid = WideShape<4, 4, 2, 2, 4, 2>;    // 128 x 128
using WideLow = WideShape<2, 4, 2, 2, 5, 2>;    // 64 x 128
using WideSmall = WideShape<2, 2, 2, 2, 8, 2>;  // 64 x 64

// Row-set launches are 1-D grids. The tiles that hold rows, in the order (group, row tile,
// column block) with column blocks fastest, are cut into 8 equal contiguous ranges, one per
// XCD (workgroup L runs on XCD L % 8, as slot L / 8 of its range). The column blocks of a row
// tile then follow one another on one XCD, which fetches the tile's rows into its L2 once for
// all of them, and a group's weights are read by the one or two XCDs whose ranges hold its
// tiles. Row counts are read on the device, so every XCD gets an equal share of the tiles
// that exist; workgroups past the end exit. rows_fast (one group with fewer rows than weight
// columns): row tiles fastest, so that each XCD fetches its own part of the weights and the
// rows, the smaller operand, are what every XCD fetches (517 rows: wo 11.5 -> 10.6 us).
template <int MODE, int ROWS>
__device__ __forceinline__ bool wide_tile(const GemmArgs& g, int& bx, int& group, int& bz) {
  const int L = (int)blockIdx.x, xcd = L % kXcds, slot = L / kXcds;
  const int lane = (int)threadIdx.x & 63;
  // row tiles of each group, 64 groups per pass (one per lane)
  int total = 0;
  for (int y0 = 0; y0 < g.grid_y; y0 += 64) {
    const int y = y0 + lane;
    const int nt = y < g.grid_y
        ? min((group_rows<MODE>(g, y + g.group_offset) + ROWS - 1) / ROWS, g.grid_z)
        : 0;
    for (int j = 0; j < 64 && y0 + j < g.grid_y; ++j) total += __builtin_amdgcn_readlane(nt, j);
  }
  total *= g.grid_x;
  const int per = (total + kXcds - 1) / kXcds;
  int item = xcd * per + slot;
  if (slot >= per || item >= total) return false;
  if (g.rows_fast) {  // one group
    const int nt = total / g.grid_x;
    bx = item / nt;
    bz = item % nt;
    group = g.group_offset;
    return true;
  }
  bx = item % g.grid_x;
  int t = item / g.grid_x;
  for (int y0 = 0; y0 < g.grid_y; y0 += 64) {
    const int y = y0 + lane;
    const int nt = y < g.grid_y
        ? min((group_rows<MODE>(g, y + g.group_offset) + ROWS - 1) / ROWS, g.grid_z)
        : 0;
    for (int j = 0; j < 64 && y0 + j < g.grid_y; ++j) {
      const int ntj = __builtin_amdgcn_readlane(nt, j);
      if (t < ntj) {
        group = y0 + j + g.group_offset;
        bz = t;
        return true;
      }
      t -= ntj;
    }
  }
  return false;
}

template <int EPI, int MODE, typename SH>
__global__ void __launch_bounds__(SH::kThreads, SH::WPS) gemm_bf16_lds_kernel(GemmArgs g) {
  constexpr bool kPair = (EPI == EPI_SWIGLU);
  constexpr int S = SH::S, RT = SH::RT, CT = SH::CT, NW = SH::kWaves, LA = SH::LA, LW = SH::LW;
  constexpr int NR = SH::kRowTiles, NC = SH::kColTiles;
  __shared__ bf16x8_t sA[S][NR][64];  // [buffer][row tile][lane]
  __shared__ bf16x8_t sW[S][NC][64];  // [buffer][column tile][lane]
  int bx = (int)blockIdx.x, group = (int)blockIdx.y + g.group_offset, bz = (int)blockIdx.z;
  if constexpr (MODE != ROWS_LOGITS) {
    if (!wide_tile<MODE, SH::kRows>(g, bx, group, bz)) return;
  }
  const int N = g.N;
  const int KT = g.K / 32;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int wr = wv / SH::WC, wc = wv % SH::WC;
  const int m16 = lane & 15, kq = lane >> 4;
  const int cnt = group_rows<MODE>(g, group);
  if constexpr (MODE == ROWS_LOGITS) {
    // output head (one group): workgroup L runs on XCD L % 8; give each XCD a contiguous
    // range of column tiles with their row tiles one after another, so the row tiles of a
    // column tile read its weights through one L2
    const int nz = (int)gridDim.z, total = (int)gridDim.x * nz;
    if (nz > 1 && total % 8 == 0) {
      const int L = bx + (int)gridDim.x * bz;
      const int w = (L & 7) * (total >> 3) + (L >> 3);
      bx = w / nz;
      bz = w % nz;
    }
  }
  const int r_wg = bz * SH::kRows;
  if (r_wg >= cnt) return;
  const int ct_wg = bx * (kPair ? NC / 2 : NC);  // first (gate) column tile
  if (ct_wg * 16 >= N) return;
  const bf16* A = reinterpret_cast<const bf16*>(g.A);
  const bf16* W = reinterpret_cast<const bf16*>(g.W) + (int64_t)group * g.w_group_stride;

  // staging: wave wv fills row tiles wv + NW h (h < LA) and weight tiles wv + NW h (h < LW).
  // A row tile's 64 16-byte chunks sit in LDS as (row m, k chunk q) at slot
  // 4 m + (q ^ (m >> 2 & 3)): the load's lane l carries row 16 t + (l >> 2), so 16 lanes
  // fetch the 64 contiguous bytes of 4 rows, and the XOR puts the 16 rows of one k chunk
  // that a fragment read takes on 16 different 16-byte bank groups
  const bf16* ga[LA];
#pragma unroll
  for (int h = 0; h < LA; ++h) {
    const int r = (wv + NW * h) * 16 + (lane >> 2);
    const int i = min(r_wg + r, cnt - 1);
    const int e = entry_load<MODE>(g, group, i);
    ga[h] = A + (int64_t)a_row_of<MODE>(g, group, e) * g.lda + ((lane & 3) ^ (lane >> 4 & 3)) * 8;
  }
  const int aslot = m16 * 4 + (kq ^ (m16 >> 2 & 3));  // this lane's fragment chunk
  const bf16* gw[LW];
#pragma unroll
  for (int h = 0; h < LW; ++h) {
    const int c = wv + NW * h;
    int ct;
    if constexpr (kPair)
      ct = c < NC / 2 ? ct_wg + c : N / 16 + ct_wg + (c - NC / 2);
    else
      ct = min(ct_wg + c, N / 16 - 1);  // tiles past N re-read the last one (never stored)
    gw[h] = W + ((int64_t)ct * KT * 64 + lane) * 8;
  }
  // k step kt into ring buffer b: LA + LW loads per wave, counted by vmcnt
  auto fetch = [&](int kt, int b) {
#pragma unroll
    for (int h = 0; h < LW; ++h) load_lds16(gw[h] + (int64_t)kt * 512, &sW[b][wv + NW * h][0]);
#pragma unroll
    for (int h = 0; h < LA; ++h) load_lds16(ga[h] + kt * 32, &sA[b][wv + NW * h][0]);
  };
  // this wave's column tiles in the staged set (SwiGLU: half gate, half their up twins)
  int wcol[CT];
#pragma unroll
  for (int j = 0; j < CT; ++j)
    wcol[j] = kPair ? (j < CT / 2 ? wc * (CT / 2) + j : NC / 2 + wc * (CT / 2) + (j - CT / 2))
                    : wc * CT + j;

  f32x4_t acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // The fragments of step kt + 1 are read from LDS while step kt's products run (one
  // workgroup on a CU has nothing else to overlap them with).
  bf16x8_t fa[2][RT], fw[2][CT];
  auto read = [&](int b, bf16x8_t (&xa)[RT], bf16x8_t (&xw)[CT]) {
#pragma unroll
    for (int i = 0; i < RT; ++i) xa[i] = sA[b][wr * RT + i][aslot];
#pragma unroll
    for (int j = 0; j < CT; ++j) xw[j] = sW[b][wcol[j]][lane];
  };
#pragma unroll
  for (int k = 0; k < S; ++k)
    if (k < KT) fetch(k, k);
  if (KT >= S)
    wait_vmcnt<(LA + LW) * (S - 1)>();
  else
    wait_vmcnt<0>();
  lds_barrier();
  read(0, fa[0], fw[0]);
  int buf = 0;  // ring buffer of step kt
  auto step = [&](int kt, bf16x8_t (&xa)[RT], bf16x8_t (&xw)[CT], bf16x8_t (&na)[RT],
                  bf16x8_t (&nw)[CT]) {
    const int next = buf == S - 1 ? 0 : buf + 1;
    if (kt + 1 < KT) {
      // this wave's loads of step kt + 1 are done once at most the S - 2 younger steps' loads
      // are outstanding (all of them near the end); the barrier then makes every wave's tiles
      // of step kt + 1 visible, and every wave's reads of step kt are in, so that the next
      // fetch may fill its buffer
      if (kt + S - 1 < KT)
        wait_vmcnt<(LA + LW) * (S - 2)>();
      else
        wait_vmcnt<0>();
      lds_barrier();
      if (kt + S < KT) fetch(kt + S, buf);
      read(next, na, nw);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xw[j], xa[i], acc[i][j], 0, 0, 0);
    buf = next;
  };
  // K is a multiple of 256: an even number of steps
  for (int kt = 0; kt < KT; kt += 2) {
    step(kt, fa[0], fw[0], fa[1], fw[1]);
    step(kt + 1, fa[1], fw[1], fa[0], fw[0]);
  }
  // lane holds columns 4 kq + e of column tile wcol[j] for row m16 of row tile wr * RT + i. The
  // row entries and what the epilogue reads (residual rows, column scales) are loaded before
  // the first store: loads and stores may alias as far as the compiler knows, and one load,
  // wait and store after another was 32 round trips at the end of every workgroup.
  constexpr int NJ = kPair ? CT / 2 : CT;
  int crow[RT], col[NJ];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int r = min(r_wg + wr * RT * 16 + i * 16 + m16, cnt - 1);
    crow[i] = entry_fix<MODE>(group, r, entry_load<MODE>(g, group, r)) + g.c_row_offset;
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) col[j] = (ct_wg + wcol[j]) * 16 + kq * 4;
  bf16x4_t pre[EPI == EPI_RESID ? RT : 1][NJ];
  if constexpr (EPI == EPI_RESID) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        pre[i][j] = *reinterpret_cast<const bf16x4_t*>(reinterpret_cast<const bf16*>(g.C) +
                                                       (int64_t)crow[i] * g.ldc + min(col[j], N - 4));
  }
  if constexpr (EPI == EPI_SCALE) {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      pre[0][j] = *reinterpret_cast<const bf16x4_t*>(reinterpret_cast<const bf16*>(g.bias) +
                                                     min(col[j], N - 4));
  }
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    if (r_wg + wr * RT * 16 + i * 16 + m16 >= cnt) continue;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if (col[j] >= N) continue;
      float v[4], u[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = acc[i][j][e];
        u[e] = kPair ? acc[i][j + CT / 2][e] : 0.f;
      }
      epilogue4(g, EPI, group, g.C, g.ldc, crow[i], col[j], v, u,
                pre[EPI == EPI_RESID ? i : 0][j]);
    }
  }
}

template <int EPI, int MODE, typename SH>
int launch_shape(const GemmArgs& a, int groups, int max_rows, hipStream_t s) {
  const int colw = EPI == EPI_SWIGLU ? SH::kCols / 2 : SH::kCols;
  GemmArgs ga = a;
  ga.grid_x = (a.N + colw - 1) / colw;
  ga.grid_y = groups;
  ga.grid_z = (max_rows + SH::kRows - 1) / SH::kRows;
  ga.rows_fast = groups == 1 && max_rows < (EPI == EPI_SWIGLU ? 2 : 1) * a.N;
  const int64_t tiles = (int64_t)ga.grid_x * ga.grid_y * ga.grid_z;
  if (tiles > (int64_t)1 << 30) return fail(PULSAR_ERR_INVALID, "gemm: wide launch too large");
  // row-set modes: a 1-D grid over (column block, group, row tile), split by wide_tile
  const dim3 grid = MODE == ROWS_LOGITS
      ? dim3((unsigned)ga.grid_x, (unsigned)ga.grid_y, (unsigned)ga.grid_z)
      : dim3((unsigned)((tiles + kXcds - 1) / kXcds * kXcds));
  gemm_bf16_lds_kernel<EPI, MODE, SH><<<grid, SH::kThreads, 0, s>>>(ga);
  PULSAR_LAUNCH_CHECK();
  return PULSAR_OK;
}

// The smallest shape whose tiles are at most two per CU, the large one when none is (128 x 128
// only below two per CU: at exactly two, the last line's 512 rows, the large tile wins). A CU that
// holds one workgroup streams its operands at 30-50 bytes/ns (outstanding misses), so a launch
// of few tiles is as slow as one tile's bytes: 128 x 256 x 1024 takes 27 us however few rows
// there are, 64 x 64 10 us. With every CU busy twice over the larger tile's fewer bytes per
// product win. us per launch in 64 x 64 / 64 x 128 / 128 x 128 / 128 x 256 tiles:
//   qkv + gate   517 rows 11.0 / 13.4 / 18.2 / 27.8   1400  20.2 / 15.3 / 19.1 / 29.7
//                2048     22.7 / 18.1 / 19.7 / 28.6   4000  38.0 / 30.4 / 25.9 / 30.3
//   wo           1400     12.8 / 14.0 / 18.9 / 28.6   4000  24.6 / 18.8 / 20.4 / 29.6
//   routed gate/up (rows each of 16 experts) 129      24.1 / 19.5 / 19.7 / 28.0
//                350      39.0 / 32.7 / 26.8 / 29.8   512   50.8 / 39.3 / 39.9 / 35.3
// The decode output head (32768 columns) goes by the same rule: 128 rows, exactly two 64 x 128
// tiles per CU, take 29 us in them and 46 in 128 x 256; more rows take the large tile.
constexpr int64_t kWideTiles = 512;
template <int EPI, int MODE>
int launch_wide(const GemmArgs& a, int groups, int max_rows, hipStream_t s) {
  if (max_rows <= 0) return PULSAR_OK;
  const int rows = a.rows_avg > 0 ? std::min(a.rows_avg, max_rows) : max_rows;
  const int64_t cols = (int64_t)a.N * (EPI == EPI_SWIGLU ? 2 : 1);
  auto tiles = [&](int r, int c) { return (int64_t)groups * ((rows + r - 1) / r) * ((cols + c - 1) / c); };
  if (tiles(64, 64) <= kWideTiles) return launch_shape<EPI, MODE, WideSmall>(a, groups, max_rows, s);
  if (tiles(64, 128) <= kWideTiles) return launch_shape<EPI, MODE, WideLow>(a, groups, max_rows, s);
  if (tiles(128, 128) < kWideTiles) return launch_shape<EPI, MODE, WideMid>(a, groups, max_rows, s);
  return launch_shape<EPI, MODE, WideLarge>(a, groups, max_rows, s);
}

}  // namespace

int launch_gemm_wide(const GemmArgs& a, int dtype, int epi, int groups, int max_rows,
                     hipStream_t s) {
  if (a.has_g0) return launch_gemm(a, dtype, epi, groups, max_rows, s);
  if (dtype != PULSAR_BF16) return launch_gemm_f32(a, epi, groups, max_rows, true, s);
  if (groups <= 0) return PULSAR_OK;
  if (a.K % 256 != 0 || a.N % 16 != 0 || (epi == EPI_SWIGLU && a.N % 128 != 0))
    return fail(PULSAR_ERR_UNSUPPORTED, "gemm: wide tiles need K % 256 == 0 and N % 16 == 0 "
                                        "(SwiGLU: N % 128 == 0)");
  // the row sets each epilogue serves in the engine
  const int m = a.row_mode;
  if (epi == EPI_QKVG && m == ROWS_PULSE)
    return launch_wide<EPI_QKVG, ROWS_PULSE>(a, groups, max_rows, s);
  if (epi == EPI_RESID && m == ROWS_PULSE)
    return launch_wide<EPI_RESID, ROWS_PULSE>(a, groups, max_rows, s);
  if (epi == EPI_SWIGLU && m == ROWS_ALL)
    return launch_wide<EPI_SWIGLU, ROWS_ALL>(a, groups, max_rows, s);
  if (epi == EPI_SWIGLU && m == ROWS_LIST)
    return launch_wide<EPI_SWIGLU, ROWS_LIST>(a, groups, max_rows, s);
  if (epi == EPI_STORE && m == ROWS_ALL)
    return launch_wide<EPI_STORE, ROWS_ALL>(a, groups, max_rows, s);
  if (epi == EPI_STORE && m == ROWS_LIST)
    return launch_wide<EPI_STORE, ROWS_LIST>(a, groups, max_rows, s);
  if (epi == EPI_SCALE && m == ROWS_LIST)
    return launch_wide<EPI_SCALE, ROWS_LIST>(a, groups, max_rows, s);
  if (epi == EPI_LOGITS && m == ROWS_LOGITS)
    return launch_wide<EPI_LOGITS, ROWS_LOGITS>(a, groups, max_rows, s);
  return fail(PULSAR_ERR_INVALID, "gemm: row mode of a wide launch");
}

}  // namespace pulsar

// Row-set GEMMs for decode and prefill: C[rows, N] = epi(A[rows, K] . W[N, K]^T), bf16
// weights stored in matrix-core tile order [N/16][K/32][64 lanes][8].
//
// Decode (gemm_bf16_kernel): a workgroup of 8 waves owns 16 output columns and walks the
// group's 32-row tiles; the waves split K, each runs v_mfma_f32_16x16x32_bf16 on two
// 16-row blocks that share the weight operand, so every weight byte is read once per
// launch. Partial tiles are summed through LDS (one tile value per wave) before the fused
// epilogue. Row sets come from the step control block (rows of one pulse, rows of one
// expert, all rows, or logits rows), so one launch serves every pulse / expert group and
// groups without rows exit before touching their weights.
//
// Prefill and other wide row sets: gemm_wide.hip.
//
// fp32: gemm_f32.hip.
#include <algorithm>

#include "gemm_common.h"

namespace pulsar {

namespace {

__device__ __forceinline__ bf16x8_t load_bf16x8(const bf16* p) {
  return *reinterpret_cast<const bf16x8_t*>(p);
}
// Non-temporal (streaming) load: for weights a launch reads once, so that they do not push
// out of the caches what later kernels read again (attention keys/values, activations).
__device__ __forceinline__ bf16x8_t load_bf16x8_nt(const bf16* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(p));
}

// Workgroup: 16 output columns of one group; 8 waves split K (few registers per wave, so
// a launch's workgroups are resident at once). The workgroup walks the
// group's 32-row tiles z, z + gridDim.z, ... keeping its weight slice in registers, so a
// launch needs only as many workgroups along z as the largest row set needs for
// parallelism (one for decode batches of up to 32 rows per group). KMUL0 > 1: the
// all-rows group has K0 = KMUL0 * K and runs KMUL0 passes over K-slices (the shared expert
// down projection fused into the routed one).
constexpr int kGemmWaves = 8;

// A launch with several row tiles per group is a 1-D grid over (column block x, group y,
// row tile z), ordered so that the z workgroups of one (x, y) run one after another on the
// same XCD: workgroup L goes to XCD L % 8, and within an XCD the slots enumerate (x, y)
// pairs with z fastest. They then share that XCD's L2 for the weight slice instead of each
// fetching it from HBM. Pairs are padded to a multiple of 8; padding workgroups exit.
// With one row tile (decode batches) the grid is the plain (x, y) grid: no index
// arithmetic ahead of the weight loads.
struct GemmBlock {
  int x, y, z;
  bool valid;
};
template <bool XCD>
__device__ __forceinline__ GemmBlock gemm_block(const GemmArgs& g) {
  if constexpr (!XCD) return GemmBlock{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, true};
  const int L = blockIdx.x, slot = L / kXcds;
  const int pair = (slot / g.grid_z) * kXcds + L % kXcds;
  GemmBlock b;
  b.z = slot % g.grid_z;
  b.x = pair % g.grid_x;
  b.y = pair / g.grid_x;
  b.valid = b.y < g.grid_y;
  return b;
}

// s_waitcnt vmcnt(n) for an n that is a constant once the caller's loops are unrolled.
__device__ __forceinline__ void wait_vmcnt_unrolled(int n) {
  switch (n) {
    case 0: wait_vmcnt<0>(); break;
    case 1: wait_vmcnt<1>(); break;
    case 2: wait_vmcnt<2>(); break;
    case 3: wait_vmcnt<3>(); break;
    case 4: wait_vmcnt<4>(); break;
    case 5: wait_vmcnt<5>(); break;
    case 6: wait_vmcnt<6>(); break;
    case 7: wait_vmcnt<7>(); break;
    default: wait_vmcnt<0>(); break;
  }
}

template <int EPI, int KITER, int MODE, int KMUL0, bool EAGER, bool XCD>
__global__ void __launch_bounds__(64 * kGemmWaves) gemm_bf16_kernel(GemmArgs g) {
  // two weight column tiles share each A operand: SwiGLU's gate and up columns, and the
  // output head's columns c and N + c (the host halves N: the head's A rows are then read
  // once per 32 vocabulary columns, not per 16)
  constexpr bool kPair = (EPI == EPI_SWIGLU || EPI == EPI_LOGITS);
  constexpr int kKPass = KITER * 32 * kGemmWaves;  // K covered by one pass of the waves
  static_assert(!EAGER || MODE == ROWS_LIST, "eager weight loads are for expert lists");
  // One LDS slice per wave: first the wave's A rows of a 16-row block (one 1 KB tile per
  // k tile and pass), then its partial tile values [value][lane] for the K-split sum (the
  // lanes of one value are consecutive words: conflict-free writes and reducing reads;
  // lane-major rows of 16 values put every 4th lane on one bank, 16-way conflicts). A wave
  // only writes its own slice, so the A staging needs no barrier.
  constexpr int kAFrags = KITER * KMUL0;
  constexpr int kRedFloats = (kPair ? 16 : 8) * 64;
  constexpr int kSliceFloats = kAFrags * 256 > kRedFloats ? kAFrags * 256 : kRedFloats;
  __shared__ __attribute__((aligned(16))) float lds_slices[kGemmWaves * kSliceFloats];
  const GemmBlock blk = gemm_block<XCD>(g);
  if (!blk.valid) return;
  // grid.y < g0_split: the optional all-rows group (group -1) when has_g0 is set. Its row
  // tiles go to g0_split x Z workgroups per column block (tile y Z + z, stride g0_split Z),
  // those of a list group to Z (tile z, stride Z): the all-rows group holds about K / E
  // times the rows of a routed expert, and one workgroup walking all of them would be the
  // launch's longest chain of dependent tiles.
  const int s0 = g.has_g0 ? g.g0_split : 0;
  const bool g0 = blk.y < s0;
  const int group = g0 ? -1 : blk.y - s0 + g.group_offset;
  const int N = g0 ? g.N0 : g.N;
  const int col0 = blk.x * 16;
  if (col0 >= N) return;
  const int zs = XCD ? g.grid_z : (int)gridDim.z;
  const int tstep = (g0 ? s0 * zs : zs) * 32;
  int tile0 = (g0 ? blk.y * zs + blk.z : blk.z) * 32;
  int cnt = 0;
  if constexpr (!EAGER) {
    cnt = group_rows<MODE>(g, group);  // uniform per workgroup
    if (tile0 >= cnt) return;
  } else {
    // the all-rows group's later tiles exist for parallelism at large steps: they check
    // the step's row count before streaming weights (the first tile never waits for it)
    if (g0 && tile0 > 0) {
      cnt = group_rows<MODE>(g, group);
      if (tile0 >= cnt) return;
    }
  }

  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = lane & 15, kq = lane >> 4;
  const int64_t lda = g0 ? g.lda0 : g.lda;
  const bf16* W = g0 ? reinterpret_cast<const bf16*>(g.W0)
                     : reinterpret_cast<const bf16*>(g.W) + (int64_t)group * g.w_group_stride;
  // Weights in matrix-core tiles [N/16][K/32][64 lanes][8]: this lane's 16 bytes of tile
  // (column tile, k tile) sit at ((ct * KT + kt) * 64 + lane) * 8, and the wave's load of a
  // tile is 1 KB contiguous. The up-projection rows of SwiGLU are column tiles N/16 on.
  const int KT = (g0 ? g.K0 : g.K) / 32;
  const bool vc = col0 + m < N;  // N is a multiple of 16: always true; kept as a guard
  const bf16* w0 = W + ((int64_t)(col0 / 16) * KT * 64 + lane) * 8;
  const bf16* w1 = W + ((int64_t)((N + col0) / 16) * KT * 64 + lane) * 8;
  const bf16* A = reinterpret_cast<const bf16*>(g0 ? g.A0 : g.A);
  void* Cout = g0 ? g.C0 : g.C;
  const int64_t ldc = g0 ? g.ldc0 : g.ldc;
  const int passes = g0 ? KMUL0 : 1;
  const int kb = wv * (KITER * 32) + kq * 8;
  const bf16x8_t zero = {};
  // every pass's weights stay in registers (the all-rows group of a KMUL0 launch loads its
  // second K half with the first, not one round trip after the first half's products)
  bf16x8_t bw[KITER * KMUL0], bu[KITER], xa[KITER];
  // k tile of step i of this wave in pass p: p * (K / 32 per pass) + wv * KITER + i
#define PULSAR_LOAD_W(pass)                                                              \
  do {                                                                                   \
    _Pragma("unroll") for (int i = 0; i < KITER; ++i) {                                  \
      const int64_t kt = (int64_t)(pass) * (kKPass / 32) + wv * KITER + i;               \
      bw[(pass) * KITER + i] = XCD ? load_bf16x8(w0 + kt * 512) : load_bf16x8_nt(w0 + kt * 512); \
      if constexpr (kPair)                                                               \
        bu[i] = XCD ? load_bf16x8(w1 + kt * 512) : load_bf16x8_nt(w1 + kt * 512);        \
    }                                                                                    \
  } while (0)
#define PULSAR_LOAD_W_REST()                                                             \
  do {                                                                                   \
    if constexpr (KMUL0 > 1) {                                                           \
      if (g0) {                                                                          \
        _Pragma("unroll") for (int p = 1; p < KMUL0; ++p) PULSAR_LOAD_W(p);              \
      }                                                                                  \
    }                                                                                    \
  } while (0)

  // Row entries of the first tile first, then the weights, then (after a scheduling
  // barrier) the A rows: vector loads retire in issue order, so waiting for the few entry
  // loads leaves every weight load in flight. Lanes past the last row re-read the last
  // entry (always in bounds) and use a zero A operand. Each lane loads two entries per
  // block: that of its fragment row m (for the A operand's zero test and the stores) and
  // that of the row sr = lane / 4 whose 16 bytes it stages into LDS.
  const int sr = lane >> 2;
  int n, i0, i1, l0, l1, si0, si1, ls0, ls1;
  if constexpr (EAGER) {
    // Most experts have rows (the host decides from the batch size): the first tile's
    // entries and the weights go out before the row count, whose scalar load retires apart
    // from them, instead of one round trip later. Entries past the count are read from the
    // list's spare capacity; the rows they name are clamped, computed and never stored.
    const int64_t cap = g.list_stride - 1;
    i0 = tile0 + m;
    i1 = tile0 + m + 16;
    const int32_t* lst = g.list + (int64_t)max(group, 0) * g.list_stride;
    si0 = tile0 + sr;
    si1 = tile0 + sr + 16;
    l0 = lst[min((int64_t)i0, cap)];
    l1 = lst[min((int64_t)i1, cap)];
    ls0 = lst[min((int64_t)si0, cap)];
    ls1 = lst[min((int64_t)si1, cap)];
    __builtin_amdgcn_sched_barrier(0);
    PULSAR_LOAD_W(0);
    // no early exit on the count: a branch on it would let the compiler test it before
    // issuing the weight loads. A workgroup without rows runs on clamped rows and stores
    // nothing.
    cnt = group_rows<MODE>(g, group);
    // Use the entries here: the wait for them then leaves the weight loads behind them in
    // flight, and the compiler cannot merge these loads into the next tile's (which would
    // put them behind the weights and the count).
    asm volatile("" ::"v"(l0), "v"(l1), "v"(ls0), "v"(ls1));
    n = max(0, min(32, cnt - tile0));
  } else {
    n = min(32, cnt - tile0);
    i0 = tile0 + min(m, n - 1);
    i1 = tile0 + min(m + 16, n - 1);
    si0 = tile0 + min(sr, n - 1);
    si1 = tile0 + min(sr + 16, n - 1);
    l0 = entry_load<MODE>(g, group, i0);
    l1 = entry_load<MODE>(g, group, i1);
    ls0 = entry_load<MODE>(g, group, si0);
    ls1 = entry_load<MODE>(g, group, si1);
    PULSAR_LOAD_W(0);
    PULSAR_LOAD_W_REST();
  }
  // One row tile (32 rows) of the group. The first tile runs outside the loop: in a
  // loop, the wait for the entries of a later tile (issued last) would also stand at the
  // first tile's A loads and make them wait for the whole weight slice.
  auto run_tile = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    const bool two = n > 16;  // second 16-row block present (uniform per workgroup)
    const int e0 = entry_fix<MODE>(group, i0, l0), e1 = entry_fix<MODE>(group, i1, l1);
    const int es0 = entry_fix<MODE>(group, si0, ls0), es1 = entry_fix<MODE>(group, si1, ls1);
    int ar0, ar1, as0, as1;  // ar: fragment row's A row (-1: zero operand); as: staged row
    if constexpr (EAGER) {
      // every lane of the first row block loads a row (clamped into the A buffer): rows
      // past the count are computed and never stored, so no A load waits on the count
      const int lim = (g0 ? g.a_rows0 : g.a_rows) - 1;
      ar0 = min(max(a_row_of<MODE>(g, group, e0), 0), lim);
      ar1 = m + 16 < n ? min(max(a_row_of<MODE>(g, group, e1), 0), lim) : -1;
      as0 = min(max(a_row_of<MODE>(g, group, es0), 0), lim);
      as1 = min(max(a_row_of<MODE>(g, group, es1), 0), lim);
    } else {
      ar0 = m < n ? a_row_of<MODE>(g, group, e0) : -1;
      ar1 = m + 16 < n ? a_row_of<MODE>(g, group, e1) : -1;
      as0 = a_row_of<MODE>(g, group, es0);  // rows past the count re-read the last row
      as1 = a_row_of<MODE>(g, group, es1);
    }
    // A rows through the wave's LDS slice: tile (pass p, k tile i) holds the block's 16
    // rows x 32 k as (row r, k chunk q) at slot 4 r + (q ^ 2 (r >> 3)); the load's lanes
    // 4 j .. 4 j + 3 fetch row j's 64 contiguous bytes (a register load's 16 lanes touched
    // 16 rows), and the fragment read (lane = row m, chunk kq) is free of bank conflicts.
    // With one pass the fragment reads wait for their own tile only (the A loads retire in
    // issue order, after the weights); a compiler barrier keeps each read behind its wait.
    bf16x8_t* astage = reinterpret_cast<bf16x8_t*>(lds_slices + wv * kSliceFloats);
    const int acl = (lane & 3) ^ ((lane >> 5) << 1);
    const int aslot = m * 4 + (kq ^ ((m >> 3) << 1));
    auto stage_a = [&](int as) {  // as: A row of block row sr
      const bf16* src = A + (int64_t)as * lda + wv * (KITER * 32) + acl * 8;
#pragma unroll
      for (int pass = 0; pass < KMUL0; ++pass) {
        if (pass >= passes) break;
#pragma unroll
        for (int i = 0; i < KITER; ++i)
          load_lds16(src + pass * kKPass + 32 * i, astage + (pass * KITER + i) * 64);
      }
    };
    // What the epilogue of this lane's output reads (the residual value or, in the gate
    // columns, the bias) goes out here, behind the weights and ahead of the rows: after the
    // products it would be one more round trip at the end of the launch. The C row of tile row
    // r is the entry held by lane r % 16 (rows 0-15: e0, 16-31: e1); entries past the row
    // count repeat the last row's.
    const int o_blk = wv >> 2, o_row = o_blk * 16 + kq * 4 + (wv & 3);
    const int o_crow = __shfl(o_blk ? e1 : e0, o_row & 15, 64) + g.c_row_offset;
    float pre = 0.f;
    if constexpr (EPI == EPI_RESID)
      pre = to_f(reinterpret_cast<const bf16*>(Cout)[(int64_t)o_crow * ldc + min(col0 + m, N - 1)]);
    if constexpr (EPI == EPI_QKVG) {
      if (col0 >= g.n_main)  // uniform
        pre = to_f(reinterpret_cast<const bf16*>(g.bias)[(int64_t)group * g.bias_group_stride +
                                                         min(col0 + m, N - 1) - g.n_main]);
    }
    f32x4_t c00 = {0.f, 0.f, 0.f, 0.f}, c10 = c00, c01 = c00, c11 = c00;
    auto wait_a = [&](int i) {  // before the fragment read of k tile i of the first pass
      if constexpr (KMUL0 == 1) {
        wait_vmcnt_unrolled(KITER - 1 - i);
        asm volatile("" ::: "memory");
      } else if (i == 0) {
        wait_vmcnt<0>();
        asm volatile("" ::: "memory");
      }
    };
    stage_a(as0);
#pragma unroll
    for (int pass = 0; pass < KMUL0; ++pass) {
      if (pass >= passes) break;
#pragma unroll
      for (int i = 0; i < KITER; ++i) {
        if (pass == 0) wait_a(i);
        xa[i] = (EAGER || ar0 >= 0) ? astage[(pass * KITER + i) * 64 + aslot] : zero;
      }
#pragma unroll
      for (int i = 0; i < KITER; ++i) {
        c00 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i], bw[pass * KITER + i], c00, 0, 0, 0);
        if constexpr (kPair) c01 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i], bu[i], c01, 0, 0, 0);
      }
    }
    if (two) {  // the second 16-row block reuses the slice once the first block's reads are in
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      stage_a(as1);
#pragma unroll
      for (int pass = 0; pass < KMUL0; ++pass) {
        if (pass >= passes) break;
#pragma unroll
        for (int i = 0; i < KITER; ++i) {
          if (pass == 0) wait_a(i);
          xa[i] = ar1 >= 0 ? astage[(pass * KITER + i) * 64 + aslot] : zero;
        }
#pragma unroll
        for (int i = 0; i < KITER; ++i) {
          c10 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i], bw[pass * KITER + i], c10, 0, 0, 0);
          if constexpr (kPair) c11 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i], bu[i], c11, 0, 0, 0);
        }
      }
    }
    // the partial values overwrite the slice: its A reads are done
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    // Partial tiles to LDS; then wave w reduces and stores tile value w of every lane:
    // row block w / 4, accumulator element w % 4 (with its up-projection twin for SwiGLU).
    float* red_w = lds_slices + wv * kSliceFloats;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      red_w[j * 64 + lane] = c00[j];
      red_w[(4 + j) * 64 + lane] = c10[j];
      if constexpr (kPair) {
        red_w[(8 + j) * 64 + lane] = c01[j];
        red_w[(12 + j) * 64 + lane] = c11[j];
      }
    }
    __syncthreads();
    {
      static_assert(kGemmWaves == 8, "one tile value per wave");
      const int blk = wv >> 2, j = wv & 3;
      float acc = 0.f, accu = 0.f;
#pragma unroll
      for (int w = 0; w < kGemmWaves; ++w) {
        acc += lds_slices[w * kSliceFloats + (blk * 4 + j) * 64 + lane];
        if constexpr (kPair) accu += lds_slices[w * kSliceFloats + (8 + blk * 4 + j) * 64 + lane];
      }
      // D layout of 16x16 MFMA: lane holds rows (lane/16)*4 + j, column lane%16
      if (vc && o_row < n) {
        epilogue<bf16>(g, EPI, group, Cout, ldc, o_crow, col0 + m, acc, accu, pre);
        if constexpr (EPI == EPI_LOGITS)
          epilogue<bf16>(g, EPI, group, Cout, ldc, o_crow, N + col0 + m, accu, 0.f, 0.f);
      }
    }
  };
  run_tile();
  tile0 += tstep;
  while (tile0 < cnt) {
    __syncthreads();  // the partial sums in LDS are consumed before the next tile's writes
    n = min(32, cnt - tile0);
    i0 = tile0 + min(m, n - 1);
    i1 = tile0 + min(m + 16, n - 1);
    si0 = tile0 + min(sr, n - 1);
    si1 = tile0 + min(sr + 16, n - 1);
    l0 = entry_load<MODE>(g, group, i0);
    l1 = entry_load<MODE>(g, group, i1);
    ls0 = entry_load<MODE>(g, group, si0);
    ls1 = entry_load<MODE>(g, group, si1);
    run_tile();
    tile0 += tstep;
  }
#undef PULSAR_LOAD_W
#undef PULSAR_LOAD_W_REST
}

// Mid-size row sets (tens to a few hundred rows per group: block verifies, large decode
// batches). A workgroup of 4 waves owns 64 rows of one group and CT weight column tiles of 16
// (SwiGLU: CT / 2 gate tiles and their up twins); wave w computes rows 16 w .. 16 w + 15
// against all CT tiles. Two 32-wide k tiles at a time, the weights and the wave's own rows go
// through a ring of S LDS stages with direct global-to-LDS loads (each wave fetches a quarter
// of the weights, all 4 read all of them; its rows it reads back alone). What bounds a launch
// is what a CU streams in: a workgroup moves (64 + 16 CT) x K x 2 bytes, most of them cold, at
// 30-50 bytes/ns per CU, so the CU with the most of them ends it (timing copies without the k
// loop or without the products put the 320-row verify's routed gate/up at 6.2 and 22.9 of
// its then 22.7 us, and rings of more buffers ran alike). The shapes are chosen at
// launch_mid_shape.
//
// Summation order: K is cut into the 8 chunks of gemm_bf16_kernel (wave w of that kernel
// takes k tiles p K/32 + w KITER + i, pass p, i < KITER), each chunk summed by one chain
// of matrix-core products from zero and the chunks added in order 0..7 to a zero start,
// as that kernel's LDS reduction does: the two kernels give identical results, so a
// caller picks either one by speed alone.
constexpr int kMidWaves = 4, kMidTileRows = 16 * kMidWaves;

// A mid-size tile: kMidTileRows rows and CT weight column tiles of 16, a ring of S stages.
template <int CT_, int S_>
struct MidShape {
  static constexpr int CT = CT_, S = S_;
  static constexpr int kStage = (2 * CT + 2 * kMidWaves) * 64;  // 16-byte chunks of a stage
  static constexpr int kLds = S * kStage;
  static_assert(CT % 2 == 0, "4 waves share the 2 CT weight loads of a stage");
  // output columns of a column block
  template <int EPI>
  static constexpr int columns() { return EPI == EPI_SWIGLU ? CT * 8 : CT * 16; }
};

// Tile of a 1-D mid-size launch: the tiles that hold rows, ordered (group, row tile,
// column block) with column blocks fastest and the fused all-rows group (has_g0, tiles of
// shape T0) first, are cut into 8 contiguous ranges, one per XCD, as in wide_tile.
template <int MODE, int EPI, class T, class T0>
__device__ __forceinline__ bool mid_tile(const GemmArgs& g, int& cb, int& group, int& rt,
                                         int& cnt) {
  const int L = (int)blockIdx.x, xcd = L % kXcds, slot = L / kXcds;
  const int lane = (int)threadIdx.x & 63;
  const int s0 = g.has_g0 ? 1 : 0;
  const int ng = g.grid_y + s0;  // at most 64 (host check)
  int rows = 0, nx = 0, items = 0;
  if (lane < ng) {
    const bool z = lane < s0;
    rows = min(group_rows<MODE>(g, z ? -1 : lane - s0 + g.group_offset), g.grid_z);
    nx = z ? (g.N0 + T0::template columns<EPI>() - 1) / T0::template columns<EPI>()
           : (g.N + T::template columns<EPI>() - 1) / T::template columns<EPI>();
    items = (rows + kMidTileRows - 1) / kMidTileRows * nx;
  }
  int total = 0;
  for (int j = 0; j < ng; ++j) total += __builtin_amdgcn_readlane(items, j);
  const int per = (total + kXcds - 1) / kXcds;
  int it = xcd * per + slot;
  if (slot >= per || it >= total) return false;
  for (int j = 0; j < ng; ++j) {
    const int ij = __builtin_amdgcn_readlane(items, j);
    if (it < ij) {
      const int nxj = __builtin_amdgcn_readlane(nx, j);
      group = j < s0 ? -1 : j - s0 + g.group_offset;
      rt = it / nxj;
      cb = it % nxj;
      cnt = __builtin_amdgcn_readlane(rows, j);
      return true;
    }
    it -= ij;
  }
  return false;
}

// One mid-size tile of K = PASSES passes of 8 KITER k tiles, visited chunk by chunk (chunk
// w: tiles p 8 KITER + w KITER + i, p < PASSES, i < KITER). smem: at least T::kLds chunks.
template <int EPI, int MODE, int KITER, int PASSES, class T>
__device__ __forceinline__ void mid_block(const GemmArgs& g, int cb, int group, int rt, int cnt,
                                          bf16x8_t* smem) {
  constexpr bool kPair = (EPI == EPI_SWIGLU);
  constexpr int CT = T::CT;
  constexpr int CK = KITER * PASSES, STEPS = 4 * CK, KB = 8 * KITER, KT = 8 * CK;
  constexpr int S = T::S < STEPS ? T::S : STEPS;  // ring buffers in use
  static_assert(S >= 2, "ring of at least 2 buffers");
  constexpr int NW = CT / 2, NA = 2;  // 1 KB loads of one wave per stage
  static_assert((S - 2) * (NW + NA) <= 63, "vmcnt range");
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = lane & 15, kq = lane >> 4;
  const bool g0 = group < 0;
  const int N = g0 ? g.N0 : g.N;
  const bf16* W = g0 ? reinterpret_cast<const bf16*>(g.W0)
                     : reinterpret_cast<const bf16*>(g.W) + (int64_t)group * g.w_group_stride;
  const bf16* A = reinterpret_cast<const bf16*>(g0 ? g.A0 : g.A);
  const int64_t lda = g0 ? g.lda0 : g.lda;
  void* Cout = g0 ? g.C0 : g.C;
  const int64_t ldc = g0 ? g.ldc0 : g.ldc;
  // k tile t of the chunk-ordered sequence; a stage's two lie side by side in memory unless
  // every k tile of a pass is a chunk of its own and there are several passes
  auto ktile = [](int t) { return ((t % CK) / KITER) * KB + (t / CK) * KITER + (t % CK) % KITER; };
  constexpr bool kAdjacent = KITER % 2 == 0 || PASSES == 1;
  // Unit u of a stage's 2 CT weight loads: weight tile u % CT of its k tile u / CT. Weight
  // tile c of the block: SwiGLU gate tiles (CT/2) cb + c for c < CT/2 and their up twins
  // N/16 on; otherwise tiles CT cb + c (tiles past N re-read the last one, never stored).
  // Wave wv takes units wv + 4 i.
  const bf16* wsrc[NW];
  int wk[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int c = (wv + 4 * i) % CT;
    wk[i] = (wv + 4 * i) / CT;
    int ct;
    if constexpr (kPair)
      ct = (c < CT / 2 ? 0 : N / 16 - CT / 2) + cb * (CT / 2) + c;
    else
      ct = min(cb * CT + c, N / 16 - 1);
    wsrc[i] = W + ((int64_t)ct * KT * 64 + lane) * 8 + (kAdjacent ? wk[i] * 512 : 0);
  }
  // The wave's 16 rows of a stage are two loads of 8 rows x 64 k: whole 128-byte lines. (One
  // k tile, half a line, per load had the next stage's load wait on the same line: 320-row
  // verify, routed gate/up 20.7 -> 18.6 us.) Lane l of load i fetches row 8 i + (l >> 3),
  // chunk (l & 7) ^ (row >> 1), so that a row's chunk q lies at slot 8 row + (q ^ (row >> 1))
  // and the fragment reads are free of LDS bank conflicts. Rows past the count re-read the
  // last row (computed, never stored); lane m's entry is that of the wave's row m.
  const int r0 = rt * kMidTileRows + wv * 16;
  const int im = min(r0 + m, cnt - 1);
  const int ent = entry_fix<MODE>(group, im, entry_load<MODE>(g, group, im));
  const bf16* asrc[NA];
  int ak[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int el = __shfl(ent, 8 * i + (lane >> 3), 64);
    const int chunk = (lane & 7) ^ (4 * i + (lane >> 4));
    ak[i] = chunk >> 2;
    asrc[i] = A + (int64_t)a_row_of<MODE>(g, group, el) * lda + (kAdjacent ? chunk : chunk & 3) * 8;
  }
  auto column = [&](int c) { return (cb * (kPair ? CT / 2 : CT) + c) * 16 + m; };
  auto fetch = [&](int j) {
    bf16x8_t* st = smem + (j % S) * T::kStage;
    const int k0 = ktile(2 * j), k1 = ktile(2 * j + 1);
#pragma unroll
    for (int i = 0; i < NW; ++i)
      load_lds16(wsrc[i] + (int64_t)(kAdjacent || !wk[i] ? k0 : k1) * 512, st + (wv + 4 * i) * 64);
#pragma unroll
    for (int i = 0; i < NA; ++i)
      load_lds16(asrc[i] + (kAdjacent || !ak[i] ? k0 : k1) * 32,
                 st + (2 * CT + 2 * wv + i) * 64);
  };
  // The residual values (the gate columns' bias) the epilogue reads go out ahead of the k loop:
  // loads and stores may alias as far as the compiler knows, so in the epilogue each of a
  // lane's 16 values waited for its load before the next one's went out (320-row verify: wo
  // 11.4 -> 9.7 us). D layout of 16x16 MFMA: lane holds rows 4 kq + j of its block, column m;
  // the C row of block row r is the entry held by lane r.
  constexpr int NPRE = EPI == EPI_RESID ? CT : 1;
  float pre[4][NPRE] = {};
  if constexpr (EPI == EPI_RESID) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t at = (int64_t)(__shfl(ent, kq * 4 + j, 64) + g.c_row_offset) * ldc;
#pragma unroll
      for (int c = 0; c < CT; ++c)
        pre[j][c] = to_f(reinterpret_cast<const bf16*>(Cout)[at + min(column(c), N - 1)]);
    }
  }
  float gate_bias[EPI == EPI_QKVG ? CT : 1] = {};
  if constexpr (EPI == EPI_QKVG) {
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int col = min(column(c), N - 1);
      if (col >= g.n_main)
        gate_bias[c] = to_f(reinterpret_cast<const bf16*>(
            g.bias)[(int64_t)group * g.bias_group_stride + col - g.n_main]);
    }
  }
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[CT], tot[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) tot[c] = zero;
#pragma unroll
  for (int j = 0; j < S - 1; ++j) fetch(j);
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    // stages stay in program order (the scheduler would otherwise keep several chunks'
    // accumulators live at once)
    __builtin_amdgcn_sched_barrier(0);
    // stage s's loads are done once at most the S - 2 younger stages' loads are
    // outstanding; the barrier publishes every wave's loads of stage s and retires stage
    // s - 1, whose buffer the next fetch fills
    if (s + S - 2 < STEPS)
      wait_vmcnt<(S - 2) * (NW + NA)>();
    else
      wait_vmcnt<0>();
    lds_barrier();
    if (s + S - 1 < STEPS) fetch(s + S - 1);
    const bf16x8_t* st = smem + (s % S) * T::kStage;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int t = 2 * s + h;
      bf16x8_t fw[CT];
#pragma unroll
      for (int c = 0; c < CT; ++c) fw[c] = st[(h * CT + c) * 64 + lane];
      const bf16x8_t xa = st[(2 * CT + 2 * wv) * 64 + m * 8 + ((4 * h + kq) ^ (m >> 1))];
      // a chunk's chain starts from zero
#pragma unroll
      for (int c = 0; c < CT; ++c)
        acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa, fw[c], t % CK == 0 ? zero : acc[c], 0,
                                                         0, 0);
      if ((t + 1) % CK == 0) {
#pragma unroll
        for (int c = 0; c < CT; ++c) tot[c] += acc[c];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int crow = __shfl(ent, kq * 4 + j, 64) + g.c_row_offset;
    if (r0 + kq * 4 + j >= cnt) continue;
    if constexpr (kPair) {
#pragma unroll
      for (int c = 0; c < CT / 2; ++c)
        epilogue<bf16>(g, EPI, group, Cout, ldc, crow, column(c), tot[c][j], tot[c + CT / 2][j],
                       0.f);
    } else {
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        if (column(c) < N)
          epilogue<bf16>(g, EPI, group, Cout, ldc, crow, column(c), tot[c][j], 0.f,
                         EPI == EPI_RESID  ? pre[j][NPRE > 1 ? c : 0]
                         : EPI == EPI_QKVG ? gate_bias[EPI == EPI_QKVG ? c : 0]
                                           : 0.f);
      }
    }
  }
}

// The groups in tiles of shape T, the fused all-rows group (K0 = KMUL0 K) in shape T0.
template <int EPI, int MODE, int KITER, int KMUL0, class T, class T0>
__global__ void __launch_bounds__(64 * kMidWaves, 2) gemm_bf16_mid_kernel(GemmArgs g) {
  __shared__ bf16x8_t smem[T::kLds > T0::kLds ? T::kLds : T0::kLds];
  int cb, group, rt, cnt;
  if (!mid_tile<MODE, EPI, T, T0>(g, cb, group, rt, cnt)) return;
  if constexpr (MODE == ROWS_LIST) {
    if (group < 0) {
      mid_block<EPI, MODE, KITER, KMUL0, T0>(g, cb, group, rt, cnt, smem);
      return;
    }
  }
  mid_block<EPI, MODE, KITER, 1, T>(g, cb, group, rt, cnt, smem);
}

template <int EPI, int MODE, int KMUL0, bool EAGER, bool XCD>
void launch_bf16_kx(const GemmArgs& a, dim3 grid, hipStream_t s) {
  constexpr int T = 64 * kGemmWaves;
  switch (a.K) {
    case 256: gemm_bf16_kernel<EPI, 1, MODE, KMUL0, EAGER, XCD><<<grid, T, 0, s>>>(a); break;
    case 512: gemm_bf16_kernel<EPI, 2, MODE, KMUL0, EAGER, XCD><<<grid, T, 0, s>>>(a); break;
    case 1024: gemm_bf16_kernel<EPI, 4, MODE, KMUL0, EAGER, XCD><<<grid, T, 0, s>>>(a); break;
    default: gemm_bf16_kernel<EPI, 8, MODE, KMUL0, EAGER, XCD><<<grid, T, 0, s>>>(a); break;
  }
}

template <int EPI, int MODE, int KMUL0, bool EAGER = false>
void launch_bf16_k(const GemmArgs& a, dim3 grid, hipStream_t s) {
  if (a.grid_z > 1) {
    // 1-D launch in the XCD-aware order of gemm_block
    const int pairs = (a.grid_x * a.grid_y + kXcds - 1) / kXcds * kXcds;
    launch_bf16_kx<EPI, MODE, KMUL0, EAGER, true>(a, dim3((unsigned)(pairs * a.grid_z)), s);
  } else {
    launch_bf16_kx<EPI, MODE, KMUL0, EAGER, false>(a, grid, s);
  }
}

// Row tiles walked by one workgroup of an expert-list or logits launch (weights stay in
// registers across them). Launches over the rows of a pulse (the attention projections,
// whose weights are a few MiB) give every 32-row tile its own workgroup: their tiles run
// in parallel, and the re-read weight slices come from the XCD's L2 (XCD-aware order
// below). The output head (64 MiB) measured slower that way at 320 rows (61 -> 75 us).
constexpr int kTilesPerWorkgroup = 4;
constexpr int kG0Split = 4;

template <int EPI>
int launch_one(const GemmArgs& a, int groups, int max_rows, hipStream_t s) {
  const int tiles = (max_rows + 31) / 32;
  if (tiles <= 0 || groups <= 0) return PULSAR_OK;
  int gy = groups + (a.has_g0 ? 1 : 0);
  const int nmax = a.has_g0 ? std::max(a.N, a.N0) : a.N;
  const int k0 = a.has_g0 ? a.K0 : a.K;
  if (a.K != 256 && a.K != 512 && a.K != 1024 && a.K != 2048)
    return fail(PULSAR_ERR_UNSUPPORTED, "gemm: K must be 256, 512, 1024 or 2048");
  if (a.has_g0 && (a.row_mode != ROWS_LIST || a.ctl == nullptr))
    return fail(PULSAR_ERR_INVALID,
                "gemm: the all-rows group fuses into list launches with a control block only");
  if (k0 != a.K && k0 != 2 * a.K)
    return fail(PULSAR_ERR_UNSUPPORTED, "gemm: the all-rows group needs K0 = K or 2K");
  const int per_wg = a.row_mode == ROWS_PULSE ? 1 : kTilesPerWorkgroup;
  const int gz = (tiles + per_wg - 1) / per_wg;
  // the all-rows group: one row tile per workgroup, up to kG0Split rows of the grid
  const int s0 = a.has_g0 ? std::min(kG0Split, (tiles + gz - 1) / gz) : 0;
  gy = groups + s0;
  dim3 grid((unsigned)((nmax + 15) / 16), (unsigned)gy, (unsigned)gz);
  GemmArgs ga = a;
  ga.g0_split = s0;
  ga.grid_x = (int)grid.x;
  ga.grid_y = (int)grid.y;
  ga.grid_z = (int)grid.z;
  switch (a.row_mode) {
    case ROWS_PULSE: launch_bf16_k<EPI, ROWS_PULSE, 1>(ga, grid, s); break;
    case ROWS_LIST:
      if (a.eager_w) {
        if (EPI != EPI_SWIGLU || k0 != a.K)
          return fail(PULSAR_ERR_UNSUPPORTED,
                      "gemm: eager expert launches are SwiGLU with K0 == K");
        if (a.a_rows < 1 || (a.has_g0 && a.a_rows0 < 1))
          return fail(PULSAR_ERR_INVALID, "gemm: eager expert launches need A row counts");
        if constexpr (EPI == EPI_SWIGLU) launch_bf16_k<EPI, ROWS_LIST, 1, true>(ga, grid, s);
      } else {
        if (k0 == a.K)
          launch_bf16_k<EPI, ROWS_LIST, 1>(ga, grid, s);
        else
          launch_bf16_k<EPI, ROWS_LIST, 2>(ga, grid, s);
      }
      break;
    case ROWS_ALL: launch_bf16_k<EPI, ROWS_ALL, 1>(ga, grid, s); break;
    case ROWS_LOGITS: launch_bf16_k<EPI, ROWS_LOGITS, 1>(ga, grid, s); break;
    default: return fail(PULSAR_ERR_INVALID, "gemm: row mode");
  }
  PULSAR_LAUNCH_CHECK();
  return PULSAR_OK;
}

template <int EPI, int MODE, int KMUL0, class T, class T0>
void launch_mid_k(const GemmArgs& a, dim3 grid, hipStream_t s) {
  constexpr int B = 64 * kMidWaves;
  switch (a.K) {
    case 256: gemm_bf16_mid_kernel<EPI, MODE, 1, KMUL0, T, T0><<<grid, B, 0, s>>>(a); break;
    case 512: gemm_bf16_mid_kernel<EPI, MODE, 2, KMUL0, T, T0><<<grid, B, 0, s>>>(a); break;
    case 1024: gemm_bf16_mid_kernel<EPI, MODE, 4, KMUL0, T, T0><<<grid, B, 0, s>>>(a); break;
    default: gemm_bf16_mid_kernel<EPI, MODE, 8, KMUL0, T, T0><<<grid, B, 0, s>>>(a); break;
  }
}

// Dense launches (rows of a pulse, all rows: one group) take 64 x 32 tiles, which give a few
// hundred rows enough workgroups (320 rows: QKV 9.5 us in 64 x 64 tiles, 7.6 in 64 x 32;
// output projection 9.3 and 7.4; 32 x 64 lies within 0.7 us of 64 x 32, 32 x 32 gained 0.3 on the
// one and lost 1.2 on the other). Expert lists take 64 x 128 (320-row verify: routed gate/up
// 18.8 us, 256 rows 16.6; 18.6 and 18.8 in 64 x 64, 18.1 and 21.5 in 96 x 64, 17.6 and 22.8 in
// 96 x 128: rows less evenly spread over the experts); an all-rows group of twice the K takes tiles of half
// the columns there, or its few tiles of twice the bytes end the launch (routed down 13.8 us
// in one shape, 12.8 so; 256 rows 12.9 and 11.4).
using MidDense = MidShape<2, 4>;
using MidList = MidShape<8, 3>;
using MidListK2 = MidShape<4, 3>;

template <int EPI>
int launch_mid_shape(const GemmArgs& a, int groups, int max_rows, hipStream_t s) {
  const bool list = a.row_mode == ROWS_LIST, k2 = a.has_g0 && a.K0 == 2 * a.K;
  const int cw = list ? MidList::columns<EPI>() : MidDense::columns<EPI>();
  const int cw0 = k2 ? MidListK2::columns<EPI>() : MidList::columns<EPI>();
  // SwiGLU blocks pair gate columns with their up twins: whole blocks only
  if (a.N % (EPI == EPI_SWIGLU ? cw : 16) != 0 ||
      (a.has_g0 && a.N0 % (EPI == EPI_SWIGLU ? cw0 : 16) != 0))
    return fail(PULSAR_ERR_UNSUPPORTED, "gemm: mid-size tiles need N % 16 == 0 (SwiGLU: a "
                                        "multiple of the column block)");
  GemmArgs ga = a;
  ga.grid_y = groups;
  ga.grid_z = max_rows;
  const int64_t tiles = ((int64_t)max_rows + kMidTileRows - 1) / kMidTileRows;
  int64_t items = groups * tiles * ((a.N + cw - 1) / cw);
  if (a.has_g0) items += tiles * ((a.N0 + cw0 - 1) / cw0);
  if (items > (int64_t)1 << 30) return fail(PULSAR_ERR_INVALID, "gemm: mid-size launch too large");
  const dim3 grid((unsigned)((items + kXcds - 1) / kXcds * kXcds));
  switch (a.row_mode) {
    case ROWS_PULSE: launch_mid_k<EPI, ROWS_PULSE, 1, MidDense, MidDense>(ga, grid, s); break;
    case ROWS_ALL: launch_mid_k<EPI, ROWS_ALL, 1, MidDense, MidDense>(ga, grid, s); break;
    case ROWS_LIST:
      if (k2)
        launch_mid_k<EPI, ROWS_LIST, 2, MidList, MidListK2>(ga, grid, s);
      else
        launch_mid_k<EPI, ROWS_LIST, 1, MidList, MidList>(ga, grid, s);
      break;
    default: return fail(PULSAR_ERR_INVALID, "gemm: row mode of a mid-size launch");
  }
  PULSAR_LAUNCH_CHECK();
  return PULSAR_OK;
}

template <int EPI>
int launch_mid(const GemmArgs& a, int groups, int max_rows, hipStream_t s) {
  if (groups <= 0 || max_rows <= 0) return PULSAR_OK;
  if (a.K != 256 && a.K != 512 && a.K != 1024 && a.K != 2048)
    return fail(PULSAR_ERR_UNSUPPORTED, "gemm: K must be 256, 512, 1024 or 2048");
  if (a.has_g0 && (a.row_mode != ROWS_LIST || a.ctl == nullptr))
    return fail(PULSAR_ERR_INVALID,
                "gemm: the all-rows group fuses into list launches with a control block only");
  if (a.has_g0 && a.K0 != a.K && a.K0 != 2 * a.K)
    return fail(PULSAR_ERR_UNSUPPORTED, "gemm: the all-rows group needs K0 = K or 2K");
  if (groups + (a.has_g0 ? 1 : 0) > 64)
    return fail(PULSAR_ERR_UNSUPPORTED, "gemm: mid-size tiles take at most 64 groups");
  return launch_mid_shape<EPI>(a, groups, max_rows, s);
}

}  // namespace

int launch_gemm_mid(const GemmArgs& a, int dtype, int epi, int groups, int max_rows,
                    hipStream_t s) {
  if (dtype != PULSAR_BF16) return launch_gemm(a, dtype, epi, groups, max_rows, s);
  switch (epi) {
    case EPI_STORE: return launch_mid<EPI_STORE>(a, groups, max_rows, s);
    case EPI_QKVG: return launch_mid<EPI_QKVG>(a, groups, max_rows, s);
    case EPI_RESID: return launch_mid<EPI_RESID>(a, groups, max_rows, s);
    case EPI_SWIGLU: return launch_mid<EPI_SWIGLU>(a, groups, max_rows, s);
  }
  return launch_gemm(a, dtype, epi, groups, max_rows, s);
}

int launch_gemm(const GemmArgs& a, int dtype, int epi, int groups, int max_rows, hipStream_t s) {
  if (a.K % 256 != 0)
    return fail(PULSAR_ERR_UNSUPPORTED, "gemm: K must be a multiple of 256");
  if (dtype != PULSAR_BF16) return launch_gemm_f32(a, epi, groups, max_rows, false, s);
  switch (epi) {
    case EPI_STORE: return launch_one<EPI_STORE>(a, groups, max_rows, s);
    case EPI_QKVG: return launch_one<EPI_QKVG>(a, groups, max_rows, s);
    case EPI_RESID: return launch_one<EPI_RESID>(a, groups, max_rows, s);
    case EPI_SWIGLU: return launch_one<EPI_SWIGLU>(a, groups, max_rows, s);
    case EPI_LOGITS: {
      // column pairs (c, N/2 + c) per workgroup
      if (a.N % 32 != 0) return fail(PULSAR_ERR_UNSUPPORTED, "gemm: logits N % 32 != 0");
      GemmArgs h = a;
      h.N = a.N / 2;
      return launch_one<EPI_LOGITS>(h, groups, max_rows, s);
    }
    case EPI_LOGITS_RAW: return launch_one<EPI_LOGITS_RAW>(a, groups, max_rows, s);
    case EPI_SCALE: return launch_one<EPI_SCALE>(a, groups, max_rows, s);
  }
  return fail(PULSAR_ERR_INVALID, "gemm: unknown epilogue");
}

}  // namespace pulsar

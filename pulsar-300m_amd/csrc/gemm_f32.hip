// Row-set GEMMs in fp32 (weights row-major [N][K]): C[rows, N] = epi(A[rows, K] . W[N, K]^T).
//
// A few rows (decode): one wave per output column, lanes split K with 128-bit loads, wave64
// reduction. Prefill: 32 x 32 tiles on the matrix cores.
#include <algorithm>

#include "gemm_common.h"

namespace pulsar {

namespace {

// Resolve the (A row, C row) pairs of this workgroup's 32-row tile into LDS (launches without
// an all-rows group).
// Returns the number of valid rows (0 => nothing to do).
__device__ int resolve_rows(const GemmArgs& g, int group, int tile, int* a_row, int* c_row) {
  __shared__ int s_n;
  const int mode = g.row_mode;
  if (threadIdx.x == 0) {
    int n = 0;
    switch (mode) {
      case ROWS_PULSE: {
        const int cnt = g.ctl->pulse_count[group];
        n = cnt - tile * 32;
        break;
      }
      case ROWS_LIST:
        n = g.list_count[group * kCountStride] - tile * 32;
        break;
      case ROWS_ALL: {
        const int tot = g.ctl ? g.ctl->n_rows : g.m_fixed;
        n = tot - tile * 32;
        break;
      }
      case ROWS_LOGITS:
        n = g.ctl->n_lrows - tile * 32;
        break;
    }
    s_n = n < 0 ? 0 : (n > 32 ? 32 : n);
  }
  __syncthreads();
  const int n = s_n;
  if (threadIdx.x < 32) {
    const int m = threadIdx.x;
    int ar = -1, cr = -1;
    if (m < n) {
      const int i = tile * 32 + m;
      switch (mode) {
        case ROWS_PULSE:
          ar = cr = g.ctl->pulse_start[group] + i;
          break;
        case ROWS_LIST: {
          const int e = g.list[(int64_t)group * g.list_stride + i];
          ar = e / g.a_div;
          cr = e;
          break;
        }
        case ROWS_ALL:
          ar = cr = i;
          break;
        case ROWS_LOGITS:
          ar = cr = i;
          break;
      }
    }
    a_row[m] = ar;
    c_row[m] = cr < 0 ? -1 : cr + g.c_row_offset;
  }
  __syncthreads();
  return n;
}

// What an output's epilogue reads: the residual value, or a gate column's bias.
template <int EPI>
__device__ __forceinline__ float epilogue_operand(const GemmArgs& g, int group, const void* C,
                                                  int64_t ldc, int crow, int col) {
  if constexpr (EPI == EPI_RESID)
    return reinterpret_cast<const float*>(C)[(int64_t)crow * ldc + col];
  if constexpr (EPI == EPI_QKVG)
    return col < g.n_main ? 0.f
                          : reinterpret_cast<const float*>(
                                g.bias)[(int64_t)group * g.bias_group_stride + col - g.n_main];
  return 0.f;
}

// A few rows: 4 waves per workgroup, one output column per wave, 32-row tile. The wave's
// weights (K up to 256 KI) go out as soon as the row count is known and stay in registers for
// every row; the row entries are loaded behind them, one per lane, and broadcast, and two
// rows' operands are in flight at a time. With the rows resolved through LDS first and the
// weights read again for each row, one row after another, 2 rows of a 1024-wide model took
// 5.5 us for qkv + gate, 5.0 for wo, 9.7 for the shared + routed gate/up (up to 36 MB: 3.9
// TB/s now) and 19.7 for the output head; here 5.0, 4.5, 9.2 and 14.8. KI = 0: any K, weights read per pair of rows.
template <int EPI, int KI>
__global__ void __launch_bounds__(256) gemm_f32_kernel(GemmArgs g) {
  constexpr bool kPair = (EPI == EPI_SWIGLU);
  const int group = (int)blockIdx.y + g.group_offset - (g.has_g0 ? 1 : 0);
  const bool g0 = group < 0;
  const int N = g0 ? g.N0 : g.N;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = (int)blockIdx.x * 4 + wv, r0 = (int)blockIdx.z * 32;
  if (col >= N) return;
  const int mode = g0 ? ROWS_ALL : g.row_mode;
  int cnt = 0, first = 0;
  switch (mode) {
    case ROWS_PULSE:
      cnt = g.ctl->pulse_count[group];
      first = g.ctl->pulse_start[group];
      break;
    case ROWS_LIST: cnt = g.list_count[group * kCountStride]; break;
    case ROWS_ALL: cnt = g.ctl ? g.ctl->n_rows : g.m_fixed; break;
    case ROWS_LOGITS: cnt = g.ctl->n_lrows; break;
  }
  const int n = min(32, cnt - r0);
  if (n <= 0) return;
  const float* A = reinterpret_cast<const float*>(g0 ? g.A0 : g.A);
  const int64_t lda = g0 ? g.lda0 : g.lda, ldw = g0 ? g.ldw0 : g.ldw;
  const float* W = g0 ? reinterpret_cast<const float*>(g.W0)
                      : reinterpret_cast<const float*>(g.W) + (int64_t)group * g.w_group_stride;
  void* Cout = g0 ? g.C0 : g.C;
  const int64_t ldc = g0 ? g.ldc0 : g.ldc;
  const float* w0 = W + (int64_t)col * ldw + lane * 4;
  const float* w1 = W + (int64_t)(N + col) * ldw + lane * 4;
  const int steps = (g0 ? g.K0 : g.K) / 256;
  f32x4_t wr[KI > 0 ? KI : 1], ur[kPair && KI > 0 ? KI : 1];
  if constexpr (KI > 0) {
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      if (i >= steps) break;  // a group of a shorter K than the all-rows group's
      wr[i] = *reinterpret_cast<const f32x4_t*>(w0 + 256 * i);
      if constexpr (kPair) ur[i] = *reinterpret_cast<const f32x4_t*>(w1 + 256 * i);
    }
  }
  // lane i: entry (C row) and A row of tile row i
  const int i = r0 + min(lane, n - 1);
  const int entry = mode == ROWS_LIST ? g.list[(int64_t)group * g.list_stride + i] : first + i;
  const int arow = mode == ROWS_LIST ? entry / g.a_div : entry;
  for (int r = 0; r < n; r += 2) {
    const int r2 = min(r + 1, n - 1);
    const float* a0 = A + (int64_t)__builtin_amdgcn_readlane(arow, r) * lda + lane * 4;
    const float* a1 = A + (int64_t)__builtin_amdgcn_readlane(arow, r2) * lda + lane * 4;
    const int c0 = __builtin_amdgcn_readlane(entry, r) + g.c_row_offset;
    const int c1 = __builtin_amdgcn_readlane(entry, r2) + g.c_row_offset;
    const float p0 = epilogue_operand<EPI>(g, group, Cout, ldc, c0, col);
    const float p1 = epilogue_operand<EPI>(g, group, Cout, ldc, c1, col);
    float s[2] = {0.f, 0.f}, u[2] = {0.f, 0.f};
    auto dot = [](const f32x4_t& a, const f32x4_t& b) {
      return a[0] * b[0] + a[1] * b[1] + a[2] * b[2] + a[3] * b[3];
    };
    auto add = [&](const f32x4_t& x0, const f32x4_t& x1, const f32x4_t& w, const f32x4_t& v) {
      s[0] += dot(x0, w);
      s[1] += dot(x1, w);
      if constexpr (kPair) {
        u[0] += dot(x0, v);
        u[1] += dot(x1, v);
      }
    };
    if constexpr (KI > 0) {
      f32x4_t x0[KI], x1[KI];
#pragma unroll
      for (int k = 0; k < KI; ++k) {
        if (k >= steps) break;
        x0[k] = *reinterpret_cast<const f32x4_t*>(a0 + 256 * k);
        x1[k] = *reinterpret_cast<const f32x4_t*>(a1 + 256 * k);
      }
#pragma unroll
      for (int k = 0; k < KI; ++k) {
        if (k >= steps) break;
        add(x0[k], x1[k], wr[k], ur[kPair ? k : 0]);
      }
    } else {
      for (int k = 0; k < steps; ++k) {
        const f32x4_t w = *reinterpret_cast<const f32x4_t*>(w0 + 256 * k);
        f32x4_t v = w;
        if constexpr (kPair) v = *reinterpret_cast<const f32x4_t*>(w1 + 256 * k);
        add(*reinterpret_cast<const f32x4_t*>(a0 + 256 * k),
            *reinterpret_cast<const f32x4_t*>(a1 + 256 * k), w, v);
      }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      s[q] = wave_sum(s[q]);
      if constexpr (kPair) u[q] = wave_sum(u[q]);
    }
    if (lane == 0) epilogue<float>(g, EPI, group, Cout, ldc, c0, col, s[0], u[0], p0);
    if (lane == 1 && r + 1 < n) epilogue<float>(g, EPI, group, Cout, ldc, c1, col, s[1], u[1], p1);
  }
}

// Rows of a prompt: a workgroup computes a 32-row x 32-column tile (SwiGLU: 32 gate columns and
// their up twins) with v_mfma_f32_16x16x4_f32; wave w sums k in [w K/4, (w + 1) K/4) and the
// four partial tiles meet in LDS, so that a workgroup reads each operand byte once and a short
// prompt's launches fill the chip (128 rows, N = 1024: 128 workgroups of 256 KB). Lane
// (m = l % 16, q = l / 16) loads 16 bytes, k0 + 4 q .. + 3, of row or column m: product j of a
// 16-wide k chunk then takes element j of each, the same permutation of k on both sides. The
// next 64 k of the wave are in flight during one 64's products. One wave per column and row
// after row took 44-61 us per projection of 128 rows (14-16 here), 84 for the routed down (21)
// and 237 for the routed gate/up (36).
template <int EPI>
__global__ void __launch_bounds__(256, 2) gemm_f32_tile_kernel(GemmArgs g) {
  constexpr bool kPair = (EPI == EPI_SWIGLU);
  constexpr int NT = kPair ? 4 : 2;  // 16-column tiles (SwiGLU: 2 gate, 2 up)
  constexpr int CH = 4;              // 16-wide chunks loaded together
  __shared__ int a_row[32], c_row[32];
  __shared__ float red[4][2][NT][4][64];  // [wave][row tile][column tile][value][lane]
  const int group = (int)blockIdx.y + g.group_offset;
  const int N = g.N, col0 = (int)blockIdx.x * 32;
  const int n = resolve_rows(g, group, blockIdx.z, a_row, c_row);
  if (n == 0) return;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, m = lane & 15, kq = lane >> 4;
  const int64_t koff = (int64_t)wv * (g.K / 4) + kq * 4;
  const float* W = reinterpret_cast<const float*>(g.W) + (int64_t)group * g.w_group_stride + koff;
  const float* ap[2];
  const float* wp[NT];
#pragma unroll
  for (int t = 0; t < 2; ++t) {  // rows past the tile's count re-read its first (never stored)
    const int i = t * 16 + m;
    ap[t] = reinterpret_cast<const float*>(g.A) + (int64_t)a_row[i < n ? i : 0] * g.lda + koff;
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int c = min(col0 + (t & 1) * 16 + m, N - 1) + (t >> 1) * N;
    wp[t] = W + (int64_t)c * g.ldw;
  }
  f32x4_t acc[2][NT];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int c = 0; c < NT; ++c) acc[t][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  f32x4_t av[2][CH][2], wv4[2][CH][NT];
  auto load = [&](int b, int k) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
#pragma unroll
      for (int t = 0; t < 2; ++t) av[b][c][t] = *reinterpret_cast<const f32x4_t*>(ap[t] + k + 16 * c);
#pragma unroll
      for (int t = 0; t < NT; ++t) wv4[b][c][t] = *reinterpret_cast<const f32x4_t*>(wp[t] + k + 16 * c);
    }
  };
  auto mul = [&](int b) {
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int u = 0; u < NT; ++u)
            acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[b][c][t][j], wv4[b][c][u][j], acc[t][u], 0, 0, 0);
  };
  const int steps = g.K / 256;  // of 64 k per wave
  load(0, 0);
  for (int s = 0; s < steps; s += 2) {
    if (s + 1 < steps) load(1, (s + 1) * 64);
    mul(0);
    if (s + 1 < steps) {
      if (s + 2 < steps) load(0, (s + 2) * 64);
      mul(1);
    }
  }
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) red[wv][t][u][j][lane] = acc[t][u][j];
  __syncthreads();
  // D layout of 16x16: lane holds rows 4 (lane / 16) + j, column lane % 16
  const int row = threadIdx.x >> 3, t = row >> 4, j = row & 3, l0 = ((row & 15) >> 2) * 16;
  if (row >= n) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int c = (threadIdx.x & 7) * 4 + e, u = c >> 4, l = l0 + (c & 15);
    if (col0 + c >= N) break;
    float v = 0.f, up = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      v += red[w][t][u][j][l];
      if constexpr (kPair) up += red[w][t][u + 2][j][l];
    }
    epilogue<float>(g, EPI, group, g.C, g.ldc, c_row[row], col0 + c, v, up,
                    epilogue_operand<EPI>(g, group, g.C, g.ldc, c_row[row], col0 + c));
  }
}

template <int EPI>
int launch_f32(const GemmArgs& a, int groups, int max_rows, bool tiles, hipStream_t s) {
  const int nt = (max_rows + 31) / 32;
  if (nt <= 0 || groups <= 0) return PULSAR_OK;
  if (tiles) {
    const dim3 grid((unsigned)((a.N + 31) / 32), (unsigned)groups, (unsigned)nt);
    gemm_f32_tile_kernel<EPI><<<grid, 256, 0, s>>>(a);
  } else {
    const int nmax = a.has_g0 ? std::max(a.N, a.N0) : a.N;
    const dim3 grid((unsigned)((nmax + 3) / 4), (unsigned)(groups + (a.has_g0 ? 1 : 0)), (unsigned)nt);
    // registers for the weights of the common widths
    switch (a.has_g0 ? std::max(a.K, a.K0) : a.K) {
      case 256: gemm_f32_kernel<EPI, 1><<<grid, 256, 0, s>>>(a); break;
      case 512: gemm_f32_kernel<EPI, 2><<<grid, 256, 0, s>>>(a); break;
      case 1024: gemm_f32_kernel<EPI, 4><<<grid, 256, 0, s>>>(a); break;
      default: gemm_f32_kernel<EPI, 0><<<grid, 256, 0, s>>>(a); break;
    }
  }
  PULSAR_LAUNCH_CHECK();
  return PULSAR_OK;
}

}  // namespace

int launch_gemm_f32(const GemmArgs& a, int epi, int groups, int max_rows, bool tiles,
                    hipStream_t s) {
  if (tiles && (a.has_g0 || a.K % 256 != 0))
    return fail(PULSAR_ERR_UNSUPPORTED, "gemm: fp32 tiles take K % 256 == 0 and no all-rows group");
  switch (epi) {
    case EPI_STORE: return launch_f32<EPI_STORE>(a, groups, max_rows, tiles, s);
    case EPI_QKVG: return launch_f32<EPI_QKVG>(a, groups, max_rows, tiles, s);
    case EPI_RESID: return launch_f32<EPI_RESID>(a, groups, max_rows, tiles, s);
    case EPI_SWIGLU: return launch_f32<EPI_SWIGLU>(a, groups, max_rows, tiles, s);
    case EPI_LOGITS: return launch_f32<EPI_LOGITS>(a, groups, max_rows, tiles, s);
    case EPI_LOGITS_RAW: return launch_f32<EPI_LOGITS_RAW>(a, groups, max_rows, tiles, s);
    case EPI_SCALE: return launch_f32<EPI_SCALE>(a, groups, max_rows, tiles, s);
  }
  return fail(PULSAR_ERR_INVALID, "gemm: unknown epilogue");
}

}  // namespace pulsar

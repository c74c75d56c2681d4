// Backward ops of the pulsar_cuda surface (the reference's training path through
// model.forward), written for gfx950 (wave64). Each is the exact gradient of the matching
// forward op, in fp32 arithmetic with outputs in the reference's dtypes: activations in the
// activation dtype, norm / conv weights in fp32. Weight gradients are summed with fp32
// atomics (one per element per workgroup), so their rounding depends on scheduling order,
// as the reference's does.
#include <algorithm>
#include <string>
#include <type_traits>

#include "common.h"

namespace pulsar {

namespace {

__global__ void fill_f32_kernel(float* p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

template <typename T>
__global__ void fill_zero_kernel(T* p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = from_f<T>(0.f);
}
__global__ void fill_zero_vec_kernel(uint4* p, int64_t n) {
  const int64_t i0 = (int64_t)blockIdx.x * 1024 + threadIdx.x;
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (i0 + u * 256 < n) p[i0 + u * 256] = make_uint4(0u, 0u, 0u, 0u);
}

#define PULSAR_TRY_STATUS(expr)     \
  do {                              \
    const int _st = (expr);         \
    if (_st != PULSAR_OK) return _st; \
  } while (0)

int zero_f32(float* p, int64_t n, hipStream_t s) {
  if (n <= 0) return PULSAR_OK;
  fill_f32_kernel<<<blocks_for(n, 256), 256, 0, s>>>(p, n);
  PULSAR_LAUNCH_CHECK();
  return PULSAR_OK;
}

// ---------------------------------------------------------------------------
// RMSNorm: y = w * x * r, r = rsqrt(mean(x^2) + eps) (saved by the forward).
//   dx = r * w * dy - x * r^3 * sum(dy * x * w) / D ;  dw = sum_rows dy * x * r
// Workgroups stride over rows; a thread keeps its columns' dw partials in registers
// (D <= 256 * kNormCols) and adds them once.
// ---------------------------------------------------------------------------
constexpr int kNormCols = 32;

template <typename T>
__global__ void __launch_bounds__(256) rmsnorm_bwd_kernel(const T* __restrict__ dy,
                                                          const T* __restrict__ x,
                                                          const float* __restrict__ w,
                                                          const float* __restrict__ rsq,
                                                          T* __restrict__ dx,
                                                          float* __restrict__ dw, int64_t rows,
                                                          int dim) {
  __shared__ float red[16];
  float acc[kNormCols];
#pragma unroll
  for (int j = 0; j < kNormCols; ++j) acc[j] = 0.f;
  const float inv_dim = 1.0f / (float)dim;
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const T* dyr = dy + row * dim;
    const T* xr = x + row * dim;
    const float r = rsq[row];
    float part = 0.f;
#pragma unroll
    for (int j = 0; j < kNormCols; ++j) {
      const int i = threadIdx.x + j * 256;
      if (i < dim) {
        const float g = to_f(dyr[i]), xv = to_f(xr[i]);
        part += g * xv * w[i];
        acc[j] += g * xv * r;
      }
    }
    const float tot = block_sum(part, red);
    const float c = r * r * r * tot * inv_dim;
#pragma unroll
    for (int j = 0; j < kNormCols; ++j) {
      const int i = threadIdx.x + j * 256;
      if (i < dim) dx[row * dim + i] = from_f<T>(r * w[i] * to_f(dyr[i]) - to_f(xr[i]) * c);
    }
    __syncthreads();  // red is reused by the next row's sum
  }
#pragma unroll
  for (int j = 0; j < kNormCols; ++j) {
    const int i = threadIdx.x + j * 256;
    if (i < dim) atomicAdd(&dw[i], acc[j]);
  }
}

// The same over 16-byte chunks: one wave per row (no barrier between rows), RPI rows of a
// wave in flight at a time, lane l holding chunks l + 64 j of a row and the dw partials of
// their columns; the 4 waves' partials meet in LDS and each column is added once per
// workgroup. dim % kVec == 0 and dim <= 64 kVec NC. Bound by memory: 16384 rows of 1024 in
// bf16 took 137 us in 2-byte loads with 1024 workgroups' atomics, 27.5 us here (512
// workgroups; 3.7 TB/s).
template <typename T, int NC, int RPI>
__global__ void __launch_bounds__(256) rmsnorm_bwd_vec_kernel(const T* __restrict__ dy,
                                                              const T* __restrict__ x,
                                                              const float* __restrict__ w,
                                                              const float* __restrict__ rsq,
                                                              T* __restrict__ dx,
                                                              float* __restrict__ dw,
                                                              int64_t rows, int dim) {
  constexpr int V = kVec<T>;
  __shared__ __attribute__((aligned(16))) float red[4][64 * NC * V];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nch = dim / V;
  int at[NC];  // element offset of chunk j in its row; chunks past it re-read the last one as zero
  float wt[NC][V], acc[NC][V];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int c = lane + 64 * j;
    at[j] = min(c, nch - 1) * V;
    ldv<V>(w + at[j], wt[j]);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      if (c >= nch) wt[j][e] = 0.f;  // its factor is zero, but the weight may be infinite
      acc[j][e] = 0.f;
    }
  }
  const float inv_dim = 1.0f / (float)dim;
  const int64_t step = (int64_t)gridDim.x * 4 * RPI;
  for (int64_t row0 = ((int64_t)blockIdx.x * 4 + wv) * RPI; row0 < rows; row0 += step) {
    uint4 rg[RPI][NC], rx[RPI][NC];
    float r[RPI];
#pragma unroll
    for (int i = 0; i < RPI; ++i) {
      const int64_t row = row0 + i < rows ? row0 + i : rows - 1;
      r[i] = rsq[row];
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        rg[i][j] = *reinterpret_cast<const uint4*>(dy + row * dim + at[j]);
        rx[i][j] = *reinterpret_cast<const uint4*>(x + row * dim + at[j]);
        if (lane + 64 * j >= nch) rg[i][j] = rx[i][j] = make_uint4(0u, 0u, 0u, 0u);
      }
    }
#pragma unroll
    for (int i = 0; i < RPI; ++i) {
      if (row0 + i >= rows) break;
      float part = 0.f;
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        float g[V], xv[V];
        unpackv<T>(rg[i][j], g);
        unpackv<T>(rx[i][j], xv);
#pragma unroll
        for (int e = 0; e < V; ++e) {
          part += g[e] * xv[e] * wt[j][e];
          acc[j][e] += g[e] * xv[e] * r[i];
        }
      }
      const float c = r[i] * r[i] * r[i] * wave_sum(part) * inv_dim;
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        float g[V], xv[V], o[V];
        unpackv<T>(rg[i][j], g);
        unpackv<T>(rx[i][j], xv);
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = r[i] * wt[j][e] * g[e] - xv[e] * c;
        if (lane + 64 * j < nch) stv<V>(dx + (row0 + i) * dim + at[j], o);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NC; ++j) stv<V>(&red[wv][(lane + 64 * j) * V], acc[j]);
  __syncthreads();
  for (int i = threadIdx.x; i < dim; i += 256)
    unsafeAtomicAdd(&dw[i], red[0][i] + red[1][i] + red[2][i] + red[3][i]);
}

// ---------------------------------------------------------------------------
// QK RMSNorm + RoPE (head_dim 64): y = rope(n), n = x * r * w[h]. One wave per vector.
//   dn = rope^T(dy) (rotation by -theta: dn_i = dy_i c + dy_{i+32} s,
//        dn_{i+32} = dy_{i+32} c - dy_i s)
//   dx = r * w * dn - x * r^3 * sum(dn * x * w) / 64 ;  dw[h] = sum dn * x * r
// Grid (workgroups per head, H): the waves of head h stride over its B*T vectors, keep
// their dw partial in a register and add it once.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) qk_norm_rope_bwd_kernel(
    const T* __restrict__ dy, const T* __restrict__ x, int64_t sB, int64_t sH, int64_t sT,
    int64_t dB, int64_t dH, int64_t dT, int H, int T_, int64_t per_head,
    const float* __restrict__ w, const float* __restrict__ rsq, const float* __restrict__ cs,
    const float* __restrict__ sn, T* __restrict__ dx, float* __restrict__ dw) {
  const int h = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x / 64);
  const int j = lane & 31;
  const float wv = w[h * 64 + lane];
  float dwacc = 0.f;
  for (int64_t i = (int64_t)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6); i < per_head;
       i += nwaves) {
    const int64_t b = i / T_;
    const int t = (int)(i % T_);
    const int64_t v = (b * H + h) * T_ + t;  // vector index in [B, H, T] order
    const float g = to_f(dy[v * 64 + lane]);
    const float gp = __shfl_xor(g, 32, 64);
    const float c = cs[t * 32 + j], s = sn[t * 32 + j];
    const float dn = lane < 32 ? g * c + gp * s : g * c - gp * s;
    const float xv = to_f(x[b * sB + h * sH + (int64_t)t * sT + lane]);
    const float r = rsq[v];
    const float tot = wave_sum(dn * xv * wv);
    dx[b * dB + h * dH + (int64_t)t * dT + lane] =
        from_f<T>(r * wv * dn - xv * r * r * r * tot * (1.0f / 64.0f));
    dwacc += dn * xv * r;
  }
  atomicAdd(&dw[h * 64 + lane], dwacc);
}

// The same with 8 lanes per vector and 8 elements per lane (lanes 0-3 of a group hold the
// first half, lanes 4-7 the second: a lane's rotate-half partners sit in lane ^ 4), two
// vectors of a group in flight. A workgroup's 32 groups serve one head; their dw partials
// meet in LDS. per_head below 2^31 and strides and pointers of whole 16-byte chunks. 8 x 2048
// tokens, 16 query heads and 4 key heads, bf16: 119 -> 40 us for both.
template <typename T>
__global__ void __launch_bounds__(256) qk_norm_rope_bwd_vec_kernel(
    const T* __restrict__ dy, const T* __restrict__ x, int64_t sB, int64_t sH, int64_t sT,
    int64_t dB, int64_t dH, int64_t dT, int H, int T_, int per_head,
    const float* __restrict__ w, const float* __restrict__ rsq, const float* __restrict__ cs,
    const float* __restrict__ sn, T* __restrict__ dx, float* __restrict__ dw) {
  __shared__ __attribute__((aligned(16))) float red[32][64];
  const int h = blockIdx.y, grp = threadIdx.x >> 3, j = threadIdx.x & 7;
  const float sgn = j < 4 ? 1.f : -1.f;
  float wv[8], acc[8];
  ldv<8>(w + h * 64 + j * 8, wv);
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  const int step = (int)gridDim.x * 32;
  constexpr int U = 2;
  // every group runs the same count of passes (lane exchanges inside); vectors past the end
  // re-read the last one and are neither stored nor summed
  for (int64_t i0 = (int64_t)blockIdx.x * 32; i0 < per_head; i0 += (int64_t)U * step) {
    float g[U][8], xv[U][8], c[U][8], s[U][8], r[U];
    int64_t out[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t iw = i0 + (int64_t)u * step + grp;
      ok[u] = iw < per_head;
      const int i = ok[u] ? (int)iw : per_head - 1;
      const int b = i / T_, t = i - b * T_;
      const int64_t v = ((int64_t)b * H + h) * T_ + t;
      out[u] = b * dB + h * dH + (int64_t)t * dT + j * 8;
      r[u] = rsq[v];
      ldv<8>(dy + v * 64 + j * 8, g[u]);
      ldv<8>(x + b * sB + h * sH + (int64_t)t * sT + j * 8, xv[u]);
      ldv<8>(cs + (int64_t)t * 32 + (j & 3) * 8, c[u]);
      ldv<8>(sn + (int64_t)t * 32 + (j & 3) * 8, s[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float dn[8], part = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float gp = __shfl_xor(g[u][e], 4, 64);
        dn[e] = g[u][e] * c[u][e] + sgn * (gp * s[u][e]);
        part += dn[e] * xv[u][e] * wv[e];
      }
      part += __shfl_xor(part, 1, 64);
      part += __shfl_xor(part, 2, 64);
      part += __shfl_xor(part, 4, 64);
      if (!ok[u]) continue;
      const float k = r[u] * r[u] * r[u] * part * (1.0f / 64.0f);
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        o[e] = r[u] * wv[e] * dn[e] - xv[u][e] * k;
        acc[e] += dn[e] * xv[u][e] * r[u];
      }
      stv<8>(dx + out[u], o);
    }
  }
  stv<8>(&red[grp][j * 8], acc);
  __syncthreads();
  if (threadIdx.x < 64) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 32; ++i) t += red[i][threadIdx.x];
    unsafeAtomicAdd(&dw[h * 64 + threadIdx.x], t);
  }
}

// ---------------------------------------------------------------------------
// Attention gate + transpose: out[b,t,h,d] = a[b,h,t,d] * sigmoid(l[b,t,h]). One wave per
// (b, t, h): d_a = grad * g ; d_l = sum_d(grad * a) * g * (1 - g).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) attn_gate_bwd_kernel(const T* __restrict__ go,
                                                            const T* __restrict__ a,
                                                            const float* __restrict__ gl,
                                                            T* __restrict__ da,
                                                            float* __restrict__ dl, int H,
                                                            int T_, int64_t nvec) {
  const int64_t hv = (int64_t)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
  if (hv >= nvec) return;
  const int lane = threadIdx.x & 63;
  const int h = (int)(hv % H);
  const int t = (int)((hv / H) % T_);
  const int64_t b = hv / ((int64_t)H * T_);
  const int64_t ai = ((b * H + h) * T_ + t) * 64 + lane;
  const float g = sigmoidf_(gl[hv]);
  const float gv = to_f(go[hv * 64 + lane]);
  const float dot = wave_sum(gv * to_f(a[ai]));
  da[ai] = from_f<T>(gv * g);
  if (lane == 0) dl[hv] = dot * g * (1.0f - g);
}

// The same with 8 lanes per (b, t, h) and 8 elements per lane (8 x 2048 tokens, 16 heads,
// bf16: 62 -> 24 us, 4.2 TB/s).
template <typename T>
__global__ void __launch_bounds__(256) attn_gate_bwd_vec_kernel(const T* __restrict__ go,
                                                                const T* __restrict__ a,
                                                                const float* __restrict__ gl,
                                                                T* __restrict__ da,
                                                                float* __restrict__ dl, int H,
                                                                int T_, int nvec) {
  const int64_t hw = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 3;
  const int j = threadIdx.x & 7;
  const bool ok = hw < nvec;
  const int hv = ok ? (int)hw : nvec - 1;
  const int bt = hv / H, h = hv - bt * H, b = bt / T_, t = bt - b * T_;
  const int64_t ai = (((int64_t)b * H + h) * T_ + t) * 64 + j * 8;
  float gv[8], av[8];
  ldv<8>(go + (int64_t)hv * 64 + j * 8, gv);
  ldv<8>(a + ai, av);
  const float g = sigmoidf_(gl[hv]);
  float dot = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    dot += gv[e] * av[e];
    gv[e] *= g;
  }
  dot += __shfl_xor(dot, 1, 64);
  dot += __shfl_xor(dot, 2, 64);
  dot += __shfl_xor(dot, 4, 64);
  if (!ok) return;
  stv<8>(da + ai, gv);
  if (j == 0) dl[hv] = dot * g * (1.0f - g);
}

// ---------------------------------------------------------------------------
// SwiGLU: out = silu(gate) * up with gu = [gate | up] per row.
//   d_gate = dout * up * s * (1 + gate * (1 - s)), s = sigmoid(gate) ; d_up = dout * silu(gate)
// ---------------------------------------------------------------------------
template <typename T>
__global__ void swiglu_bwd_kernel(const T* __restrict__ dout, const T* __restrict__ gu,
                                  T* __restrict__ dgu, int64_t d_ff, int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int64_t r = i / d_ff, c = i % d_ff;
  const float gt = to_f(gu[r * 2 * d_ff + c]), up = to_f(gu[r * 2 * d_ff + d_ff + c]);
  const float d = to_f(dout[i]);
  const float sg = sigmoidf_(gt);
  dgu[r * 2 * d_ff + c] = from_f<T>(d * up * sg * (1.0f + gt * (1.0f - sg)));
  dgu[r * 2 * d_ff + d_ff + c] = from_f<T>(d * gt * sg);
}

// The same on 16-byte chunks (32-bit indices: total below 2^31); at the copy rate: 81920 rows
// of 512 in bf16 116 -> 82 us (5.1 TB/s).
template <typename T>
__global__ void __launch_bounds__(256) swiglu_bwd_vec_kernel(const T* __restrict__ dout,
                                                             const T* __restrict__ gu,
                                                             T* __restrict__ dgu, uint32_t d_ff,
                                                             uint32_t total) {
  constexpr int V = kVec<T>;
  const uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) * V;
  if (i >= total) return;
  const uint32_t r = i / d_ff, c = i - r * d_ff;
  const int64_t at = (int64_t)r * 2 * d_ff + c;
  float gt[V], up[V], d[V], dg[V], du[V];
  ldv<V>(gu + at, gt);
  ldv<V>(gu + at + d_ff, up);
  ldv<V>(dout + i, d);
#pragma unroll
  for (int e = 0; e < V; ++e) {
    const float sg = sigmoidf_(gt[e]);
    dg[e] = d[e] * up[e] * sg * (1.0f + gt[e] * (1.0f - sg));
    du[e] = d[e] * gt[e] * sg;
  }
  stv<V>(dgu + at, dg);
  stv<V>(dgu + at + d_ff, du);
}

// Lane k < K: the row e_k C + slot_k of token t's k-th assignment in an [E, C, D] tensor,
// -1 for a dropped one (and for the other lanes). K <= 64 and E C below 2^31.
__device__ __forceinline__ int kept_row(const int64_t* idx, const int32_t* slots, int64_t t, int K,
                                        int64_t E, int64_t C, int lane) {
  if (lane >= K) return -1;
  const int64_t e = idx[t * K + lane];
  const int32_t sl = slots[t * K + lane];
  return e >= 0 && e < E && sl >= 0 && sl < C ? (int)(e * C + sl) : -1;
}

// ---------------------------------------------------------------------------
// MoE dispatch: expert_inputs[e, slot] = x[t] for every kept assignment (e, slot) of t.
//   dx[t] = sum over t's kept assignments, in top-k order, of d_expert_inputs[e, slot]
// ---------------------------------------------------------------------------
template <typename T>
__global__ void dispatch_bwd_kernel(const T* __restrict__ dei, const int64_t* __restrict__ idx,
                                    const int32_t* __restrict__ slots, T* __restrict__ dx,
                                    int64_t D, int K, int64_t E, int64_t C) {
  const int64_t t = blockIdx.x;
  for (int64_t d = threadIdx.x; d < D; d += blockDim.x) {
    float acc = 0.f;
    for (int k = 0; k < K; ++k) {
      const int64_t e = idx[t * K + k];
      const int32_t sl = slots[t * K + k];
      if (e >= 0 && e < E && sl >= 0 && sl < C) acc += to_f(dei[(e * C + sl) * D + d]);
    }
    dx[t * D + d] = from_f<T>(acc);
  }
}

// The same, one wave per token on 16-byte chunks: the token's K slots are read by lanes
// 0 .. K - 1 and broadcast, and four rows' chunks are loaded before the first is summed
// (16384 tokens of 1024, top-4, bf16: 102 -> 40 us, 4.2 TB/s).
template <typename T>
__global__ void __launch_bounds__(256) dispatch_bwd_vec_kernel(const T* __restrict__ dei,
                                                               const int64_t* __restrict__ idx,
                                                               const int32_t* __restrict__ slots,
                                                               T* __restrict__ dx, int64_t N,
                                                               int D, int K, int64_t E,
                                                               int64_t C) {
  constexpr int V = kVec<T>;
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= N) return;
  const int nrow = kept_row(idx, slots, t, K, E, C, lane);
  // every lane runs every pass, those past the row re-reading its last chunk: the broadcasts
  // below read lanes 0 .. K - 1, which a row of fewer chunks than K would have switched off
  for (int c0 = 0; c0 < D; c0 += 64 * V) {
    const int c = c0 + lane * V, cl = min(c, D - V);
    float acc[V];
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] = 0.f;
    for (int k0 = 0; k0 < K; k0 += 4) {
      uint4 r[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        // branch-free: dropped assignments read row 0 and count as zero
        const int at = k0 + q < K ? __builtin_amdgcn_readlane(nrow, k0 + q) : -1;
        r[q] = *reinterpret_cast<const uint4*>(dei + (int64_t)max(at, 0) * D + cl);
        if (at < 0) r[q] = make_uint4(0u, 0u, 0u, 0u);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v[V];
        unpackv<T>(r[q], v);
#pragma unroll
        for (int e = 0; e < V; ++e) acc[e] += v[e];
      }
    }
    if (c < D) stv<V>(dx + t * D + c, acc);
  }
}

// ---------------------------------------------------------------------------
// MoE combine: out[t] = shared[t] + sum_k w[t,k] * eo[e_k, slot_k] (kept assignments).
//   d_eo[e_k, slot_k] = w[t,k] * dout[t] ; d_w[t,k] = sum_d dout[t] * eo[e_k, slot_k]
//   (0 for dropped assignments; rows of d_eo no assignment names stay 0)
// One workgroup per token; the K dot products are reduced over the workgroup.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) combine_bwd_kernel(
    const T* __restrict__ dout, const T* __restrict__ eo, const int64_t* __restrict__ idx,
    const uint16_t* __restrict__ w_bf16, const int32_t* __restrict__ slots, T* __restrict__ deo,
    uint16_t* __restrict__ dw_bf16, int64_t D, int K, int64_t E, int64_t C) {
  __shared__ float red[16];
  const int64_t t = blockIdx.x;
  for (int k = 0; k < K; ++k) {
    const int64_t e = idx[t * K + k];
    const int32_t sl = slots[t * K + k];
    const bool kept = e >= 0 && e < E && sl >= 0 && sl < C;
    float part = 0.f;
    if (kept) {
      const float wk = bf2f(bf16{w_bf16[t * K + k]});
      const int64_t base = (e * C + sl) * D;
      for (int64_t d = threadIdx.x; d < D; d += blockDim.x) {
        const float g = to_f(dout[t * D + d]);
        part += g * to_f(eo[base + d]);
        deo[base + d] = from_f<T>(wk * g);
      }
    }
    const float dot = block_sum(part, red);
    if (threadIdx.x == 0) dw_bf16[t * K + k] = f2bf(kept ? dot : 0.f).u;
    __syncthreads();
  }
}

// The same, one wave per token on 16-byte chunks: no barriers, the token's gradient row read
// once (NC chunks a lane in registers) and the next expert row's loads out before this one's
// reduction. D % kVec == 0 and D <= 64 kVec NC. 16384 tokens of 1024, top-4, bf16: 132 ->
// 58 us, and the zero fill of d_expert_outputs 73 -> 22 us in 16-byte stores.
template <typename T, int NC>
__global__ void __launch_bounds__(256) combine_bwd_vec_kernel(
    const T* __restrict__ dout, const T* __restrict__ eo, const int64_t* __restrict__ idx,
    const uint16_t* __restrict__ w_bf16, const int32_t* __restrict__ slots, T* __restrict__ deo,
    uint16_t* __restrict__ dw_bf16, int64_t N, int D, int K, int64_t E, int64_t C) {
  constexpr int V = kVec<T>;
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= N) return;
  const int nrow = kept_row(idx, slots, t, K, E, C, lane);
  const float wl = bf2f(bf16{lane < K ? w_bf16[t * K + lane] : (uint16_t)0});
  // branch-free loads: lanes past the row re-read its last chunk and count as zero, dropped
  // assignments read row 0 and are not stored
  uint4 g[NC], row[2][NC];
  auto load = [&](const T* p, uint4* r) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int c = (lane + 64 * j) * V;
      r[j] = *reinterpret_cast<const uint4*>(p + min(c, D - V));
      if (c >= D) r[j] = make_uint4(0u, 0u, 0u, 0u);
    }
  };
  load(dout + t * D, g);
  auto fetch = [&](int k, uint4* r) {
    load(eo + (int64_t)max(__builtin_amdgcn_readlane(nrow, k), 0) * D, r);
  };
  fetch(0, row[0]);
  auto term = [&](int k, uint4* cur, uint4* nxt) {
    if (k + 1 < K) fetch(k + 1, nxt);
    const int at = __builtin_amdgcn_readlane(nrow, k);
    const float wk = lane_bcast(wl, k);
    float part = 0.f;
    T* dst = deo + (int64_t)max(at, 0) * D;
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      float gv[V], ev[V], o[V];
      unpackv<T>(g[j], gv);
      unpackv<T>(cur[j], ev);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        part += gv[e] * ev[e];
        o[e] = wk * gv[e];
      }
      const int c = (lane + 64 * j) * V;
      if (at >= 0 && c < D) stv<V>(dst + c, o);
    }
    const float dot = wave_sum(part);
    if (lane == 0) dw_bf16[t * K + k] = f2bf(at >= 0 ? dot : 0.f).u;
  };
  for (int k = 0; k < K; k += 2) {
    term(k, row[0], row[1]);
    if (k + 1 < K) term(k + 1, row[1], row[0]);
  }
}

// ---------------------------------------------------------------------------
// Router top-k. Forward: c = l - mean(l), s = sigmoid(c), top-k of s + bias (indices given),
// w_k = s_k / (sum_top s + 1e-6); z_loss = zw * mean_tokens(lse(c)^2); probs_mean =
// mean_tokens(s). Backward per token (one thread):
//   g_e = 2 zw dz lse(c) softmax(c)_e / N                      (z-loss)
//       + sum_k [e = e_k] (dw_k - sum_j dw_j w_j) s_k (1 - s_k) / (sum_top s + 1e-6)
//       + dpm_e s_e (1 - s_e) / N                               (probs_mean)
//   d_l = g - mean(g)                                           (centring)
// ---------------------------------------------------------------------------
// EM (16 or 32) >= E register slots in unrolled loops: every register-array index is a
// compile-time constant (runtime indices would move the arrays to scratch memory).
template <typename L, int EM>
__global__ void router_bwd_kernel(const uint16_t* __restrict__ dtw, const L* __restrict__ logits,
                                  const int64_t* __restrict__ idx, L* __restrict__ dl,
                                  float zw, const float* __restrict__ dz,
                                  const float* __restrict__ dpm, int64_t N, int E, int K) {
  const int64_t tok = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (tok >= N) return;
  float c[EM], s[EM], g[EM];
  float mean = 0.f;
#pragma unroll
  for (int e = 0; e < EM; ++e) {
    c[e] = e < E ? to_f(logits[tok * E + e]) : 0.f;
    if (e < E) mean += c[e];
  }
  mean /= (float)E;
  float mx = -INFINITY;
#pragma unroll
  for (int e = 0; e < EM; ++e) {
    c[e] -= mean;
    s[e] = sigmoidf_(c[e]);
    if (e < E) mx = fmaxf(mx, c[e]);
    g[e] = 0.f;
  }
  const float zeff = zw * (dz ? dz[0] : 1.0f);
  if (zeff > 0.f) {
    float se = 0.f;
#pragma unroll
    for (int e = 0; e < EM; ++e)
      if (e < E) se += expf(c[e] - mx);
    se = fmaxf(se, 1e-20f);
    const float lse = mx + logf(se);
    const float f = 2.0f * zeff * lse / (float)N;
#pragma unroll
    for (int e = 0; e < EM; ++e) g[e] = f * expf(c[e] - mx) / se;
  }
  float den = 1e-6f, sdu = 0.f;
  int ek[8];
  float d[8], us[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    ek[k] = -1;
    d[k] = us[k] = 0.f;
    if (k >= K) continue;
    ek[k] = (int)idx[tok * K + k];
    d[k] = bf2f(bf16{dtw[tok * K + k]});
    float u = 0.f;
#pragma unroll
    for (int e = 0; e < EM; ++e)
      if (e < E && e == ek[k]) u = s[e];
    us[k] = u;
    den += u;
    sdu += d[k] * u;
  }
  const float dbar = sdu / den;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (k >= K) continue;
    const float u = us[k];
    const float add = (d[k] - dbar) / den * u * (1.0f - u);
#pragma unroll
    for (int e = 0; e < EM; ++e)
      if (e < E && e == ek[k]) g[e] += add;
  }
  if (dpm) {
#pragma unroll
    for (int e = 0; e < EM; ++e)
      if (e < E) g[e] += dpm[e] / (float)N * s[e] * (1.0f - s[e]);
  }
  float gm = 0.f;
#pragma unroll
  for (int e = 0; e < EM; ++e)
    if (e < E) gm += g[e];
  gm /= (float)E;
#pragma unroll
  for (int e = 0; e < EM; ++e)
    if (e < E) dl[tok * E + e] = from_f<L>(g[e] - gm);
}

// ---------------------------------------------------------------------------
// Causal depthwise conv k=4 with residual: y_t = x_t + sum_k w[d,k] x_{t-k}.
//   dx_t = dout_t + sum_k w[d,k] dout_{t+k} (t + k < T) ;  dw[d,k] = sum_{b,t} dout_t x_{t-k}
// dw: a thread owns one channel of a chunk of tokens and adds its 4 sums once.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void conv_k4_bwd_dx_kernel(const T* __restrict__ dout, const float* __restrict__ w,
                                      T* __restrict__ dx, int64_t T_, int64_t D,
                                      int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int64_t d = i % D;
  const int64_t t = (i / D) % T_;
  float acc = to_f(dout[i]);
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (t + k < T_) acc += w[d * 4 + k] * to_f(dout[i + k * D]);
  dx[i] = from_f<T>(acc);
}

constexpr int kConvChunk = 256;  // tokens per workgroup row of the dw pass

template <typename T>
__global__ void conv_k4_bwd_dw_kernel(const T* __restrict__ dout, const T* __restrict__ x,
                                      float* __restrict__ dw, int64_t T_, int64_t D,
                                      int64_t ntok) {
  const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= D) return;
  const int64_t t0 = (int64_t)blockIdx.y * kConvChunk;
  const int64_t t1 = t0 + kConvChunk < ntok ? t0 + kConvChunk : ntok;
  float a[4] = {0.f, 0.f, 0.f, 0.f};
  for (int64_t n = t0; n < t1; ++n) {
    const int64_t t = n % T_;  // position within its sequence
    const float g = to_f(dout[n * D + d]);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (t >= k) a[k] += g * to_f(x[(n - k) * D + d]);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) atomicAdd(&dw[d * 4 + k], a[k]);
}

// Both gradients in one pass over dout and x, kVec channels per thread. A thread walks
// `groups` runs of kConvRun consecutive tokens of one sequence: the run's rows of x and of
// dout (3 rows ahead) are loaded before the first use, the 3 rows a run shares with the
// last one ride along in registers, and its 4 kVec dw sums stay there. A workgroup is 32
// channel chunks x 8 such tasks, whose dw sums meet in LDS. D % kVec == 0, 16-byte-aligned
// tensors. Two passes of 2-byte loads, the dw one a serial chain of 256 tokens per thread,
// took 98 + 173 us for 8 x 2048 tokens of 1024 in bf16 (15 + 134 us for 3 x 777 in fp32);
// this 24 us (9.9 us). Runs of 8 tokens take 252 registers, runs of 4 201.
constexpr int kConvRun = 4, kConvTasks = 8, kConvCols = 32;
template <typename T>
__global__ void __launch_bounds__(kConvCols* kConvTasks) conv_k4_bwd_vec_kernel(
    const T* __restrict__ dout, const T* __restrict__ x, const float* __restrict__ w,
    T* __restrict__ dx, float* __restrict__ dw, int64_t B, int64_t T_, int64_t D, int groups) {
  constexpr int V = kVec<T>, R = kConvRun;
  __shared__ __attribute__((aligned(16))) float red[kConvTasks][kConvCols * V * 4];
  const int tx = threadIdx.x % kConvCols, ty = threadIdx.x / kConvCols;
  const int64_t span = (int64_t)R * groups, ntask = (T_ + span - 1) / span;
  const int64_t task = (int64_t)blockIdx.y * kConvTasks + ty;
  const int64_t b = task / ntask, t_lo = (task - b * ntask) * span;
  const int64_t d0 = ((int64_t)blockIdx.x * kConvCols + tx) * V;
  float a[V][4];
#pragma unroll
  for (int e = 0; e < V; ++e) a[e][0] = a[e][1] = a[e][2] = a[e][3] = 0.f;
  if (b < B && d0 < D) {
    const T* xb = x + b * T_ * D + d0;
    const T* gb = dout + b * T_ * D + d0;
    T* ob = dx + b * T_ * D + d0;
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    auto row = [&](const T* p, int64_t t) {  // a row's chunk, zero outside the sequence
      const int64_t tc = t < 0 ? 0 : (t < T_ ? t : T_ - 1);
      const uint4 v = *reinterpret_cast<const uint4*>(p + tc * D);
      return t >= 0 && t < T_ ? v : zero;
    };
    float wd[4 * V];
    ldv<4 * V>(w + d0 * 4, wd);
    const int64_t t_hi = t_lo + span < T_ ? t_lo + span : T_;
    uint4 rx[R + 3], rg[R + 3];  // x rows t - 3 .. t + R - 1, dout rows t .. t + R + 2
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      rx[R + i] = row(xb, t_lo - 3 + i);
      rg[R + i] = row(gb, t_lo + i);
    }
    for (int64_t t = t_lo; t < t_hi; t += R) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        rx[i] = rx[R + i];
        rg[i] = rg[R + i];
      }
#pragma unroll
      for (int i = 0; i < R; ++i) {
        rx[3 + i] = row(xb, t + i);
        rg[3 + i] = row(gb, t + 3 + i);
      }
      // rings: dout rows t + i .. t + i + 3, x rows t + i - 3 .. t + i
      float gv[4][V], xv[4][V];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        unpackv<T>(rg[i], gv[i]);
        unpackv<T>(rx[i], xv[i]);
      }
      // a term whose other row lies outside the sequence is left out (not multiplied by
      // zero: its factor may be infinite); runs away from the ends need no test
      auto run = [&](auto edge) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
          unpackv<T>(rg[i + 3], gv[(i + 3) & 3]);
          unpackv<T>(rx[i + 3], xv[(i + 3) & 3]);
          if (decltype(edge)::value && t + i >= t_hi) break;
          float o[V];
#pragma unroll
          for (int e = 0; e < V; ++e) o[e] = gv[i & 3][e];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            if (!decltype(edge)::value || t + i + k < T_) {
#pragma unroll
              for (int e = 0; e < V; ++e) o[e] += wd[4 * e + k] * gv[(i + k) & 3][e];
            }
            if (!decltype(edge)::value || t + i >= k) {
#pragma unroll
              for (int e = 0; e < V; ++e) a[e][k] += gv[i & 3][e] * xv[(i + 3 - k) & 3][e];
            }
          }
          stv<V>(ob + (t + i) * D, o);
        }
      };
      if (t >= 3 && t + R + 3 <= T_)
        run(std::false_type{});
      else
        run(std::true_type{});
    }
  }
#pragma unroll
  for (int e = 0; e < V; ++e) stv<4>(&red[ty][(tx * V + e) * 4], a[e]);
  __syncthreads();
  const int64_t c0 = (int64_t)blockIdx.x * kConvCols * V * 4;
  for (int i = threadIdx.x; i < kConvCols * V * 4; i += kConvCols * kConvTasks) {
    float t = 0.f;
#pragma unroll
    for (int q = 0; q < kConvTasks; ++q) t += red[q][i];
    if (c0 + i < D * 4) unsafeAtomicAdd(&dw[c0 + i], t);
  }
}

}  // namespace

}  // namespace pulsar

using namespace pulsar;

extern "C" {

int pulsar_rmsnorm_backward(const void* dy, const void* x, const float* w, const float* rsqrt,
                            void* dx, float* dw, int64_t rows, int64_t dim, int dtype,
                            hipStream_t stream) {
  PULSAR_REQUIRE(rows >= 0 && dim > 0, "rmsnorm backward: rows >= 0 and dim > 0 required");
  PULSAR_REQUIRE(dim <= 256 * kNormCols, "rmsnorm backward supports dim <= 8192");
  PULSAR_TRY_STATUS(zero_f32(dw, dim, stream));
  if (rows == 0) return PULSAR_OK;
  PULSAR_REQUIRE(dy && x && w && rsqrt && dx && dw, "rmsnorm backward: null pointer");
  return dispatch_dtype(dtype, [&](auto tag) {
    using T = decltype(tag);
    constexpr int V = kVec<T>;
    if (dim % V == 0 && dim <= 2048 && aligned16(dy) && aligned16(x) && aligned16(w) &&
        aligned16(dx)) {
      constexpr int RPI = 2;
      const unsigned g = (unsigned)std::min<int64_t>(512, (rows + 4 * RPI - 1) / (4 * RPI));
      auto run = [&](auto nc) {
        rmsnorm_bwd_vec_kernel<T, decltype(nc)::value, RPI><<<g, 256, 0, stream>>>(
            (const T*)dy, (const T*)x, w, rsqrt, (T*)dx, dw, rows, (int)dim);
      };
      using std::integral_constant;
      if (dim <= 64 * V) run(integral_constant<int, 1>{});
      else if (dim <= 128 * V) run(integral_constant<int, 2>{});
      else if (dim <= 256 * V) run(integral_constant<int, 4>{});
      else if constexpr (V == 4) run(integral_constant<int, 8>{});
      PULSAR_LAUNCH_CHECK();
      return PULSAR_OK;
    }
    const unsigned grid = (unsigned)(rows < 1024 ? rows : 1024);
    rmsnorm_bwd_kernel<T><<<grid, 256, 0, stream>>>((const T*)dy, (const T*)x, w, rsqrt, (T*)dx,
                                                    dw, rows, (int)dim);
    PULSAR_LAUNCH_CHECK();
    return PULSAR_OK;
  });
}

int pulsar_qk_rmsnorm_rope_backward(const void* dy, const void* x, int64_t sB, int64_t sH,
                                    int64_t sT, void* dx, int64_t dB, int64_t dH, int64_t dT,
                                    int64_t B, int64_t H, int64_t T, int64_t head_dim,
                                    const float* w, const float* rsqrt, const float* cos,
                                    const float* sin, float* dw, int dtype,
                                    hipStream_t stream) {
  if (head_dim != 64)
    return fail(PULSAR_ERR_INVALID,
                "qk_rmsnorm_rope requires head_dim == 64, got " + std::to_string(head_dim));
  PULSAR_REQUIRE(B >= 0 && H > 0 && T > 0, "qk_rmsnorm_rope backward: bad shape");
  PULSAR_REQUIRE(H <= 65535, "qk_rmsnorm_rope backward: at most 65535 heads");
  PULSAR_TRY_STATUS(zero_f32(dw, H * 64, stream));
  const int64_t per_head = B * T;
  if (per_head == 0) return PULSAR_OK;
  // up to 64 workgroups (256 waves) per head; each wave adds its dw partial once
  const unsigned gx = (unsigned)std::min<int64_t>(64, (per_head + 3) / 4);
  return dispatch_dtype(dtype, [&](auto tag) {
    using T_ = decltype(tag);
    constexpr int V = kVec<T_>;
    if (sB % V == 0 && sH % V == 0 && sT % V == 0 && dB % V == 0 && dH % V == 0 && dT % V == 0 &&
        per_head < (int64_t)1 << 31 && aligned16(dy) && aligned16(x) && aligned16(dx) &&
        aligned16(w) && aligned16(cos) && aligned16(sin)) {
      // about 1024 workgroups over all heads, each of 32 vectors a pass
      const int64_t most = std::max<int64_t>(1, 1024 / H);
      const unsigned gv = (unsigned)std::min<int64_t>(most, (per_head + 31) / 32);
      qk_norm_rope_bwd_vec_kernel<T_><<<dim3(gv, (unsigned)H), 256, 0, stream>>>(
          (const T_*)dy, (const T_*)x, sB, sH, sT, dB, dH, dT, (int)H, (int)T, (int)per_head, w,
          rsqrt, cos, sin, (T_*)dx, dw);
      PULSAR_LAUNCH_CHECK();
      return PULSAR_OK;
    }
    qk_norm_rope_bwd_kernel<T_><<<dim3(gx, (unsigned)H), 256, 0, stream>>>(
        (const T_*)dy, (const T_*)x, sB, sH, sT, dB, dH, dT, (int)H, (int)T, per_head, w, rsqrt,
        cos, sin, (T_*)dx, dw);
    PULSAR_LAUNCH_CHECK();
    return PULSAR_OK;
  });
}

int pulsar_fused_attn_gate_backward(const void* grad_out, const void* attn,
                                    const float* gate_logits, void* d_attn, float* d_gate,
                                    int64_t B, int64_t H, int64_t T, int64_t head_dim,
                                    int dtype, hipStream_t stream) {
  if (head_dim != 64)
    return fail(PULSAR_ERR_INVALID,
                "fused_attn_gate requires head_dim == 64, got " + std::to_string(head_dim));
  const int64_t nvec = B * H * T;
  if (nvec == 0) return PULSAR_OK;
  return dispatch_dtype(dtype, [&](auto tag) {
    using T_ = decltype(tag);
    if (nvec < (int64_t)1 << 31 && aligned16(grad_out) && aligned16(attn) && aligned16(d_attn)) {
      attn_gate_bwd_vec_kernel<T_><<<blocks_for(nvec, 32), 256, 0, stream>>>(
          (const T_*)grad_out, (const T_*)attn, gate_logits, (T_*)d_attn, d_gate, (int)H, (int)T,
          (int)nvec);
      PULSAR_LAUNCH_CHECK();
      return PULSAR_OK;
    }
    attn_gate_bwd_kernel<T_><<<blocks_for(nvec, 4), 256, 0, stream>>>(
        (const T_*)grad_out, (const T_*)attn, gate_logits, (T_*)d_attn, d_gate, (int)H, (int)T,
        nvec);
    PULSAR_LAUNCH_CHECK();
    return PULSAR_OK;
  });
}

int pulsar_fused_swiglu_backward(const void* dout, const void* gu, void* dgu, int64_t rows,
                                 int64_t d_ff, int dtype, hipStream_t stream) {
  PULSAR_REQUIRE(rows >= 0 && d_ff > 0, "swiglu backward: bad shape");
  const int64_t total = rows * d_ff;
  if (total == 0) return PULSAR_OK;
  return dispatch_dtype(dtype, [&](auto tag) {
    using T_ = decltype(tag);
    constexpr int V = kVec<T_>;
    if (d_ff % V == 0 && total < (int64_t)1 << 31 && aligned16(dout) && aligned16(gu) &&
        aligned16(dgu)) {
      swiglu_bwd_vec_kernel<T_><<<blocks_for(total / V, 256), 256, 0, stream>>>(
          (const T_*)dout, (const T_*)gu, (T_*)dgu, (uint32_t)d_ff, (uint32_t)total);
      PULSAR_LAUNCH_CHECK();
      return PULSAR_OK;
    }
    swiglu_bwd_kernel<T_><<<blocks_for(total, 256), 256, 0, stream>>>(
        (const T_*)dout, (const T_*)gu, (T_*)dgu, d_ff, total);
    PULSAR_LAUNCH_CHECK();
    return PULSAR_OK;
  });
}

int pulsar_moe_dispatch_backward(const void* d_expert_inputs, const int64_t* topk_idx,
                                 const int32_t* slots, void* dx, int64_t N, int64_t D,
                                 int64_t K, int64_t E, int64_t C, int dtype,
                                 hipStream_t stream) {
  PULSAR_REQUIRE(N >= 0 && D > 0 && K >= 0 && E > 0 && C >= 0, "dispatch backward: bad shape");
  if (N == 0) return PULSAR_OK;
  return dispatch_dtype(dtype, [&](auto tag) {
    using T_ = decltype(tag);
    if (D % kVec<T_> == 0 && D < (int64_t)1 << 30 && K <= 64 && E * C > 0 && E * C < (int64_t)1 << 31 &&
        aligned16(d_expert_inputs) && aligned16(dx)) {
      dispatch_bwd_vec_kernel<T_><<<blocks_for(N, 4), 256, 0, stream>>>(
          (const T_*)d_expert_inputs, topk_idx, slots, (T_*)dx, N, (int)D, (int)K, E, C);
      PULSAR_LAUNCH_CHECK();
      return PULSAR_OK;
    }
    dispatch_bwd_kernel<T_><<<(unsigned)N, 128, 0, stream>>>(
        (const T_*)d_expert_inputs, topk_idx, slots, (T_*)dx, D, (int)K, E, C);
    PULSAR_LAUNCH_CHECK();
    return PULSAR_OK;
  });
}

int pulsar_moe_combine_backward(const void* d_routed_out, const void* expert_outputs,
                                const int64_t* topk_idx, const uint16_t* topk_w_bf16,
                                const int32_t* slots, void* d_expert_outputs,
                                uint16_t* d_topk_w_bf16, int64_t N, int64_t D, int64_t K,
                                int64_t E, int64_t C, int dtype, hipStream_t stream) {
  PULSAR_REQUIRE(N >= 0 && D > 0 && K >= 0 && E > 0 && C >= 0, "combine backward: bad shape");
  return dispatch_dtype(dtype, [&](auto tag) {
    using T_ = decltype(tag);
    const int64_t n_eo = E * C * D;
    constexpr int V = kVec<T_>;
    const bool vec = D % V == 0 && D <= 256 * V && K <= 64 && n_eo > 0 &&
                     E * C < (int64_t)1 << 31 &&
                     aligned16(d_routed_out) && aligned16(expert_outputs) &&
                     aligned16(d_expert_outputs);
    if (n_eo > 0 && vec) {
      fill_zero_vec_kernel<<<blocks_for(n_eo / V, 1024), 256, 0, stream>>>(
          (uint4*)d_expert_outputs, n_eo / V);
      PULSAR_LAUNCH_CHECK();
    } else if (n_eo > 0) {
      fill_zero_kernel<T_><<<blocks_for(n_eo, 256), 256, 0, stream>>>((T_*)d_expert_outputs, n_eo);
      PULSAR_LAUNCH_CHECK();
    }
    if (N > 0 && K > 0 && vec) {
      auto run = [&](auto nc) {
        combine_bwd_vec_kernel<T_, decltype(nc)::value><<<blocks_for(N, 4), 256, 0, stream>>>(
            (const T_*)d_routed_out, (const T_*)expert_outputs, topk_idx, topk_w_bf16, slots,
            (T_*)d_expert_outputs, d_topk_w_bf16, N, (int)D, (int)K, E, C);
      };
      if (D <= 64 * V) run(std::integral_constant<int, 1>{});
      else if (D <= 128 * V) run(std::integral_constant<int, 2>{});
      else run(std::integral_constant<int, 4>{});
      PULSAR_LAUNCH_CHECK();
    } else if (N > 0 && K > 0) {
      combine_bwd_kernel<T_><<<(unsigned)N, 256, 0, stream>>>(
          (const T_*)d_routed_out, (const T_*)expert_outputs, topk_idx, topk_w_bf16, slots,
          (T_*)d_expert_outputs, d_topk_w_bf16, D, (int)K, E, C);
      PULSAR_LAUNCH_CHECK();
    }
    return PULSAR_OK;
  });
}

int pulsar_moe_router_topk_backward(const uint16_t* d_topk_w_bf16, const void* logits,
                                    int logits_dtype, const int64_t* topk_idx,
                                    float z_loss_weight, const float* d_z_loss,
                                    const float* d_probs_mean, void* d_logits, int64_t N,
                                    int64_t E, int64_t K, hipStream_t stream) {
  if (E < 1 || E > 32)
    return fail(PULSAR_ERR_INVALID,
                "moe_router_topk_backward supports E <= 32, got " + std::to_string(E));
  if (K < 1 || K > 8 || K > E)
    return fail(PULSAR_ERR_INVALID, "top_k must be in [1, min(8, E)], got " + std::to_string(K));
  PULSAR_REQUIRE(N >= 0, "router backward: N must be >= 0");
  if (N == 0) return PULSAR_OK;
  return dispatch_dtype(logits_dtype, [&](auto tag) {
    using L = decltype(tag);
    if (E <= 16)
      router_bwd_kernel<L, 16><<<blocks_for(N, 128), 128, 0, stream>>>(
          d_topk_w_bf16, (const L*)logits, topk_idx, (L*)d_logits, z_loss_weight, d_z_loss,
          d_probs_mean, N, (int)E, (int)K);
    else
      router_bwd_kernel<L, 32><<<blocks_for(N, 128), 128, 0, stream>>>(
          d_topk_w_bf16, (const L*)logits, topk_idx, (L*)d_logits, z_loss_weight, d_z_loss,
          d_probs_mean, N, (int)E, (int)K);
    PULSAR_LAUNCH_CHECK();
    return PULSAR_OK;
  });
}

int pulsar_causal_conv1d_k4_backward(const void* dout, const void* x, const float* w, void* dx,
                                     float* dw, int64_t B, int64_t T, int64_t D, int dtype,
                                     hipStream_t stream) {
  PULSAR_REQUIRE(B >= 0 && T >= 0 && D > 0, "conv1d_k4 backward: bad shape");
  PULSAR_TRY_STATUS(zero_f32(dw, D * 4, stream));
  const int64_t ntok = B * T, total = ntok * D;
  if (total == 0) return PULSAR_OK;
  return dispatch_dtype(dtype, [&](auto tag) {
    using T_ = decltype(tag);
    constexpr int V = kVec<T_>;
    if (D % V == 0 && aligned16(dout) && aligned16(x) && aligned16(w) && aligned16(dx)) {
      // the longest tasks that leave two workgroups for every CU: each workgroup adds its
      // columns' dw once
      const int64_t gx = (D / V + kConvCols - 1) / kConvCols;
      auto rows_y = [&](int g) {
        const int64_t span = (int64_t)kConvRun * g;
        return (B * ((T + span - 1) / span) + kConvTasks - 1) / kConvTasks;
      };
      int groups = 8;
      while (groups > 1 && gx * rows_y(groups) < 512) groups /= 2;
      const int64_t gy = rows_y(groups);
      if (gy <= 65535) {
        conv_k4_bwd_vec_kernel<T_><<<dim3((unsigned)gx, (unsigned)gy), kConvCols * kConvTasks, 0,
                                     stream>>>((const T_*)dout, (const T_*)x, w, (T_*)dx, dw, B, T,
                                               D, groups);
        PULSAR_LAUNCH_CHECK();
        return PULSAR_OK;
      }
    }
    conv_k4_bwd_dx_kernel<T_><<<blocks_for(total, 256), 256, 0, stream>>>(
        (const T_*)dout, w, (T_*)dx, T, D, total);
    PULSAR_LAUNCH_CHECK();
    const dim3 g(blocks_for(D, 256), blocks_for(ntok, kConvChunk));
    conv_k4_bwd_dw_kernel<T_><<<g, 256, 0, stream>>>((const T_*)dout, (const T_*)x, dw, T, D,
                                                      ntok);
    PULSAR_LAUNCH_CHECK();
    return PULSAR_OK;
  });
}

}  // extern "C"

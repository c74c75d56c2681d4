// Device helpers shared by the row-set GEMMs (gemm.hip, gemm_wide.hip): row sets and
// epilogues.
#pragma once

#include "engine.h"

namespace pulsar {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));


constexpr int kXcds = 8;  // MI355X: consecutive workgroups go to the 8 XCDs in turn

// One output. pre: the residual value (EPI_RESID) or the gate column's bias (EPI_QKVG), loaded
// by the caller.
template <typename T>
__device__ __forceinline__ void epilogue(const GemmArgs& g, int epi, int group, void* Cv,
                                         int64_t ldc, int crow, int col, float acc, float acc_up,
                                         float pre) {
  T* C = reinterpret_cast<T*>(Cv);
  switch (epi) {
    case EPI_STORE:
      C[(int64_t)crow * ldc + col] = from_f<T>(acc);
      break;
    case EPI_QKVG:
      if (col < g.n_main) {
        C[(int64_t)crow * ldc + col] = from_f<T>(acc);
      } else {
        const float v = rnd<T>(acc + pre);
        reinterpret_cast<T*>(g.C2)[(int64_t)crow * g.ldc2 + col - g.n_main] = from_f<T>(sigmoidf_(v));
      }
      break;
    case EPI_RESID:
      C[(int64_t)crow * ldc + col] = from_f<T>(pre + rnd<T>(acc));
      break;
    case EPI_SWIGLU: {
      const float gt = rnd<T>(acc), up = rnd<T>(acc_up);
      C[(int64_t)crow * ldc + col] = from_f<T>(gt * sigmoidf_(gt) * up);
      break;
    }
    case EPI_LOGITS: {
      float l = rnd<T>(acc);
      if (g.softcap > 0.f) {
        float t = rnd<T>(l / g.softcap);
        t = rnd<T>(tanhf(t));
        l = rnd<T>(g.softcap * t);
      }
      reinterpret_cast<float*>(Cv)[(int64_t)crow * ldc + col] = l;
      break;
    }
    case EPI_LOGITS_RAW:
      reinterpret_cast<float*>(Cv)[(int64_t)crow * ldc + col] = rnd<T>(acc);
      break;
    case EPI_SCALE: {
      const T* s = reinterpret_cast<const T*>(g.bias);
      C[(int64_t)crow * ldc + col] = from_f<T>(rnd<T>(acc) * to_f(s[col]));
      break;
    }
  }
}

// Entry i of the group: the row index (pulse / all / logits modes) or the assignment id
// (list mode; the all-rows group -1 of a fused launch takes row i). Branch-free in the row
// mode, which is a template parameter: a load pending on one path of a runtime switch
// would make the join wait for every load in flight, weights included.
template <int MODE>
__device__ __forceinline__ int entry_load(const GemmArgs& g, int group, int i) {
  if constexpr (MODE == ROWS_PULSE) return g.ctl->pulse_start[group] + i;
  if constexpr (MODE == ROWS_LIST) return g.list[(int64_t)max(group, 0) * g.list_stride + i];
  return i;
}
// Applied after the weight loads are issued (the only use of the loaded value).
template <int MODE>
__device__ __forceinline__ int entry_fix(int group, int i, int v) {
  if constexpr (MODE == ROWS_LIST) return group < 0 ? i : v;
  return v;
}
template <int MODE>
__device__ __forceinline__ int a_row_of(const GemmArgs& g, int group, int raw) {
  if constexpr (MODE == ROWS_LIST) {
    if (group < 0) return raw;
    // a_div is 1 (expert output rows) or the top-k count (token rows). A power of two takes
    // a shift instead of the ~30-instruction integer division; entries are non-negative
    // (only the spare-capacity entries of eager launches may not be, and their rows are
    // clamped, computed and never stored).
    const int d = g.a_div;
    if ((d & (d - 1)) == 0) return raw >> __builtin_ctz((unsigned)d);
    return raw / d;
  }
  return raw;
}
template <int MODE>
__device__ __forceinline__ int group_rows(const GemmArgs& g, int group) {
  if constexpr (MODE == ROWS_PULSE) return g.ctl->pulse_count[group];
  if constexpr (MODE == ROWS_LOGITS) return g.ctl->n_lrows;
  if constexpr (MODE == ROWS_LIST) {
    // the fused all-rows group (-1) exists only in launches with a step control block
    return group >= 0 ? g.list_count[group * kCountStride] : g.ctl->n_rows;
  }
  return g.ctl ? g.ctl->n_rows : g.m_fixed;
}

// Four consecutive output columns of one row (col0 % 4 == 0, never straddling n_main). pre:
// the row's residual values (EPI_RESID) or the columns' scales (EPI_SCALE), loaded before.
__device__ __forceinline__ void epilogue4(const GemmArgs& g, int epi, int group, void* Cv,
                                          int64_t ldc, int crow, int col0, const float* v,
                                          const float* u, const bf16x4_t& pre) {
  bf16* C = reinterpret_cast<bf16*>(Cv);
  bf16x4_t o;
  switch (epi) {
    case EPI_STORE:
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = (__bf16)v[j];
      break;
    case EPI_RESID: {
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = (__bf16)((float)pre[j] + rnd<bf16>(v[j]));
      break;
    }
    case EPI_SWIGLU:
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float gt = rnd<bf16>(v[j]), up = rnd<bf16>(u[j]);
        o[j] = (__bf16)(gt * sigmoidf_(gt) * up);
      }
      break;
    case EPI_SCALE: {
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = (__bf16)(rnd<bf16>(v[j]) * (float)pre[j]);
      break;
    }
    case EPI_LOGITS:
    case EPI_LOGITS_RAW: {
      // fp32 store of bf16-rounded logits, softcapped with the scalar epilogue's roundings
      float4 lv;
      float* lp = &lv.x;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float l = rnd<bf16>(v[j]);
        if (epi == EPI_LOGITS && g.softcap > 0.f) {
          float t = rnd<bf16>(l / g.softcap);
          t = rnd<bf16>(tanhf(t));
          l = rnd<bf16>(g.softcap * t);
        }
        lp[j] = l;
      }
      *reinterpret_cast<float4*>(reinterpret_cast<float*>(Cv) + (int64_t)crow * ldc + col0) = lv;
      return;
    }
    default:  // EPI_QKVG: q/k/v columns stored, gate columns through the scalar epilogue
      if (col0 >= g.n_main) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          epilogue<bf16>(g, epi, group, Cv, ldc, crow, col0 + j, v[j], 0.f,
                         to_f(reinterpret_cast<const bf16*>(
                             g.bias)[(int64_t)group * g.bias_group_stride + col0 + j - g.n_main]));
        return;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = (__bf16)v[j];
      break;
  }
  *reinterpret_cast<bf16x4_t*>(C + (int64_t)crow * ldc + col0) = o;
}

}  // namespace pulsar

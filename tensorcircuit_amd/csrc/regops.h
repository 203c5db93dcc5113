// Gates and gradient generators on 2^R amplitudes held in registers, shared by
// the per-gate kernels (kernels.hip) and the table-driven tile passes
// (tile_pass.hip), and the tile offsets and row sums that the Pauli kernels use
// as well.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.h"

namespace tcm {

// An amplitude in registers.  A plain pair: float2 is a vector type to the
// compiler, and arrays of vectors changed in the branches of an op switch cost
// 16 to 48 register moves per op and spill.
template <typename T>
struct alignas(2 * sizeof(T)) A2 {
  T x, y;
};
template <typename T>
__device__ __forceinline__ A2<T> ma(T a, T b) { return A2<T>{a, b}; }
// Im(conj(a) b), Re(conj(a) b)
template <typename T>
__device__ __forceinline__ T imcj(A2<T> a, A2<T> b) { return a.x * b.y - a.y * b.x; }
template <typename T>
__device__ __forceinline__ T recj(A2<T> a, A2<T> b) { return a.x * b.x + a.y * b.y; }

template <typename T>
__device__ __forceinline__ const T* mptr(int moff, const T* mt, const T* ct) {
  return moff >= 0 ? mt + moff : ct + (-moff - 1);
}

// state offset of tile position x from its block's base: the L low tile bits
// are contiguous, the others' runs are at ro (linear over disjoint bit sets)
__device__ __forceinline__ uint32_t run_dep(const uint32_t* __restrict__ ro, int L, uint32_t x) {
  return ro[x >> L] + (x & ((1u << L) - 1));
}

// one DPP row-shift of a double (lanes without a source read 0)
template <int CTRL>
__device__ __forceinline__ double dpp_shr(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double read_lane(double x, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                          __builtin_amdgcn_readlane(__double2loint(x), lane));
}
// fp64 sum over a full 64-lane wave, uniform result: inclusive row prefix
// sums by DPP row_shr 1/2/4/8 leave each 16-lane row's total in its last
// lane; the four row totals are read back as scalars.
__device__ __forceinline__ double wave_sum_dpp(double x) {
  x += dpp_shr<0x111>(x);
  x += dpp_shr<0x112>(x);
  x += dpp_shr<0x114>(x);
  x += dpp_shr<0x118>(x);
  return (read_lane(x, 15) + read_lane(x, 31)) + (read_lane(x, 47) + read_lane(x, 63));
}

// ---------------------------------------------------------------------------
// slot dispatch: runtime register slot -> compile-time template argument.
// Plain switches (no lambdas capturing the register array) so that the
// per-thread amplitude array stays in VGPRs.
// ---------------------------------------------------------------------------
#define TCM_SW1(R, s, ...)                                          \
  switch (s) {                                                      \
    case 0: { constexpr int S_ = 0; __VA_ARGS__; } break;           \
    case 1: if constexpr (R > 1) { constexpr int S_ = 1; __VA_ARGS__; } break; \
    case 2: if constexpr (R > 2) { constexpr int S_ = 2; __VA_ARGS__; } break; \
    case 3: if constexpr (R > 3) { constexpr int S_ = 3; __VA_ARGS__; } break; \
    case 4: if constexpr (R > 4) { constexpr int S_ = 4; __VA_ARGS__; } break; \
    default: break;                                                 \
  }

#define TCM_SW2B(R, A_, s1, ...)                                                         \
  switch (s1) {                                                                          \
    case 0: if constexpr (A_ != 0) { constexpr int B_ = 0; __VA_ARGS__; } break;         \
    case 1: if constexpr (R > 1 && A_ != 1) { constexpr int B_ = 1; __VA_ARGS__; } break; \
    case 2: if constexpr (R > 2 && A_ != 2) { constexpr int B_ = 2; __VA_ARGS__; } break; \
    case 3: if constexpr (R > 3 && A_ != 3) { constexpr int B_ = 3; __VA_ARGS__; } break; \
    case 4: if constexpr (R > 4 && A_ != 4) { constexpr int B_ = 4; __VA_ARGS__; } break; \
    default: break;                                                                      \
  }

#define TCM_SW2(R, s0, s1, ...)                                                           \
  switch (s0) {                                                                           \
    case 0: { constexpr int A_ = 0; TCM_SW2B(R, A_, s1, __VA_ARGS__) } break;             \
    case 1: if constexpr (R > 1) { constexpr int A_ = 1; TCM_SW2B(R, A_, s1, __VA_ARGS__) } break; \
    case 2: if constexpr (R > 2) { constexpr int A_ = 2; TCM_SW2B(R, A_, s1, __VA_ARGS__) } break; \
    case 3: if constexpr (R > 3) { constexpr int A_ = 3; TCM_SW2B(R, A_, s1, __VA_ARGS__) } break; \
    case 4: if constexpr (R > 4) { constexpr int A_ = 4; TCM_SW2B(R, A_, s1, __VA_ARGS__) } break; \
    default: break;                                                                       \
  }

// ---------------------------------------------------------------------------
// in-register gate application on v[0 .. 2^R): register index bit S <-> the
// gate qubit.  DAG applies U^dagger.
// ---------------------------------------------------------------------------
template <typename T, int R, int S, bool DAG>
__device__ __forceinline__ void ap_u1(A2<T>* v, const T* m) {
  T ar = m[0], ai = m[1], br = m[2], bi = m[3], cr = m[4], ci = m[5], dr = m[6], di = m[7];
  if constexpr (DAG) {
    T tr = br, ti = bi;
    br = cr; bi = -ci;
    cr = tr; ci = -ti;
    ai = -ai; di = -di;
  }
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    if (j & (1 << S)) continue;
    A2<T> x = v[j], y = v[j | (1 << S)];
    v[j] = ma<T>(ar * x.x - ai * x.y + br * y.x - bi * y.y, ar * x.y + ai * x.x + br * y.y + bi * y.x);
    v[j | (1 << S)] = ma<T>(cr * x.x - ci * x.y + dr * y.x - di * y.y, cr * x.y + ci * x.x + dr * y.y + di * y.x);
  }
}

template <typename T, int R, int S, bool DAG>
__device__ __forceinline__ void ap_r1(A2<T>* v, const T* m) {
  T a = m[0], b = m[1], c = m[2], d = m[3];
  if constexpr (DAG) {
    T t = b; b = c; c = t;
  }
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    if (j & (1 << S)) continue;
    A2<T> x = v[j], y = v[j | (1 << S)];
    v[j] = ma<T>(a * x.x + b * y.x, a * x.y + b * y.y);
    v[j | (1 << S)] = ma<T>(c * x.x + d * y.x, c * x.y + d * y.y);
  }
}

template <typename T, int R, int S, bool DAG>
__device__ __forceinline__ void ap_d1(A2<T>* v, const T* m) {
  T d0r = m[0], d0i = m[1], d1r = m[2], d1i = m[3];
  if constexpr (DAG) { d0i = -d0i; d1i = -d1i; }
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    A2<T> x = v[j];
    if (j & (1 << S)) v[j] = ma<T>(d1r * x.x - d1i * x.y, d1r * x.y + d1i * x.x);
    else v[j] = ma<T>(d0r * x.x - d0i * x.y, d0r * x.y + d0i * x.x);
  }
}

template <typename T, int R, int S>
__device__ __forceinline__ void ap_x1(A2<T>* v) {
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    if (j & (1 << S)) continue;
    A2<T> t = v[j];
    v[j] = v[j | (1 << S)];
    v[j | (1 << S)] = t;
  }
}

// 2-qubit: matrix index r = (bit S0) << 1 | (bit S1)
template <typename T, int R, int S0, int S1, bool DAG>
__device__ __forceinline__ void ap_u2(A2<T>* v, const T* m) {
  T mr[16], mi[16];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if constexpr (DAG) {
        mr[r * 4 + c] = m[2 * (c * 4 + r)];
        mi[r * 4 + c] = -m[2 * (c * 4 + r) + 1];
      } else {
        mr[r * 4 + c] = m[2 * (r * 4 + c)];
        mi[r * 4 + c] = m[2 * (r * 4 + c) + 1];
      }
    }
  constexpr int m0 = 1 << S0, m1 = 1 << S1;
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    if (j & (m0 | m1)) continue;
    const int idx[4] = {j, j | m1, j | m0, j | m0 | m1};
    A2<T> x[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) x[c] = v[idx[c]];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      T sr = 0, si = 0;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        sr += mr[r * 4 + c] * x[c].x - mi[r * 4 + c] * x[c].y;
        si += mr[r * 4 + c] * x[c].y + mi[r * 4 + c] * x[c].x;
      }
      v[idx[r]] = ma<T>(sr, si);
    }
  }
}

template <typename T, int R, int S0, int S1, bool DAG>
__device__ __forceinline__ void ap_d2(A2<T>* v, const T* m) {
  T dr[4], di[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    dr[r] = m[2 * r];
    di[r] = DAG ? -m[2 * r + 1] : m[2 * r + 1];
  }
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    const int r = (((j >> S0) & 1) << 1) | ((j >> S1) & 1);
    A2<T> x = v[j];
    v[j] = ma<T>(dr[r] * x.x - di[r] * x.y, dr[r] * x.y + di[r] * x.x);
  }
}

template <typename T, int R, int S0, int S1>
__device__ __forceinline__ void ap_cx(A2<T>* v) {
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    if (!(j & (1 << S0)) || (j & (1 << S1))) continue;
    A2<T> t = v[j];
    v[j] = v[j | (1 << S1)];
    v[j | (1 << S1)] = t;
  }
}

template <typename T, int R, int S0, int S1>
__device__ __forceinline__ void ap_cz(A2<T>* v) {
#pragma unroll
  for (int j = 0; j < (1 << R); ++j)
    if ((j & (1 << S0)) && (j & (1 << S1))) v[j] = ma<T>(-v[j].x, -v[j].y);
}

template <typename T, int R, int S0, int S1>
__device__ __forceinline__ void ap_swap(A2<T>* v) {
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    if (!(j & (1 << S0)) || (j & (1 << S1))) continue;
    const int jj = (j ^ (1 << S0)) | (1 << S1);
    A2<T> t = v[j];
    v[j] = v[jj];
    v[jj] = t;
  }
}

// apply one op (kinds with a register form) on v
template <typename T, int R, bool DAG>
__device__ __forceinline__ void apply_op(A2<T>* v, const DOp& op, const T* mt, const T* ct) {
  switch (op.kind) {
    case OK_U1: {
      const T* m = mptr<T>(op.moff, mt, ct);
      TCM_SW1(R, op.s0, ap_u1<T, R, S_, DAG>(v, m))
    } break;
    case OK_R1: {
      const T* m = mptr<T>(op.moff, mt, ct);
      TCM_SW1(R, op.s0, ap_r1<T, R, S_, DAG>(v, m))
    } break;
    case OK_D1: {
      const T* m = mptr<T>(op.moff, mt, ct);
      TCM_SW1(R, op.s0, ap_d1<T, R, S_, DAG>(v, m))
    } break;
    case OK_X1:
      TCM_SW1(R, op.s0, ap_x1<T, R, S_>(v))
      break;
    case OK_U2: {
      const T* m = mptr<T>(op.moff, mt, ct);
      TCM_SW2(R, op.s0, op.s1, ap_u2<T, R, A_, B_, DAG>(v, m))
    } break;
    case OK_D2: {
      const T* m = mptr<T>(op.moff, mt, ct);
      TCM_SW2(R, op.s0, op.s1, ap_d2<T, R, A_, B_, DAG>(v, m))
    } break;
    case OK_CX:
      TCM_SW2(R, op.s0, op.s1, ap_cx<T, R, A_, B_>(v))
      break;
    case OK_CZ:
      TCM_SW2(R, op.s0, op.s1, ap_cz<T, R, A_, B_>(v))
      break;
    case OK_SWAP:
      TCM_SW2(R, op.s0, op.s1, ap_swap<T, R, A_, B_>(v))
      break;
    default:
      break;
  }
}

// ---------------------------------------------------------------------------
// gradient kernels on registers: Im <l | G | p> summed over the thread's
// amplitudes (p = psi after the gate, l = lambda after the gate)
// ---------------------------------------------------------------------------
template <typename T, int R, int S>
__device__ __forceinline__ T g_x(const A2<T>* p, const A2<T>* l) {
  T a = 0;
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    if (j & (1 << S)) continue;
    const int jj = j | (1 << S);
    a += imcj<T>(l[j], p[jj]) + imcj<T>(l[jj], p[j]);
  }
  return a;
}
template <typename T, int R, int S>
__device__ __forceinline__ T g_y(const A2<T>* p, const A2<T>* l) {
  T a = 0;
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    if (j & (1 << S)) continue;
    const int jj = j | (1 << S);
    a += recj<T>(l[jj], p[j]) - recj<T>(l[j], p[jj]);
  }
  return a;
}
template <typename T, int R, int S>
__device__ __forceinline__ T g_z(const A2<T>* p, const A2<T>* l) {
  T a = 0;
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    T t = imcj<T>(l[j], p[j]);
    a += (j & (1 << S)) ? -t : t;
  }
  return a;
}
template <typename T, int R, int S>
__device__ __forceinline__ T g_p1(const A2<T>* p, const A2<T>* l) {
  T a = 0;
#pragma unroll
  for (int j = 0; j < (1 << R); ++j)
    if (j & (1 << S)) a += imcj<T>(l[j], p[j]);
  return a;
}
template <typename T, int R, int S0, int S1>
__device__ __forceinline__ T g_xx(const A2<T>* p, const A2<T>* l) {
  T a = 0;
  constexpr int m = (1 << S0) | (1 << S1);
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) a += imcj<T>(l[j], p[j ^ m]);
  return a;
}
template <typename T, int R, int S0, int S1>
__device__ __forceinline__ T g_yy(const A2<T>* p, const A2<T>* l) {
  T a = 0;
  constexpr int m = (1 << S0) | (1 << S1);
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    T t = imcj<T>(l[j], p[j ^ m]);
    const int par = ((j >> S0) ^ (j >> S1)) & 1;
    a += par ? t : -t;
  }
  return a;
}
template <typename T, int R, int S0, int S1>
__device__ __forceinline__ T g_zz(const A2<T>* p, const A2<T>* l) {
  T a = 0;
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    T t = imcj<T>(l[j], p[j]);
    const int par = ((j >> S0) ^ (j >> S1)) & 1;
    a += par ? -t : t;
  }
  return a;
}
// general Hermitian generator, 2x2 (U1 layout) on slot S
template <typename T, int R, int S>
__device__ __forceinline__ T g_m1(const A2<T>* p, const A2<T>* l, const T* g) {
  T a = 0;
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    if (j & (1 << S)) continue;
    const int jj = j | (1 << S);
    A2<T> x = p[j], y = p[jj];
    A2<T> u = ma<T>(g[0] * x.x - g[1] * x.y + g[2] * y.x - g[3] * y.y, g[0] * x.y + g[1] * x.x + g[2] * y.y + g[3] * y.x);
    A2<T> w = ma<T>(g[4] * x.x - g[5] * x.y + g[6] * y.x - g[7] * y.y, g[4] * x.y + g[5] * x.x + g[6] * y.y + g[7] * y.x);
    a += imcj<T>(l[j], u) + imcj<T>(l[jj], w);
  }
  return a;
}
template <typename T, int R, int S0, int S1>
__device__ __forceinline__ T g_m2(const A2<T>* p, const A2<T>* l, const T* g) {
  T a = 0;
  constexpr int m0 = 1 << S0, m1 = 1 << S1;
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) {
    if (j & (m0 | m1)) continue;
    const int idx[4] = {j, j | m1, j | m0, j | m0 | m1};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      T sr = 0, si = 0;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const T gr = g[2 * (r * 4 + c)], gi = g[2 * (r * 4 + c) + 1];
        sr += gr * p[idx[c]].x - gi * p[idx[c]].y;
        si += gr * p[idx[c]].y + gi * p[idx[c]].x;
      }
      a += imcj<T>(l[idx[r]], ma<T>(sr, si));
    }
  }
  return a;
}

template <typename T, int R>
__device__ __forceinline__ T grad_op(const A2<T>* p, const A2<T>* l, int gen, int s0, int s1, const T* ct, int goff) {
  T a = 0;
  switch (gen) {
    case GN_X: TCM_SW1(R, s0, a = (g_x<T, R, S_>(p, l))) break;
    case GN_Y: TCM_SW1(R, s0, a = (g_y<T, R, S_>(p, l))) break;
    case GN_Z: TCM_SW1(R, s0, a = (g_z<T, R, S_>(p, l))) break;
    case GN_P1: TCM_SW1(R, s0, a = (g_p1<T, R, S_>(p, l))) break;
    case GN_XX: TCM_SW2(R, s0, s1, a = (g_xx<T, R, A_, B_>(p, l))) break;
    case GN_YY: TCM_SW2(R, s0, s1, a = (g_yy<T, R, A_, B_>(p, l))) break;
    case GN_ZZ: TCM_SW2(R, s0, s1, a = (g_zz<T, R, A_, B_>(p, l))) break;
    case GN_M1: TCM_SW1(R, s0, a = (g_m1<T, R, S_>(p, l, ct + goff))) break;
    case GN_M2: TCM_SW2(R, s0, s1, a = (g_m2<T, R, A_, B_>(p, l, ct + goff))) break;
    default: break;
  }
  return a;
}

// gradient of a diagonal-generator member from precomputed im[j] = Im(conj(l_j) p_j)
template <typename T, int R, int S>
__device__ __forceinline__ T gm_p1(const T* im) {
  T a = 0;
#pragma unroll
  for (int j = 0; j < (1 << R); ++j)
    if ((j >> S) & 1) a += im[j];
  return a;
}
template <typename T, int R, int S0, int S1>
__device__ __forceinline__ T gm_zz(const T* im) {
  T a = 0;
#pragma unroll
  for (int j = 0; j < (1 << R); ++j) a += (((j >> S0) ^ (j >> S1)) & 1) ? -im[j] : im[j];
  return a;
}
}  // namespace tcm

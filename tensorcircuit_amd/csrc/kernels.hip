// HIP kernels of libtcm for CDNA4 (gfx950): gate application (one kernel per
// gate, and LDS-tiled fused passes), adjoint reverse sweeps, Pauli-sum
// energies / H|psi>, and the fp64 reductions behind them.
//
// State layout: [batch][2^n] complex (float2 or double2), qubit 0 = the most
// significant index bit (circuit.py:803-810).  A gate on qubit q acts on index
// bit n-1-q.
#include <hip/hip_runtime.h>

#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>

#include "kernels.h"
#include "regops.h"

namespace tcm {

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ V2<T> mk(T a, T b) {
  V2<T> r;
  r.x = a;
  r.y = b;
  return r;
}

__device__ __forceinline__ uint32_t swz(uint32_t t) {
  return t ^ (((t >> 4) ^ (t >> 8) ^ (t >> 12) ^ (t >> 16)) & 0xFu);
}

// Offset (in amplitudes, from the block base) of tile element x: the tile's
// L low bits are contiguous in the state and the run-offset table `ro` maps
// the tile bits above them to their state bit positions.  The map is linear
// over disjoint bit sets, so element it * nthr + tid sits at
// tile_dep(it * nthr) (block-uniform, scalar loads) + tile_dep(tid).
__device__ __forceinline__ uint32_t tile_dep(const uint32_t* ro, int L, uint32_t x) {
  return ro[x >> L] + (x & ((1u << L) - 1));
}

// a pointer known to be the same in every lane, moved to scalar registers
template <typename P>
__device__ __forceinline__ P* uniform_ptr(P* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return reinterpret_cast<P*>(((uint64_t)hi << 32) | lo);
}

// insert a zero bit at position b
__device__ __forceinline__ uint64_t ins0(uint64_t x, int b) {
  uint64_t lo = x & ((1ull << b) - 1);
  return ((x >> b) << (b + 1)) | lo;
}

// block-wide sum of (a, b) in fp64; result valid in thread 0.  blockDim.x
// must be a multiple of 64 and <= 1024.
__device__ __forceinline__ void block_sum2(double& a, double& b) {
  __shared__ double red[2][16];
  a = wave_sum_dpp(a);
  b = wave_sum_dpp(b);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    red[0][w] = a;
    red[1][w] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int nw = blockDim.x >> 6;
    double sa = 0, sb = 0;
    for (int i = 0; i < nw; ++i) {
      sa += red[0][i];
      sb += red[1][i];
    }
    a = sa;
    b = sb;
  }
  __syncthreads();
}

// A diagonal entry in the working type.  For a phase in float, of the 9 pairs
// around it the one with the least 16 (|z| - 1)^2 + (angle error)^2: an angle
// error is a small unitary, which hardly moves the energy of a scrambled
// state, a length error is not, and the same one acts on half the state.
// Over 64 random 24-qubit, 20-layer circuits the nearest pair gave energies
// 1.6e-7 and norms 4.0e-7 off (rms), this 0.9e-7 and 0.9e-7 (with store_shears
// and the low parts of the factors).
__device__ __forceinline__ void store_diagonal(double* o, double re, double im) {
  o[0] = re;
  o[1] = im;
}
__device__ __forceinline__ void store_diagonal(float* o, double re, double im) {
  const float c0 = (float)re, s0 = (float)im;
  o[0] = c0;
  o[1] = s0;
  if (fabs(re * re + im * im - 1.0) > 1e-9 || c0 == 0.0f || s0 == 0.0f) return;
  double best = 1e300;
  for (int a = -1; a <= 1; ++a)
    for (int b = -1; b <= 1; ++b) {
      const float c = __int_as_float(__float_as_int(c0) + a), s = __int_as_float(__float_as_int(s0) + b);
      const double r = 0.5 * ((double)c * c + (double)s * s - 1.0), t = (double)s * re - (double)c * im;
      const double e = 16.0 * r * r + t * t;
      if (e < best) {
        best = e;
        o[0] = c;
        o[1] = s;
      }
    }
}

// a phase rounded to u, or (sg = -1) its conjugate, and at o + low the part of
// (re, sg im) that this cuts off
template <typename T>
__device__ __forceinline__ void put_phase(T* o, int low, const T* u, double re, double im, double sg) {
  o[0] = u[0];
  o[1] = (T)sg * u[1];
  o[low] = (T)(re - (double)u[0]);
  o[low + 1] = (T)(sg * (im - (double)u[1]));
}

// t = tan(ph / 2) and s = sin(ph) of the three shears, from cs = cos ph >= 0
// and sn = sin ph.  In float, of the 9 pairs around them the one whose matrix
// M = [[1 - ts, -t (2 - ts)], [s, 1 - ts]] has the least 16 |symmetric part|^2
// + |angle error|^2 of M R(ph)^T - 1 (see store_diagonal).
__device__ __forceinline__ void store_shears(double* o, double cs, double sn) {
  o[0] = sn / (1.0 + cs);
  o[1] = sn;
}
__device__ __forceinline__ void store_shears(float* o, double cs, double sn) {
  const float t0 = (float)(sn / (1.0 + cs)), s0 = (float)sn;
  o[0] = t0;
  o[1] = s0;
  if (t0 == 0.0f || s0 == 0.0f) return;
  double best = 1e300;
  for (int a = -1; a <= 1; ++a)
    for (int b = -1; b <= 1; ++b) {
      const float tf = __int_as_float(__float_as_int(t0) + a), sf = __int_as_float(__float_as_int(s0) + b);
      const double t = tf, s = sf, d = 1.0 - t * s, m = -t * (1.0 + d);
      const double e00 = d * cs - m * sn - 1.0, e01 = d * sn + m * cs, e10 = s * cs - d * sn, e11 = s * sn + d * cs - 1.0;
      const double h = 0.5 * (e01 + e10), g = 0.5 * (e10 - e01);
      const double e = 16.0 * (0.5 * (e00 * e00 + e11 * e11) + h * h) + g * g;
      if (e < best) {
        best = e;
        o[0] = tf;
        o[1] = sf;
      }
    }
}

// The entries kRotShear.. of an rx or ry recipe from c = cos phi, s = sin phi:
// three shears (Paeth), the rotation by phi' is x -= t y, y += s' x, x -= t y
// with t = tan(phi' / 2), s' = sin phi'; phi' is phi brought into [-pi/2, pi/2]
// (|t| <= 1) by R(phi) = -R(phi - pi), the sign kept in sigma.  All from c and
// s, whose reduction of the angle is exact: by the remainder of phi, a unit of
// pi was lost with every turn (1e-8 after 10^8).
template <typename T>
__device__ __forceinline__ void put_rotation(T* o, double c, double s) {
  const double sigma = c < 0.0 ? -1.0 : 1.0;
  store_shears(o + kRotShear, sigma * c, sigma * s);
  o[kRotSigma] = (T)sigma;
}

// ---------------------------------------------------------------------------
// matrix preparation: 2^wlog threads evaluate every recipe of one batch item of
// one schedule from its parameters.  A chain of a few loads and 64-bit sines, so
// the schedules of a call (forward and reverse, or the programs of an uneven
// batch) share a launch: 2 of 5 us became one of 6 us at 12 qubits x 4
// layers, 9 of 9 us one of 9 us for 9 programs.  Blocks are 1024 threads
// where a batch item has more than 512 entries
// and its block would be alone on its CU (2 of 63 us with 256 threads,
// one of 27 us, for 1420 gates and 4 parameter sets), else 256.
// Items of few entries share a block (2^20 parameter sets of one rotation,
// complex64, forward on 2 qubits: 1.62 ms with a block each, 0.05 ms).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(1024) k_prep(PrepJobs J) {
  int q = 0;
  while (q + 1 < J.njobs && (int64_t)blockIdx.x >= J.job[q + 1].block0) ++q;
  const DRecipe* __restrict__ rec = (const DRecipe*)J.job[q].rec;
  const DFactor* __restrict__ fac = (const DFactor*)J.job[q].fac;
  const T* __restrict__ ct = (const T*)J.job[q].ctab;
  const int nrec = J.job[q].nrec, first_dg = J.job[q].first_dg, dg_log = J.job[q].dg_log;
  const int wlog = J.job[q].wlog, W = 1 << wlog, lane = threadIdx.x & (W - 1);
  const int64_t b = (((int64_t)blockIdx.x - J.job[q].block0) * blockDim.x + threadIdx.x) >> wlog;
  const bool have = b < J.job[q].batch;
  T* mt = (T*)J.job[q].mtab + b * J.job[q].mstride;
  const T* __restrict__ pr = (const T*)J.job[q].params;
  if (pr) pr += b * J.job[q].pstride;
  for (int i = lane; i < first_dg && have; i += W) {
    const DRecipe r = rec[i];
    if (r.kind < 0) continue;
    double a = r.param >= 0 ? r.scale * (double)pr[r.param] : r.theta;
    T* o = mt + r.out;
    switch (r.kind) {
      case TCM_G_RX: {
        double c, s;
        sincos(0.5 * a, &s, &c);
        T u[2];
        store_diagonal(u, c, s);
        o[0] = u[0]; o[1] = 0; o[2] = 0; o[3] = -u[1]; o[4] = 0; o[5] = -u[1]; o[6] = u[0]; o[7] = 0;
        if (r.extra) put_rotation(o, c, s);
      } break;
      case TCM_G_RY: {
        double c, s;
        sincos(0.5 * a, &s, &c);
        T u[2];
        store_diagonal(u, c, s);
        o[0] = u[0]; o[1] = -u[1]; o[2] = u[1]; o[3] = u[0];
        if (r.extra) put_rotation(o, c, s);
      } break;
      case TCM_G_RZ:
      case TCM_G_RZZ: {
        // rz: entries by the bit; rzz: by the parity of the two bits
        const bool rz = r.kind == TCM_G_RZ;
        const int ne = rz ? 2 : 4, low = 2 * ne;
        double c, s;
        T u[2];
        sincos(0.5 * a, &s, &c);
        store_diagonal(u, c, s);
        for (int e = 0; e < ne; ++e) put_phase(o + 2 * e, low, u, c, s, ((e >> 1) ^ e) & 1 ? 1.0 : -1.0);
        if (r.extra) {
          const T one[2] = {1, 0};
          sincos(a, &s, &c);
          store_diagonal(u, c, s);
          T* q = o + 2 * low;
          for (int e = 0; e < ne; ++e) {
            if (((e >> 1) ^ e) & 1) put_phase(q + 2 * e, low, u, c, s, 1.0);
            else put_phase(q + 2 * e, low, one, 1.0, 0.0, 1.0);
          }
        }
      } break;
      case TCM_G_RXX:
      case TCM_G_RYY: {
        double c, s;
        sincos(0.5 * a, &s, &c);
        for (int q = 0; q < 32; ++q) o[q] = 0;
        for (int d = 0; d < 4; ++d) o[2 * (d * 4 + d)] = (T)c;
        if (r.kind == TCM_G_RXX) {
          // -i s XX : anti-diagonal ones
          for (int d = 0; d < 4; ++d) o[2 * (d * 4 + (3 - d)) + 1] = (T)-s;
        } else {
          // -i s YY : YY[0][3] = -1, YY[1][2] = 1, YY[2][1] = 1, YY[3][0] = -1
          o[2 * (0 * 4 + 3) + 1] = (T)s;
          o[2 * (1 * 4 + 2) + 1] = (T)-s;
          o[2 * (2 * 4 + 1) + 1] = (T)-s;
          o[2 * (3 * 4 + 0) + 1] = (T)s;
        }
      } break;
      case TCM_G_PHASE: {
        double c, s;
        sincos(a, &s, &c);
        o[0] = 1; o[1] = 0; o[2] = (T)c; o[3] = (T)s;
      } break;
      case TCM_G_EXP1: {
        // cos(a) I - i sin(a) G, G from the constant table (full matrix)
        double c, s;
        sincos(a, &s, &c);
        const T* g = ct + r.goff;
        const int d = (r.layout == OK_U1 || r.layout == OK_D1) ? 2 : 4;
        if (r.layout == OK_D1 || r.layout == OK_D2) {
          for (int q = 0; q < d; ++q) {
            double gr = g[2 * (q * d + q)], gi = g[2 * (q * d + q) + 1];
            o[2 * q] = (T)(c + s * gi);
            o[2 * q + 1] = (T)(-s * gr);
          }
        } else {
          for (int rr = 0; rr < d; ++rr)
            for (int cc = 0; cc < d; ++cc) {
              double gr = g[2 * (rr * d + cc)], gi = g[2 * (rr * d + cc) + 1];
              o[2 * (rr * d + cc)] = (T)((rr == cc ? c : 0.0) + s * gi);
              o[2 * (rr * d + cc) + 1] = (T)(-s * gr);
            }
        }
      } break;
      case TCM_G_EXPG: {
        // (I - Q) + cos(a) Q - i sin(a) G; G then Q = G^2 in the constant table
        double c, s;
        sincos(a, &s, &c);
        const int d = (r.layout == OK_U1 || r.layout == OK_D1) ? 2 : 4;
        const T* g = ct + r.goff;
        const T* q = g + 2 * d * d;
        if (r.layout == OK_D1 || r.layout == OK_D2) {
          for (int k = 0; k < d; ++k) {
            const int e = 2 * (k * d + k);
            o[2 * k] = (T)(1.0 + (c - 1.0) * (double)q[e] + s * (double)g[e + 1]);
            o[2 * k + 1] = (T)((c - 1.0) * (double)q[e + 1] - s * (double)g[e]);
          }
        } else {
          for (int rr = 0; rr < d; ++rr)
            for (int cc = 0; cc < d; ++cc) {
              const int e = 2 * (rr * d + cc);
              o[e] = (T)((rr == cc ? 1.0 : 0.0) + (c - 1.0) * (double)q[e] + s * (double)g[e + 1]);
              o[e + 1] = (T)((c - 1.0) * (double)q[e + 1] - s * (double)g[e]);
            }
        }
      } break;
      default: break;
    }
  }
  __syncthreads();
  // fused diagonals (recipes first_dg..nrec-1): products of member diagonals
  // over the group index j; lane t takes recipe first_dg + (t >> dg_log)
  // and entry t & (2^dg_log - 1), so all recipes are built side by side
  const int ndg = nrec - first_dg;
  for (int t = lane; t < (ndg << dg_log) && have; t += W) {
    const DRecipe r = rec[first_dg + (t >> dg_log)];
    const int j = t & ((1 << dg_log) - 1);
    if (r.kind >= 0 || j >= (1 << r.R)) continue;
    T* o = mt + r.out;
    {
      double pr_ = 1.0, pi_ = 0.0;
      for (int f = 0; f < r.nfac; ++f) {
        const DFactor F = fac[r.goff + f];
        double er, ei;
        if (F.layout == OK_CZ) {
          er = (((j >> F.s0) & 1) && ((j >> F.s1) & 1)) ? -1.0 : 1.0;
          ei = 0.0;
        } else {
          const T* src = F.src >= 0 ? mt + F.src : ct + (-F.src - 1);
          int idx = F.layout == OK_D1 ? ((j >> F.s0) & 1) : ((((j >> F.s0) & 1) << 1) | ((j >> F.s1) & 1));
          er = src[2 * idx];
          ei = src[2 * idx + 1];
          if (F.low) {
            er += src[F.low + 2 * idx];
            ei += src[F.low + 2 * idx + 1];
          }
        }
        double nr = pr_ * er - pi_ * ei, ni = pr_ * ei + pi_ * er;
        pr_ = nr;
        pi_ = ni;
      }
      if (r.extra) {
        // scalars: the 2^R threads of the recipe take every 2^R-th each, then
        // multiply across them
        const int G = 1 << r.R;
        double xr = 1.0, xi = 0.0;
        for (int f = j; f < r.extra; f += G) {
          const DFactor F = fac[r.goff + r.nfac + f];
          const T* src = mt + F.src;
          const double er = (double)src[0] + (double)src[F.low], ei = (double)src[1] + (double)src[F.low + 1];
          const double nr = xr * er - xi * ei;
          xi = xr * ei + xi * er;
          xr = nr;
        }
        for (int off = 1; off < G; off <<= 1) {
          const double er = __shfl_xor(xr, off, 64), ei = __shfl_xor(xi, off, 64), nr = xr * er - xi * ei;
          xi = xr * ei + xi * er;
          xr = nr;
        }
        const double nr = pr_ * xr - pi_ * xi;
        pi_ = pr_ * xi + pi_ * xr;
        pr_ = nr;
      }
      store_diagonal(o + 2 * j, pr_, pi_);
    }
  }
}

// |0..0> on every state of the batch
template <typename T>
__global__ void k_init_zero(V2<T>* __restrict__ st, int64_t total, int64_t N) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x)
    st[i] = mk<T>((i % N) == 0 ? T(1) : T(0), T(0));
}

// ---------------------------------------------------------------------------
// plain kernels: one launch per gate, grid-stride over (batch, item)
// ---------------------------------------------------------------------------
template <typename T, int KIND, bool DAG>
__global__ void __launch_bounds__(256) k_plain1(DOp op, const T* __restrict__ mtab, int64_t mstride,
                                                const T* __restrict__ ct, A2<T>* __restrict__ st,
                                                int64_t sstride, int n, int64_t batch) {
  const int64_t items = 1ll << (n - 1);
  const int64_t total = items * batch;
  const int b0 = op.s0;
  for (int64_t w = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; w < total; w += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = w >> (n - 1);
    const int64_t idx = w & (items - 1);
    const uint64_t i0 = ins0(idx, b0), i1 = i0 | (1ull << b0);
    A2<T>* s = st + b * sstride;
    A2<T> v[2] = {s[i0], s[i1]};
    const T* mt = mtab + b * mstride;
    DOp o = op;
    o.s0 = 0;
    apply_op<T, 1, DAG>(v, o, mt, ct);
    s[i0] = v[0];
    s[i1] = v[1];
  }
}

template <typename T, int KIND, bool DAG>
__global__ void __launch_bounds__(256) k_plain2(DOp op, const T* __restrict__ mtab, int64_t mstride,
                                                const T* __restrict__ ct, A2<T>* __restrict__ st,
                                                int64_t sstride, int n, int64_t batch) {
  const int64_t items = 1ll << (n - 2);
  const int64_t total = items * batch;
  const int ba = op.s0, bb = op.s1;  // bit of qubit 0 (matrix MSB), qubit 1
  const int lo = ba < bb ? ba : bb, hi = ba < bb ? bb : ba;
  for (int64_t w = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; w < total; w += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = w >> (n - 2);
    const int64_t idx = w & (items - 1);
    const uint64_t i00 = ins0(ins0(idx, lo), hi);
    const uint64_t ma = 1ull << ba, mb = 1ull << bb;
    A2<T>* s = st + b * sstride;
    // register index: bit 1 <-> qubit 0 (matrix MSB), bit 0 <-> qubit 1
    A2<T> v[4] = {s[i00], s[i00 | mb], s[i00 | ma], s[i00 | ma | mb]};
    const T* mt = mtab + b * mstride;
    DOp o = op;
    o.s0 = 1;
    o.s1 = 0;
    apply_op<T, 2, DAG>(v, o, mt, ct);
    s[i00] = v[0];
    s[i00 | mb] = v[1];
    s[i00 | ma] = v[2];
    s[i00 | ma | mb] = v[3];
  }
}

// dense k-qubit gate (k = K), constant matrix; bits[0] = matrix MSB
template <typename T, int K, bool DAG>
__global__ void __launch_bounds__(256) k_plaink(DOp op, const int32_t* __restrict__ ukbits,
                                                const T* __restrict__ ct, V2<T>* __restrict__ st,
                                                int64_t sstride, int n, int64_t batch) {
  const int64_t items = 1ll << (n - K);
  const int64_t total = items * batch;
  int bits[K], sorted[K];
  for (int i = 0; i < K; ++i) sorted[i] = bits[i] = ukbits[op.mem0 + i];
  for (int i = 0; i < K; ++i)
    for (int j = i + 1; j < K; ++j)
      if (sorted[j] < sorted[i]) { int t = sorted[i]; sorted[i] = sorted[j]; sorted[j] = t; }
  const T* m = ct + (-op.moff - 1);
  constexpr int D = 1 << K;
  for (int64_t w = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; w < total; w += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = w >> (n - K);
    uint64_t base = w & (items - 1);
    for (int i = 0; i < K; ++i) base = ins0(base, sorted[i]);
    V2<T>* s = st + b * sstride;
    V2<T> x[D];
    uint64_t ad[D];
#pragma unroll
    for (int c = 0; c < D; ++c) {
      uint64_t a = base;
#pragma unroll
      for (int i = 0; i < K; ++i)
        if ((c >> (K - 1 - i)) & 1) a |= 1ull << bits[i];
      ad[c] = a;
      x[c] = s[a];
    }
    for (int r = 0; r < D; ++r) {
      T sr = 0, si = 0;
#pragma unroll
      for (int c = 0; c < D; ++c) {
        T mr, mi;
        if constexpr (DAG) { mr = m[2 * (c * D + r)]; mi = -m[2 * (c * D + r) + 1]; }
        else { mr = m[2 * (r * D + c)]; mi = m[2 * (r * D + c) + 1]; }
        sr += mr * x[c].x - mi * x[c].y;
        si += mr * x[c].y + mi * x[c].x;
      }
      s[ad[r]] = mk<T>(sr, si);
    }
  }
}

// plain adjoint step for a 1- or 2-qubit gate: gradient partial (if the gate
// is trainable), then psi <- U^dag psi, lambda <- U^dag lambda.
// grid = (slots, batch); partial[b * pstride + blockIdx.x]
template <typename T, int NQ>
__global__ void __launch_bounds__(256) k_plain_adj(DOp op, const T* __restrict__ mtab, int64_t mstride,
                                                   const T* __restrict__ ct, const A2<T>* psi_in, A2<T>* psi_out,
                                                   const A2<T>* lam_in, A2<T>* lam_out, int64_t sstride, int n,
                                                   double* __restrict__ part, int64_t pstride) {
  const int64_t items = 1ll << (n - NQ);
  const int64_t b = blockIdx.y;
  const T* mt = mtab + b * mstride;
  const A2<T>* pi = psi_in + b * sstride;
  const A2<T>* li = lam_in + b * sstride;
  A2<T>* po = psi_out ? psi_out + b * sstride : nullptr;
  A2<T>* lo_ = lam_out + b * sstride;
  double acc = 0.0;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < items; idx += (int64_t)gridDim.x * blockDim.x) {
    if constexpr (NQ == 1) {
      const int b0 = op.s0;
      const uint64_t i0 = ins0(idx, b0), i1 = i0 | (1ull << b0);
      A2<T> p[2] = {pi[i0], pi[i1]}, l[2] = {li[i0], li[i1]};
      if (op.gen != GN_NONE) acc += (double)grad_op<T, 1>(p, l, op.gen, 0, -1, ct, op.goff);
      DOp o = op;
      o.s0 = 0;
      apply_op<T, 1, true>(p, o, mt, ct);
      apply_op<T, 1, true>(l, o, mt, ct);
      if (po) { po[i0] = p[0]; po[i1] = p[1]; }
      lo_[i0] = l[0];
      lo_[i1] = l[1];
    } else {
      const int ba = op.s0, bb = op.s1;
      const int lo = ba < bb ? ba : bb, hi = ba < bb ? bb : ba;
      const uint64_t i00 = ins0(ins0(idx, lo), hi);
      const uint64_t ma = 1ull << ba, mb = 1ull << bb;
      const uint64_t ad[4] = {i00, i00 | mb, i00 | ma, i00 | ma | mb};
      A2<T> p[4], l[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) { p[c] = pi[ad[c]]; l[c] = li[ad[c]]; }
      if (op.gen != GN_NONE) acc += (double)grad_op<T, 2>(p, l, op.gen, 1, 0, ct, op.goff);
      DOp o = op;
      o.s0 = 1;
      o.s1 = 0;
      apply_op<T, 2, true>(p, o, mt, ct);
      apply_op<T, 2, true>(l, o, mt, ct);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (po) po[ad[c]] = p[c];
        lo_[ad[c]] = l[c];
      }
    }
  }
  if (op.gop >= 0) {
    double dummy = 0.0;
    block_sum2(acc, dummy);
    if (threadIdx.x == 0) part[b * pstride + blockIdx.x] = acc;
  }
}

// ---------------------------------------------------------------------------
// dense 5-qubit gate on FP32 matrix cores.  The state is viewed as a
// 32 x (2^(n-5)) matrix X (rows = the 5 gate bits, row MSB = gate qubit 0,
// columns = all other bits) and Y = U X is computed per 32-column chunk by
// one wave with v_mfma_f32_32x32x2f32 (K = 2 per instruction), as three
// real products (Gauss's complex multiplication):
//   P1 = Ur Xr,  P2 = Ui Xi,  P3 = (Ur + Ui)(Xr + Xi),
//   Yr = P1 - P2,  Yi = P3 - P1 - P2.
// Operand layouts (CDNA3/4): lane l supplies A[l % 32][l / 32] and
// B[l / 32][l % 32]; accumulator register r of lane l holds
// D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
// ---------------------------------------------------------------------------
typedef float tcm_v16f __attribute__((ext_vector_type(16)));
// two complex64 amplitudes (one 16-byte access; a native vector, so copies
// stay in registers)
typedef float tcm_v4f __attribute__((ext_vector_type(4)));

template <bool DAG>
__global__ void __launch_bounds__(256) k_mfma_u5(DOp op, const int32_t* __restrict__ ukbits,
                                                 const float* __restrict__ ct, float2* __restrict__ st,
                                                 int64_t sstride, int n, int64_t batch) {
  const int lane = threadIdx.x & 63;
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
  const float* U = ct + (-op.moff - 1);
  int bits[5], sorted[5];
  for (int i = 0; i < 5; ++i) sorted[i] = bits[i] = ukbits[op.mem0 + i];
  for (int i = 0; i < 5; ++i)
    for (int j = i + 1; j < 5; ++j)
      if (sorted[j] < sorted[i]) { int t = sorted[i]; sorted[i] = sorted[j]; sorted[j] = t; }
  // A operands for the 16 K-steps: U[i][2s + l/32] (U^dag: conj(U[2s + l/32][i]))
  const int ai = lane & 31, ak = lane >> 5;
  float ur[16], ui[16];
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    const int kk = 2 * s + ak;
    if (DAG) {
      ur[s] = U[2 * (kk * 32 + ai)];
      ui[s] = -U[2 * (kk * 32 + ai) + 1];
    } else {
      ur[s] = U[2 * (ai * 32 + kk)];
      ui[s] = U[2 * (ai * 32 + kk) + 1];
    }
  }
  // index offset of gate row r (5 bits, MSB = bits[0])
  auto rowoff = [&](int r) {
    uint64_t o = 0;
#pragma unroll
    for (int i = 0; i < 5; ++i)
      if ((r >> (4 - i)) & 1) o |= 1ull << bits[i];
    return o;
  };
  const int64_t ncol = 1ll << (n - 5);
  const int64_t chunks_per_state = ncol >> 5;
  const int64_t nchunks = chunks_per_state * batch;
  // chunk ch: 32 consecutive columns of one state; the next chunk's loads
  // are issued before this chunk's matrix-core work (software pipelining)
  auto chunk_ptr = [&](int64_t ch) {
    const int64_t b = ch / chunks_per_state;
    const uint64_t c = ((uint64_t)(ch % chunks_per_state) << 5) + (lane & 31);
    uint64_t base = c;
#pragma unroll
    for (int i = 0; i < 5; ++i) base = ins0(base, sorted[i]);
    return st + b * sstride + base;
  };
  if (wave >= nchunks) return;
  float2* s = chunk_ptr(wave);
  float2 x[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) x[q] = s[rowoff(2 * q + ak)];
  for (int64_t ch = wave; ch < nchunks; ch += nwaves) {
    const bool more = ch + nwaves < nchunks;
    float2* sn = more ? chunk_ptr(ch + nwaves) : s;
    float2 xn[16];
    if (more) {
#pragma unroll
      for (int q = 0; q < 16; ++q) xn[q] = sn[rowoff(2 * q + ak)];
    }
    tcm_v16f p1 = {0}, p2 = {0}, p3 = {0};
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      p1 = __builtin_amdgcn_mfma_f32_32x32x2f32(ur[q], x[q].x, p1, 0, 0, 0);
      p2 = __builtin_amdgcn_mfma_f32_32x32x2f32(ui[q], x[q].y, p2, 0, 0, 0);
      p3 = __builtin_amdgcn_mfma_f32_32x32x2f32(ur[q] + ui[q], x[q].x + x[q].y, p3, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = 8 * (r >> 2) + 4 * ak + (r & 3);
      s[rowoff(row)] = make_float2(p1[r] - p2[r], p3[r] - p1[r] - p2[r]);
    }
    if (more) {
#pragma unroll
      for (int q = 0; q < 16; ++q) x[q] = xn[q];
      s = sn;
    }
  }
}

// f(0), f(1), ..., f(N - 1) with compile-time indices (register arrays
// indexed by them stay in registers)
template <int N, typename F>
__device__ __forceinline__ void unrolled(F&& f) {
  if constexpr (N > 0) {
    unrolled<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// One tile pass of dense 5-qubit blocks on FP32 matrix cores.  A tile is the
// 2^K amplitudes whose index bits are the pass's tile bits; each block
// multiplies the tile, viewed as 32 rows (the block's 5 tile bits, first bit
// most significant) x 2^(K-5) columns (the other tile bits, ascending), by
// its 32x32 complex matrix U.  Wave w takes the 32-column chunk w and forms
// Y = U X from three real products (Gauss's complex multiplication):
//   P1 = Ur Xr,  P2 = Ui Xi,  P3 = (Ur + Ui)(Xr + Xi),
//   Yr = P1 - P2,  Yi = P3 - P1 - P2,
// 48 v_mfma_f32_32x32x2f32 per chunk instead of the 64 of four products.
// Waves own disjoint columns, so only the block boundary needs a barrier.
// The kernel is persistent: a block stages the A operands of all the pass's
// blocks in LDS once, then runs tiles blockIdx.x, blockIdx.x + gridDim.x, ...
// and loads the next tile's amplitudes into registers while the matrix
// cores work on the current one.  Row offsets are XORs of the 5 gate bits'
// swizzled offsets (the swizzle is linear over XOR).  512 threads; LDS =
// 8 << K bytes (tile) + nmop * (8 KiB A operands, [block][K-step][lane], +
// the gate-bit and column offsets).
template <int K>
__global__ void __launch_bounds__(512) k_mfma_tile(const DPass* __restrict__ passes, int pi,
                                                   const DOp* __restrict__ dop, const int32_t* __restrict__ ukbits,
                                                   const uint32_t* __restrict__ runoff, const float* __restrict__ ct,
                                                   const float2* src, float2* st, int64_t sstride, int64_t ntiles) {
  // src: the states read, st itself or others (the first pass of a circuit on
  // given inputs).  Each thread moves PER2 pairs of adjacent amplitudes (16-byte accesses)
  constexpr int NTHR = 512, PER2 = (1 << K) / (2 * NTHR), CHUNKS = 1 << (K - 10), NCOL = 1 << (K - 5);
  extern __shared__ __align__(16) unsigned char smem[];
  float2* tile = reinterpret_cast<float2*>(smem);
  const DPass* P = uniform_ptr(passes + pi);
  const int L = P->L, nbl = P->nblk_log, nmop = P->nmop;
  float2* amat = tile + (1 << K);
  // per block: the swizzled offsets of its 5 gate bits, then the swizzled
  // offsets of its NCOL columns
  uint32_t* ebits = reinterpret_cast<uint32_t*>(amat + nmop * 1024);
  uint32_t* xcol = ebits + nmop * 8;
  const int tid = threadIdx.x;
  int64_t t = blockIdx.x;
  if (t >= ntiles) return;
  const DOp* ops = dop + P->mop0;
  const uint32_t* ro = runoff + P->runoff0;
  // Every table read happens here, before the first store: reads inside the
  // tile loop would be vector loads queued behind the prefetch and the stores.
  // A operands: lane l of K-step q supplies U[l % 32][2q + l / 32]
  for (int idx = tid; idx < nmop * 1024; idx += NTHR) {
    const int o = idx >> 10, q = (idx >> 6) & 15, ln = idx & 63;
    const float* U = ct + (-ops[o].moff - 1);
    const int e = 2 * ((ln & 31) * 32 + 2 * q + (ln >> 5));
    amat[idx] = make_float2(U[e], U[e + 1]);
  }
  if (tid < nmop * 8) {
    const int32_t* ub = ukbits + ops[tid >> 3].mem0;
    const int i = tid & 7;
    ebits[tid] = i < 5 ? swz(1u << ub[i]) : 0u;
  }
  // column c of a block -> the tile bits outside the block, ascending
  for (int idx = tid; idx < nmop * NCOL; idx += NTHR) {
    const int32_t* ub = ukbits + ops[idx / NCOL].mem0;
    uint32_t bm = 0;
    for (int j = 0; j < 5; ++j) bm |= 1u << ub[j];
    const uint32_t col = (uint32_t)(idx % NCOL);
    uint32_t cb = 0;
    for (int b = 0, j = 0; b < K; ++b)
      if (!((bm >> b) & 1)) {
        if ((col >> j) & 1) cb |= 1u << b;
        ++j;
      }
    xcol[idx] = swz(cb);
  }
  uint64_t bmask = 0;
  for (int i = 0; i < nbl; ++i) bmask |= 1ull << P->blk_bits[i];
  // pair it of this thread: tile elements x = 2 (it * NTHR + tid) and x + 1,
  // adjacent in the state (the low L >= 4 tile bits are contiguous) and in
  // LDS, at slots swz(x) and swz(x) ^ 1: in reverse order when swz(x) is odd
  // (the swizzle folds bits 4, 8, 12 into bit 0)
  uint32_t roff[PER2];
  unrolled<PER2>([&](auto it) { roff[it] = tile_dep(ro, L, it * 2 * NTHR); });
  const uint32_t dlo = tile_dep(ro, L, 2 * tid);
  const uint32_t slo = swz(2 * tid);
  tcm_v4f* tile4 = reinterpret_cast<tcm_v4f*>(smem);
  auto put4 = [&](int it, tcm_v4f v) {
    const uint32_t i = swz(it * 2 * NTHR) ^ slo;
    if (i & 1) v = v.zwxy;
    tile4[i >> 1] = v;
  };
  auto get4 = [&](int it) -> tcm_v4f {
    const uint32_t i = swz(it * 2 * NTHR) ^ slo;
    tcm_v4f v = tile4[i >> 1];
    if (i & 1) v = v.zwxy;
    return v;
  };
  // tile tt: batch item tt >> nbl; its block bits (ascending) hold the low nbl bits of tt
  auto tile_at = [&](int64_t tt) {
    const uint64_t blk = (uint64_t)tt & ((1ull << nbl) - 1);
    uint64_t m = bmask, base = 0;
    for (int i = 0; i < nbl; ++i) {
      const uint64_t low = m & (~m + 1);
      if ((blk >> i) & 1) base |= low;
      m ^= low;
    }
    return (int64_t)(((uint64_t)tt >> nbl) * sstride + base);
  };
  auto in4 = [&](int64_t sp, int it) { return *reinterpret_cast<const tcm_v4f*>(src + sp + roff[it] + dlo); };
  auto out4 = [&](int64_t sp, int it) -> tcm_v4f& { return *reinterpret_cast<tcm_v4f*>(st + sp + roff[it] + dlo); };
  const int lane = tid & 63, wave = tid >> 6;
  const int ai = lane & 31, ak = lane >> 5;
  // A operands of the pass's first two blocks (filled once staged)
  float2 a0[16], a1[16];
  // block o of the pass on the tile in LDS; geta(q) gives its A operand of K-step q
  auto block = [&](int o, auto geta) {
    if (wave < CHUNKS) {
      const uint32_t* ob = ebits + o * 8;
      uint32_t e[5];
#pragma unroll
      for (int i = 0; i < 5; ++i) e[i] = __builtin_amdgcn_readfirstlane(ob[i]);
      const uint32_t xc = xcol[o * NCOL + wave * 32 + ai];
      // read rows 2q + ak; written rows 8 (r / 4) + 4 ak + r % 4
      const uint32_t rb = xc ^ (ak ? e[4] : 0u);
      const uint32_t wb = xc ^ (ak ? e[2] : 0u);
      float2 a[16], x[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        a[q] = geta(q);
        const uint32_t g = ((q & 1) ? e[3] : 0u) ^ ((q & 2) ? e[2] : 0u) ^ ((q & 4) ? e[1] : 0u) ^
                           ((q & 8) ? e[0] : 0u);
        x[q] = tile[rb ^ g];
      }
      tcm_v16f p1 = {0}, p2 = {0}, p3 = {0};
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        p1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q].x, x[q].x, p1, 0, 0, 0);
        p2 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q].y, x[q].y, p2, 0, 0, 0);
        p3 = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q].x + a[q].y, x[q].x + x[q].y, p3, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t h = ((r & 1) ? e[4] : 0u) ^ ((r & 2) ? e[3] : 0u) ^ ((r & 4) ? e[1] : 0u) ^
                           ((r & 8) ? e[0] : 0u);
        tile[wb ^ h] = make_float2(p1[r] - p2[r], p3[r] - p1[r] - p2[r]);
      }
    }
    __syncthreads();
  };
  // the pass's blocks in order, each followed by a barrier
  auto blocks = [&]() {
    block(0, [&](int q) { return a0[q]; });
    if (nmop > 1) block(1, [&](int q) { return a1[q]; });
    for (int o = 2; o < nmop; ++o) block(o, [&](int q) { return amat[o * 1024 + q * 64 + lane]; });
  };
  int64_t s = tile_at(t);
  tcm_v4f pre[PER2];
  unrolled<PER2>([&](auto it) { pre[it] = in4(s, it); });
  unrolled<PER2>([&](auto it) { put4(it, pre[it]); });
  // the first two blocks' A operands stay in registers for every tile
  __syncthreads();
  unrolled<16>([&](auto q) {
    a0[q] = amat[q * 64 + lane];
    a1[q] = amat[(nmop > 1 ? 1024 : 0) + q * 64 + lane];
  });
  // every tile but the last: the next tile's loads are issued before this
  // tile's matrix-core work; each thread then stores the LDS slots it wrote
  // and refills them with the next tile (same slots: no barrier between)
  for (;;) {
    const int64_t tn = t + gridDim.x;
    if (tn >= ntiles) break;
    const int64_t sn = tile_at(tn);
    unrolled<PER2>([&](auto it) { pre[it] = in4(sn, it); });
    __syncthreads();  // the tile (and, first time, the staged operands) in LDS
    blocks();
    unrolled<PER2>([&](auto it) {
      out4(s, it) = get4(it);
      put4(it, pre[it]);
    });
    t = tn;
    s = sn;
  }
  __syncthreads();
  blocks();
  unrolled<PER2>([&](auto it) { out4(s, it) = get4(it); });
}

// Blocks of `kern` (512 threads, `lds` bytes of LDS) resident on the whole
// device at once: the grid of a persistent kernel.
template <typename Kern>
static int64_t resident_grid(Kern kern, size_t lds) {
  static std::mutex mu;
  static std::map<std::tuple<int, const void*, size_t>, int64_t> cache;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 256;
  std::lock_guard<std::mutex> lk(mu);
  const auto key = std::make_tuple(dev, (const void*)kern, lds);
  auto it = cache.find(key);
  if (it != cache.end()) return it->second;
  int per_cu = 0, ncu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, 512, lds) != hipSuccess || per_cu < 1) per_cu = 1;
  if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || ncu < 1) ncu = 256;
  return cache[key] = (int64_t)per_cu * ncu;
}


template <int K>
static void launch_mfma_tile_k(const DPass& P, const DPass* passes_dev, int pi, const DOp* dop_dev,
                               const int32_t* ukbits_dev, const uint32_t* runoff_dev, const void* ctab, const void* src,
                               void* state, int n, int64_t batch, hipStream_t st) {
  const size_t lds = ((size_t)8 << K) + (size_t)P.nmop * (8192 + 32 + (4 << (K - 5)));
  allow_lds((const void*)k_mfma_tile<K>, lds);
  const int64_t ntiles = batch << P.nblk_log;
  const int64_t grid = std::min<int64_t>(ntiles, resident_grid(k_mfma_tile<K>, lds));
  hipLaunchKernelGGL(k_mfma_tile<K>, dim3((unsigned)grid), dim3(512), lds, st, passes_dev, pi, dop_dev, ukbits_dev,
                     runoff_dev, (const float*)ctab, (const float2*)src, (float2*)state, (int64_t)1 << n, ntiles);
}

bool launch_mfma_tile(const DPass& P, const DPass* passes_dev, int pi, const DOp* dop_dev, const int32_t* ukbits_dev,
                      const uint32_t* runoff_dev, const void* ctab, const void* src, void* state, int n, int64_t batch,
                      hipStream_t st) {
  if (P.nmop < 1 || P.nmop > kMfmaTileMaxOps || P.nblk_log != n - P.k) return false;
  switch (P.k) {
    case 10: launch_mfma_tile_k<10>(P, passes_dev, pi, dop_dev, ukbits_dev, runoff_dev, ctab, src, state, n, batch, st); return true;
    case 11: launch_mfma_tile_k<11>(P, passes_dev, pi, dop_dev, ukbits_dev, runoff_dev, ctab, src, state, n, batch, st); return true;
    case 12: launch_mfma_tile_k<12>(P, passes_dev, pi, dop_dev, ukbits_dev, runoff_dev, ctab, src, state, n, batch, st); return true;
    case 13: launch_mfma_tile_k<13>(P, passes_dev, pi, dop_dev, ukbits_dev, runoff_dev, ctab, src, state, n, batch, st); return true;
    default: return false;
  }
}

// ---------------------------------------------------------------------------
// reductions
// ---------------------------------------------------------------------------
// sum of part[s * step], s = tid, tid + nthr, ... < n: four loads in flight
__device__ __forceinline__ double strided_sum(const double* __restrict__ part, int64_t n, int step, int tid, int nthr) {
  double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
  int64_t s = tid;
  for (; s + 3 * (int64_t)nthr < n; s += 4 * (int64_t)nthr) {
    a0 += part[s * step];
    a1 += part[(s + nthr) * step];
    a2 += part[(s + 2 * (int64_t)nthr) * step];
    a3 += part[(s + 3 * (int64_t)nthr) * step];
  }
  for (; s < n; s += nthr) a0 += part[s * step];
  return (a0 + a1) + (a2 + a3);
}

// out[b * ncomp + c] = sum_s part[b * bstride + s * ncomp + c]; a block per b
// (several in turn for very many), bound by the loads that it keeps in flight (49k pairs: 86 us with 256
// threads and one load each, 20 us with 1024 and four), or by the blocks where
// there are few per b (60000 states of 2 qubits and 3 pairs, with the launches
// that make them: 155 us with 256 threads each, 131 us with 64)
__global__ void __launch_bounds__(1024) k_sum_slots(const double* __restrict__ part, int64_t bstride, int64_t nslots,
                                                    int ncomp, double* __restrict__ out, int64_t batch) {
  for (int64_t b = blockIdx.x; b < batch; b += gridDim.x) {
    double a = strided_sum(part + b * bstride, nslots, ncomp, threadIdx.x, blockDim.x), c = 0.0;
    if (ncomp > 1) c = strided_sum(part + b * bstride + 1, nslots, ncomp, threadIdx.x, blockDim.x);
    block_sum2(a, c);
    if (threadIdx.x == 0) {
      out[b * ncomp] = a;
      if (ncomp > 1) out[b * ncomp + 1] = c;
    }
  }
}

// gsum[b][gop] = sum over slots of part[b][gl][slot]; grid (ngop_pass, batch)
__global__ void k_reduce_gop(const double* __restrict__ part, int64_t pstride, int64_t nslots,
                             const int32_t* __restrict__ gop_list, int gop_single, double* __restrict__ gsum,
                             int ngop) {
  const int gl = blockIdx.x;
  const int64_t b = blockIdx.y;
  double a = 0.0, d = 0.0;
  for (int64_t s = threadIdx.x; s < nslots; s += blockDim.x) a += part[b * pstride + gl * nslots + s];
  block_sum2(a, d);
  if (threadIdx.x == 0) {
    const int gop = gop_list ? gop_list[gl] : gop_single;
    gsum[b * ngop + gop] = a;
  }
}

// The end of a reverse sweep in one launch (after a launch per pass for its
// partials, then sums, a copy and the chain rule, it was npasses + 3):
//   energy[b]  = sum_s epart[b][s].re            blocks 0 .. nenergy - 1
//   grad[b][p] = mult * sum_{gop of p} gfac[gop] * (sum of the gop's partials)
// 16 passes of a 24-qubit circuit with 4 parameter sets: 16 launches and 105 us
// before, 15 us here; a circuit of one tile: 4 launches, 14 us, before, 5 us here.
// LP threads share a (b, p): a wave, or one thread where a gop has a single
// partial (states of one tile).
template <int LP>
__global__ void __launch_bounds__(256) k_finish(const double* __restrict__ epart, int64_t nslots, int64_t nenergy,
                                                double* __restrict__ energy, const double* __restrict__ part,
                                                const DGopSum* __restrict__ gs, int ngop,
                                                const int32_t* __restrict__ p_ptr, const int32_t* __restrict__ p_gops,
                                                const double* __restrict__ gfac, double mult,
                                                double* __restrict__ grad, int nparams, int64_t batch) {
  if ((int64_t)blockIdx.x < nenergy) {
    for (int64_t b = blockIdx.x; b < batch; b += nenergy) {
      double a = strided_sum(epart + b * nslots * 2, nslots, 2, threadIdx.x, 256), c = 0.0;
      block_sum2(a, c);
      if (threadIdx.x == 0) energy[b] = a;
    }
    return;
  }
  const int64_t total = (int64_t)nparams * batch, step = (int64_t)(gridDim.x - nenergy) * (256 / LP);
  const int lane = threadIdx.x & (LP - 1);
  for (int64_t i = ((int64_t)blockIdx.x - nenergy) * (256 / LP) + threadIdx.x / LP; i < total; i += step) {
    const int64_t b = i / nparams;
    const int p = (int)(i - b * nparams);
    double a = 0.0;
    for (int q = p_ptr[p]; q < p_ptr[p + 1]; ++q) {
      const int gop = p_gops[q];
      double x;
      if (gs) {
        const DGopSum g = gs[gop];
        x = strided_sum(part + batch * g.base + (b * g.ngop + g.row) * (int64_t)g.slots, g.slots, 1, lane, LP);
      } else {
        x = lane == 0 ? part[b * ngop + gop] : 0.0;
      }
      a += gfac[gop] * x;
    }
    if (LP > 1)
      for (int off = LP / 2; off > 0; off >>= 1) a += __shfl_xor(a, off, LP);
    if (lane == 0) grad[i] = mult * a;
  }
}

// ---------------------------------------------------------------------------
// Pauli sums: one launch per flip group (terms sharing the X/Y positions).
// (P psi)[y] = i^{ny} (-1)^{popcount((y ^ flip) & yz)} psi[y ^ flip]
// (index rule of ps2coo_core, quantum.py:1461-1485)
// ---------------------------------------------------------------------------
struct PauliAcc {
  double re, im;
};

__device__ __forceinline__ PauliAcc pauli_coef(const DPTerm* __restrict__ terms, int t0, int nt, uint64_t y) {
  // sum_k w_k i^{ny_k} (-1)^{popcount(y & yz_k)}, y = the source index y ^ flip
  double re = 0.0, im = 0.0;
  for (int t = t0; t < t0 + nt; ++t) {
    const DPTerm tm = terms[t];
    double w = (__popcll(y & tm.yz) & 1) ? -tm.w : tm.w;
    switch (tm.ny & 3) {
      case 0: re += w; break;
      case 1: im += w; break;
      case 2: re -= w; break;
      default: im -= w; break;
    }
  }
  return {re, im};
}

template <typename T, bool ENERGY, bool APPLY>
__global__ void __launch_bounds__(256) k_pauli(DPGroup G, const DPTerm* __restrict__ terms, int n,
                                               const V2<T>* __restrict__ psi, int64_t sstride,
                                               V2<T>* __restrict__ out, int first, const double* __restrict__ alpha,
                                               double* __restrict__ epart, int64_t estride) {
  const int64_t b = blockIdx.y;
  const V2<T>* s = psi + b * sstride;
  V2<T>* o = APPLY ? out + b * sstride : nullptr;
  const double al = (APPLY && alpha) ? alpha[b] : 1.0;
  const int64_t N = 1ll << n;
  double er = 0.0, ei = 0.0;
  if (G.flip) {
    const int h = 63 - __clzll(G.flip);
    const int64_t items = N >> 1;
    for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < items; idx += (int64_t)gridDim.x * blockDim.x) {
      const uint64_t y0 = ins0(idx, h), y1 = y0 ^ G.flip;
      const V2<T> p0 = s[y0], p1 = s[y1];
      const PauliAcc a0 = pauli_coef(terms, G.t0, G.nt, y1);  // (H psi)[y0] = a0 * psi[y1]
      const PauliAcc a1 = pauli_coef(terms, G.t0, G.nt, y0);
      const double h0r = a0.re * p1.x - a0.im * p1.y, h0i = a0.re * p1.y + a0.im * p1.x;
      const double h1r = a1.re * p0.x - a1.im * p0.y, h1i = a1.re * p0.y + a1.im * p0.x;
      if constexpr (ENERGY) {
        er += (double)p0.x * h0r + (double)p0.y * h0i + (double)p1.x * h1r + (double)p1.y * h1i;
        ei += (double)p0.x * h0i - (double)p0.y * h0r + (double)p1.x * h1i - (double)p1.y * h1r;
      }
      if constexpr (APPLY) {
        if (first) {
          o[y0] = mk<T>((T)(al * h0r), (T)(al * h0i));
          o[y1] = mk<T>((T)(al * h1r), (T)(al * h1i));
        } else {
          V2<T> q0 = o[y0], q1 = o[y1];
          o[y0] = mk<T>((T)(q0.x + al * h0r), (T)(q0.y + al * h0i));
          o[y1] = mk<T>((T)(q1.x + al * h1r), (T)(q1.y + al * h1i));
        }
      }
    }
  } else {
    for (int64_t y = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; y < N; y += (int64_t)gridDim.x * blockDim.x) {
      const V2<T> p = s[y];
      const PauliAcc a = pauli_coef(terms, G.t0, G.nt, (uint64_t)y);
      const double hr = a.re * p.x - a.im * p.y, hi = a.re * p.y + a.im * p.x;
      if constexpr (ENERGY) {
        er += (double)p.x * hr + (double)p.y * hi;
        ei += (double)p.x * hi - (double)p.y * hr;
      }
      if constexpr (APPLY) {
        if (first) o[y] = mk<T>((T)(al * hr), (T)(al * hi));
        else {
          V2<T> q = o[y];
          o[y] = mk<T>((T)(q.x + al * hr), (T)(q.y + al * hi));
        }
      }
    }
  }
  if constexpr (ENERGY) {
    block_sum2(er, ei);
    if (threadIdx.x == 0) {
      epart[b * estride + 2 * (G.slot0 + blockIdx.x)] = er;
      epart[b * estride + 2 * (G.slot0 + blockIdx.x) + 1] = ei;
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(256) k_inner(const V2<T>* __restrict__ a, const V2<T>* __restrict__ c, int n,
                                               int64_t sstride, double* __restrict__ part, int64_t pstride) {
  const int64_t b = blockIdx.y;
  const int64_t N = 1ll << n;
  double re = 0.0, im = 0.0;
  for (int64_t y = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; y < N; y += (int64_t)gridDim.x * blockDim.x) {
    const V2<T> x = a[b * sstride + y], z = c[b * sstride + y];
    re += (double)x.x * z.x + (double)x.y * z.y;
    im += (double)x.x * z.y - (double)x.y * z.x;
  }
  block_sum2(re, im);
  if (threadIdx.x == 0) {
    part[b * pstride + 2 * blockIdx.x] = re;
    part[b * pstride + 2 * blockIdx.x + 1] = im;
  }
}

template <typename T>
__global__ void k_copy(V2<T>* __restrict__ dst, const V2<T>* __restrict__ src, int64_t total) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

// ===========================================================================
// host launchers
// ===========================================================================
static inline int grid_for(int64_t work, int64_t cap = 1 << 20) {
  int64_t g = (work + 255) / 256;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (int)g;
}

template <typename T>
void add_prep(PrepJobs& J, const Sched& S, const DeviceTables& D, const void* ctab, const void* params,
              int64_t pstride, void* mtab, int64_t batch, hipStream_t st) {
  if (S.recipes.empty() || batch <= 0) return;
  // merged-diagonal (DG) recipes follow the base recipes; their widest group
  const int nrec = (int)S.recipes.size();
  int first_dg = nrec, dg_log = 0;
  for (int i = 0; i < nrec; ++i)
    if (S.recipes[i].kind < 0) {
      if (first_dg == nrec) first_dg = i;
      dg_log = std::max(dg_log, (int)S.recipes[i].R);
    }
  for (int64_t b0 = 0; b0 < batch;) {
    const int64_t nb = std::min(batch - b0, kMaxPrepItems - J.items);
    J.job[J.njobs++] = PrepJob{D.recipes, D.factors, params ? (const T*)params + b0 * pstride : nullptr, ctab,
                               (T*)mtab + b0 * S.mtab_size, pstride, (int64_t)S.mtab_size, 0, nb,
                               nrec, first_dg, dg_log, 0};
    J.items += nb;
    J.widest = std::max({J.widest, first_dg, (nrec - first_dg) << dg_log});
    if (J.njobs == kMaxPrepJobs || J.items == kMaxPrepItems) launch_prep<T>(J, st);
    b0 += nb;
  }
}

template <typename T>
void launch_prep(PrepJobs& J, hipStream_t st) {
  const int threads = J.widest > 512 && J.items <= 1024 ? 1024 : 256;
  int64_t blocks = 0;
  for (int q = 0; q < J.njobs; ++q) {
    PrepJob& p = J.job[q];
    const int wide = std::max(p.first_dg, (p.nrec - p.first_dg) << p.dg_log);
    while ((1 << p.wlog) < std::min(wide, threads)) ++p.wlog;
    p.block0 = blocks;
    blocks += ((p.batch << p.wlog) + threads - 1) / threads;
  }
  if (blocks) hipLaunchKernelGGL(k_prep<T>, dim3((unsigned)blocks), dim3(threads), 0, st, J);
  J = PrepJobs();
}

template <typename T>
void launch_init_zero(void* state, int n, int64_t batch, hipStream_t st) {
  const int64_t total = (1ll << n) * batch;
  hipLaunchKernelGGL(k_init_zero<T>, dim3(grid_for(total)), dim3(256), 0, st, (V2<T>*)state, total, 1ll << n);
}

template <typename T>
void launch_copy(void* dst, const void* src, int64_t total, hipStream_t st) {
  hipLaunchKernelGGL(k_copy<T>, dim3(grid_for(total)), dim3(256), 0, st, (V2<T>*)dst, (const V2<T>*)src, total);
}

template <typename T, bool DAG>
void launch_plain_gate(const DOp& op, const int32_t* ukbits_dev, const void* mtab, int64_t mstride,
                       const void* ctab, void* state, int n, int64_t batch, hipStream_t st) {
  const T* mt = (const T*)mtab;
  const T* ct = (const T*)ctab;
  V2<T>* s = (V2<T>*)state;
  const int64_t N = 1ll << n;
  switch (op.kind) {
    case OK_U1: case OK_R1: case OK_D1: case OK_X1:
      hipLaunchKernelGGL((k_plain1<T, 0, DAG>), dim3(grid_for(batch * (N >> 1))), dim3(256), 0, st, op, mt, mstride,
                         ct, (A2<T>*)s, N, n, batch);
      break;
    case OK_U2: case OK_D2: case OK_CX: case OK_CZ: case OK_SWAP:
      hipLaunchKernelGGL((k_plain2<T, 0, DAG>), dim3(grid_for(batch * (N >> 2))), dim3(256), 0, st, op, mt, mstride,
                         ct, (A2<T>*)s, N, n, batch);
      break;
    case OK_UK:
      if constexpr (std::is_same<T, float>::value) {
        if (op.nmem == 5 && (op.flags & OP_F_MFMA) && n >= 10) {
          const int64_t waves = batch * (N >> 10);
          const int blocks = (int)std::min<int64_t>((waves + 3) / 4, 1 << 20);
          hipLaunchKernelGGL((k_mfma_u5<DAG>), dim3(blocks), dim3(256), 0, st, op, ukbits_dev, ct, (float2*)s,
                             N, n, batch);
          break;
        }
      }
      switch (op.nmem) {
        case 3: hipLaunchKernelGGL((k_plaink<T, 3, DAG>), dim3(grid_for(batch * (N >> 3))), dim3(256), 0, st, op, ukbits_dev, ct, s, N, n, batch); break;
        case 4: hipLaunchKernelGGL((k_plaink<T, 4, DAG>), dim3(grid_for(batch * (N >> 4))), dim3(256), 0, st, op, ukbits_dev, ct, s, N, n, batch); break;
        case 5: hipLaunchKernelGGL((k_plaink<T, 5, DAG>), dim3(grid_for(batch * (N >> 5))), dim3(256), 0, st, op, ukbits_dev, ct, s, N, n, batch); break;
      }
      break;
    default: break;
  }
}

void allow_lds(const void* kern, size_t bytes) {
  if (bytes <= 65536) return;
  static std::mutex mu;
  static std::map<std::pair<int, const void*>, size_t> done;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return;
  std::lock_guard<std::mutex> lk(mu);
  size_t& d = done[{dev, kern}];
  if (bytes <= d) return;
  (void)hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  d = bytes;
}

template <typename T>
void launch_plain_adj(const DOp& op, const void* mtab, int64_t mstride, const void* ctab, const void* psi_in,
                      void* psi_out, const void* lam_in, void* lam_out, int64_t batch, int n, int slots, double* part,
                      int64_t pstride, hipStream_t st) {
  dim3 grid((unsigned)slots, (unsigned)batch);
  const int nq = (op.kind == OK_U1 || op.kind == OK_R1 || op.kind == OK_D1 || op.kind == OK_X1) ? 1 : 2;
  if (nq == 1)
    hipLaunchKernelGGL((k_plain_adj<T, 1>), grid, dim3(256), 0, st, op, (const T*)mtab, mstride, (const T*)ctab,
                       (const A2<T>*)psi_in, (A2<T>*)psi_out, (const A2<T>*)lam_in, (A2<T>*)lam_out,
                       (int64_t)1 << n, n, part, pstride);
  else
    hipLaunchKernelGGL((k_plain_adj<T, 2>), grid, dim3(256), 0, st, op, (const T*)mtab, mstride, (const T*)ctab,
                       (const A2<T>*)psi_in, (A2<T>*)psi_out, (const A2<T>*)lam_in, (A2<T>*)lam_out,
                       (int64_t)1 << n, n, part, pstride);
}

template <typename T>
void launch_plain_adj_uk(const DOp& op, const int32_t* ukbits_dev, const void* ctab, void* psi, void* lam,
                         int64_t batch, int n, hipStream_t st) {
  launch_plain_gate<T, true>(op, ukbits_dev, nullptr, 0, ctab, psi, n, batch, st);
  launch_plain_gate<T, true>(op, ukbits_dev, nullptr, 0, ctab, lam, n, batch, st);
}

template <typename T>
void launch_pauli(const DPGroup& G, const DPTerm* terms_dev, int n, const void* psi, void* out, int first,
                  const double* alpha, double* epart, int64_t estride, int64_t batch, bool energy, bool apply,
                  hipStream_t st) {
  dim3 grid((unsigned)G.nblk, (unsigned)batch);
  const V2<T>* p = (const V2<T>*)psi;
  V2<T>* o = (V2<T>*)out;
  const int64_t ss = 1ll << n;
  if (energy && apply)
    hipLaunchKernelGGL((k_pauli<T, true, true>), grid, dim3(256), 0, st, G, terms_dev, n, p, ss, o, first, alpha, epart, estride);
  else if (energy)
    hipLaunchKernelGGL((k_pauli<T, true, false>), grid, dim3(256), 0, st, G, terms_dev, n, p, ss, o, first, alpha, epart, estride);
  else
    hipLaunchKernelGGL((k_pauli<T, false, true>), grid, dim3(256), 0, st, G, terms_dev, n, p, ss, o, first, alpha, epart, estride);
}

template <typename T>
void launch_inner(const void* a, const void* c, int n, int64_t batch, int nblk, double* part, int64_t pstride,
                  hipStream_t st) {
  hipLaunchKernelGGL(k_inner<T>, dim3((unsigned)nblk, (unsigned)batch), dim3(256), 0, st, (const V2<T>*)a,
                     (const V2<T>*)c, n, (int64_t)1 << n, part, pstride);
}

void launch_sum_slots(const double* part, int64_t bstride, int64_t nslots, int ncomp, double* out, int64_t batch,
                      hipStream_t st) {
  const int threads = nslots > 1024 ? 1024 : nslots > 64 ? 256 : 64;
  hipLaunchKernelGGL(k_sum_slots, dim3((unsigned)std::min(batch, kMaxLaunchThreads / threads)), dim3(threads), 0, st,
                     part, bstride, nslots, ncomp, out, batch);
}

void launch_reduce_gop(const double* part, int64_t pstride, int64_t nslots, const int32_t* gop_list, int gop_single,
                       int ngop_pass, double* gsum, int ngop, int64_t batch, hipStream_t st) {
  hipLaunchKernelGGL(k_reduce_gop, dim3((unsigned)ngop_pass, (unsigned)batch), dim3(256), 0, st, part, pstride,
                     nslots, gop_list, gop_single, gsum, ngop);
}

void launch_finish(const double* epart, int64_t nslots, double* energy, const double* part, const DGopSum* gs, int ngop,
                   const int32_t* p_ptr, const int32_t* p_gops, const double* gfac, double mult, double* grad,
                   int nparams, int max_slots, int64_t batch, hipStream_t st) {
  const int64_t total = grad ? (int64_t)nparams * batch : 0, nen = epart ? std::min<int64_t>(batch, 1 << 16) : 0;
  if (total + nen == 0) return;
  const bool one = !gs || max_slots == 1;
  const int64_t blocks = std::min<int64_t>((total + (one ? 255 : 3)) / (one ? 256 : 4), 1 << 20);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)(nen + blocks)), dim3(256), 0, st, epart, nslots, nen, energy, part, gs,
                       ngop, p_ptr, p_gops, gfac, mult, grad, nparams, batch);
  };
  if (one) go(k_finish<1>);
  else go(k_finish<64>);
}

// ---------------------------------------------------------------------------
// Measurement: probability vector (basecircuit.py:510-524) and
// qubit-by-qubit conditional measurement (measure_jit,
// basecircuit.py:371-445).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void k_probability(const V2<T>* __restrict__ psi, T* __restrict__ out, int64_t total) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const V2<T> x = psi[i];
    out[i] = x.x * x.x + x.y * x.y;
  }
}

// partial sums of |psi_i|^2 over the indices that agree with the outcomes
// fixed so far (fixval[b] on the fixed bits), split by index bit M.bit; the
// free bits are enumerated by depositing a counter into M.run.
// grid (nblk, batch); part[b][blk][2]
template <typename T>
__global__ void __launch_bounds__(256) k_measure_partial(const V2<T>* __restrict__ psi, int64_t sstride,
                                                         MeasureStep M, const uint64_t* __restrict__ fixval,
                                                         double* __restrict__ part) {
  const int64_t b = blockIdx.y;
  const V2<T>* s = psi + b * sstride;
  const uint64_t fv = M.first ? 0ull : fixval[b];
  const int64_t total = 1ll << M.nfree;
  double a0 = 0.0, a1 = 0.0;
  for (int64_t m = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; m < total; m += (int64_t)gridDim.x * blockDim.x) {
    uint64_t i = fv;
    for (int r = 0; r < M.nrun; ++r) {
      const int src = M.run[r] & 0xff, len = (M.run[r] >> 8) & 0xff, dst = M.run[r] >> 16;
      i |= (((uint64_t)m >> src) & ((1ull << len) - 1)) << dst;
    }
    const V2<T> x = s[i];
    const double p = (double)x.x * x.x + (double)x.y * x.y;
    if ((i >> M.bit) & 1) a1 += p;
    else a0 += p;
  }
  block_sum2(a0, a1);
  if (threadIdx.x == 0) {
    part[(b * gridDim.x + blockIdx.x) * 2] = a0;
    part[(b * gridDim.x + blockIdx.x) * 2 + 1] = a1;
  }
}

// measure_jit's decision for step k (basecircuit.py:419-431): pu = p0 / p,
// outcome 1 iff status - pu + eps > 0, p *= pu or (1 - pu); one block per
// batch item
__global__ void __launch_bounds__(256) k_measure_decide(const double* __restrict__ part, int nblk, int k, int nmeas,
                                                        int bit, const double* __restrict__ status,
                                                        uint64_t* __restrict__ fixval, double* __restrict__ prob,
                                                        double* __restrict__ outcome) {
  const int64_t b = blockIdx.x;
  double a0 = 0.0, a1 = 0.0;
  for (int i = threadIdx.x; i < nblk; i += blockDim.x) a0 += part[(b * nblk + i) * 2];
  block_sum2(a0, a1);
  if (threadIdx.x == 0) {
    const double p = k == 0 ? 1.0 : prob[b];
    const double pu = a0 / p;
    const double r = status[b * nmeas + k];
    const double eps = 0.31415926 * 1e-12;
    const int o = (r - pu + eps > 0.0) ? 1 : 0;
    prob[b] = p * (o ? 1.0 - pu : pu);
    fixval[b] = (k == 0 ? 0ull : fixval[b]) | ((uint64_t)o << bit);
    outcome[b * nmeas + k] = (double)o;
  }
}

template <typename T>
void launch_probability(const void* psi, void* out, int64_t total, hipStream_t st) {
  hipLaunchKernelGGL(k_probability<T>, dim3(grid_for(total)), dim3(256), 0, st, (const V2<T>*)psi, (T*)out, total);
}

template <typename T>
void launch_measure_step(const void* psi, int n, int64_t batch, const MeasureStep& M, int k, int nmeas,
                         const double* status, uint64_t* fixval, double* prob, double* outcome, double* part,
                         int nblk, hipStream_t st) {
  hipLaunchKernelGGL(k_measure_partial<T>, dim3((unsigned)nblk, (unsigned)batch), dim3(256), 0, st,
                     (const V2<T>*)psi, (int64_t)1 << n, M, (const uint64_t*)fixval, part);
  hipLaunchKernelGGL(k_measure_decide, dim3((unsigned)batch), dim3(256), 0, st, (const double*)part, nblk, k, nmeas,
                     M.bit, status, fixval, prob, outcome);
}

// ---------------------------------------------------------------------------
// Sparse form of a Pauli sum (PauliStringSum2COO / ps2coo_core,
// quantum.py:1304-1485).
// ---------------------------------------------------------------------------
// entry t * N + y of term t (group g): row y, column y ^ flip,
// value w (-i)^ny (-1)^popc(y & yz); grid-stride over nterms * N
template <typename T>
__global__ void k_pauli_coo(const DPGroup* __restrict__ groups, int ngroups, const DPTerm* __restrict__ terms,
                            int n, int64_t* __restrict__ rows, int64_t* __restrict__ cols, V2<T>* __restrict__ vals,
                            int64_t total) {
  const int64_t N = 1ll << n;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    const int t = (int)(e >> n);
    const uint64_t y = (uint64_t)(e & (N - 1));
    int g = 0;
    while (g + 1 < ngroups && groups[g + 1].t0 <= t) ++g;
    const DPTerm tm = terms[t];
    const double sg = (__popcll(y & tm.yz) & 1) ? -tm.w : tm.w;
    double re = 0.0, im = 0.0;
    switch (tm.ny & 3) {  // (-i)^ny
      case 0: re = sg; break;
      case 1: im = -sg; break;
      case 2: re = -sg; break;
      default: im = sg; break;
    }
    rows[e] = (int64_t)y;
    cols[e] = (int64_t)(y ^ groups[g].flip);
    vals[e] = mk<T>((T)re, (T)im);
  }
}

template <typename T>
void launch_pauli_coo(const DPGroup* groups, int ngroups, const DPTerm* terms, int n, int64_t nterms, int64_t* rows,
                      int64_t* cols, void* vals, hipStream_t st) {
  const int64_t total = nterms << n;
  hipLaunchKernelGGL(k_pauli_coo<T>, dim3(grid_for(total)), dim3(256), 0, st, groups, ngroups, terms, n, rows, cols,
                     (V2<T>*)vals, total);
}

// explicit instantiations used by engine.cpp
#define TCM_INST(T)                                                                                            \
  template void add_prep<T>(PrepJobs&, const Sched&, const DeviceTables&, const void*, const void*, int64_t,     \
                            void*, int64_t, hipStream_t);                                                        \
  template void launch_prep<T>(PrepJobs&, hipStream_t);                                                           \
  template void launch_init_zero<T>(void*, int, int64_t, hipStream_t);                                         \
  template void launch_copy<T>(void*, const void*, int64_t, hipStream_t);                                      \
  template void launch_plain_gate<T, false>(const DOp&, const int32_t*, const void*, int64_t, const void*,    \
                                            void*, int, int64_t, hipStream_t);                                 \
  template void launch_plain_gate<T, true>(const DOp&, const int32_t*, const void*, int64_t, const void*,     \
                                           void*, int, int64_t, hipStream_t);                                  \
  template void launch_plain_adj<T>(const DOp&, const void*, int64_t, const void*, const void*, void*,        \
                                    const void*, void*, int64_t, int, int, double*, int64_t, hipStream_t);     \
  template void launch_plain_adj_uk<T>(const DOp&, const int32_t*, const void*, void*, void*, int64_t, int,   \
                                       hipStream_t);                                                           \
  template void launch_pauli<T>(const DPGroup&, const DPTerm*, int, const void*, void*, int, const double*,   \
                                double*, int64_t, int64_t, bool, bool, hipStream_t);                           \
  template void launch_inner<T>(const void*, const void*, int, int64_t, int, double*, int64_t, hipStream_t); \
  template void launch_probability<T>(const void*, void*, int64_t, hipStream_t);                               \
  template void launch_measure_step<T>(const void*, int, int64_t, const MeasureStep&, int, int, const double*,  \
                                       uint64_t*, double*, double*, double*, int, hipStream_t);                \
  template void launch_pauli_coo<T>(const DPGroup*, int, const DPTerm*, int, int64_t, int64_t*, int64_t*, void*,  \
                                    hipStream_t);

TCM_INST(float)
TCM_INST(double)

}  // namespace tcm

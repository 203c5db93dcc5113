// HIP kernel of libtcm for CDNA4 (gfx950): the LDS-tiled Pauli pass of sums
// that are not compiled (any n below the pass compiler's size rule).
//
// For every amplitude a of a tile
//   h[a] = sum_groups psi[a ^ flip] sum_terms w (-i)^ny (-1)^popc(a & yz)
// (the index rule of ps2coo_core, quantum.py:1461-1485), with the partner
// read from LDS; energy += conj(psi[a]) h[a] in fp64 and, when APPLY,
// lam_out[a] = lam_in[a] (or 0) + alpha h[a].
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"
#include "regops.h"

namespace tcm {

namespace {

// a staged term: weight with the block-uniform part of its sign, Y/Z mask
// inside the tile
template <typename T>
struct Rec {
  T w;
  uint32_t yz;
};

__device__ __forceinline__ float flip_sign(float x, uint32_t odd) {
  return __uint_as_float(__float_as_uint(x) ^ (odd << 31));
}
__device__ __forceinline__ double flip_sign(double x, uint32_t odd) {
  return __hiloint2double(__double2hiint(x) ^ (int)(odd << 31), __double2loint(x));
}

// (a, b) summed over the block in fp64, valid in thread 0
__device__ __forceinline__ void sum_block(double& a, double& b) {
  __shared__ double red[2][16];
  for (int off = 32; off > 0; off >>= 1) {
    a += __shfl_xor(a, off, 64);
    b += __shfl_xor(b, off, 64);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    red[0][w] = a;
    red[1][w] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    for (int i = 1; i < (int)(blockDim.x >> 6); ++i) {
      a += red[0][i];
      b += red[1][i];
    }
}

}  // namespace

// One block per tile, 2^LE amplitudes per thread at tile positions
// it << tl | tid.  The sign of a term splits into a block part (bits outside
// the tile), a thread part and an element part, so a term costs a few
// instructions per thread, not per amplitude: terms of a group with the same
// element pattern are summed first, and the 2^LE signed copies of that sum
// are built by doubling (one multiplication by +-1 each).  What is left per
// amplitude and group is one LDS read and two multiply-adds.  The group and
// term descriptors of a chunk are staged in LDS by all threads at once: read
// in the group loop they would be one cold scalar load after another, about
// 1 us each.  Measured, 200 strings on 4 x 2^18 amplitudes, complex64: energy
// and H psi 119 us (one launch of 32 us, six of 13 us); 4668 us when
// descriptors were read from memory and signs formed per amplitude.  What
// bounds it now is the launches and, in each, the chain of LDS reads per
// group at two waves per SIMD.
template <typename T, int LE, bool ENERGY, bool APPLY>
__global__ void __launch_bounds__(1024) k_pauli_tile(PauliTileArgs S, const DPChunk* __restrict__ chunks,
                                                     const DPGroupS* __restrict__ groups,
                                                     const DPTermS* __restrict__ terms,
                                                     const uint32_t* __restrict__ runoff,
                                                     const V2<T>* __restrict__ psi, const V2<T>* lam_in,
                                                     V2<T>* lam_out, int64_t sstride,
                                                     const double* __restrict__ alpha,
                                                     double* __restrict__ epart, int64_t estride) {
  constexpr int E = 1 << LE;
  const PauliTileArg& A = S.p[blockIdx.y];
  extern __shared__ __align__(16) unsigned char smem[];
  V2<T>* tile = reinterpret_cast<V2<T>*>(smem);
  Rec<T>* recs = reinterpret_cast<Rec<T>*>(tile + (1 << S.k));
  DPGroupS* grps = reinterpret_cast<DPGroupS*>(recs + kPauliChunk);
  const int L = A.L, tl = S.k - LE, nbl = S.nblk_log;
  // tiles below 64 threads: the rest of the wave repeats them, unstored
  const uint32_t tid = threadIdx.x & ((1u << tl) - 1);
  const bool act = threadIdx.x < (1u << tl);
  const uint64_t blk = blockIdx.x & ((1ull << nbl) - 1);
  const uint64_t b = (uint64_t)blockIdx.x >> nbl;
  uint64_t base = 0, m = A.bmask;
  for (int i = 0; i < nbl; ++i) {
    const uint64_t low = m & (~m + 1);
    if ((blk >> i) & 1) base |= low;
    m ^= low;
  }
  const uint32_t* ro = runoff + A.runoff0;
  const uint32_t dlo = run_dep(ro, L, tid);
  {
    const V2<T>* s = psi + b * sstride + base;
    V2<T> r[E];
#pragma unroll
    for (int it = 0; it < E; ++it) r[it] = s[run_dep(ro, L, (uint32_t)it << tl) + dlo];
#pragma unroll
    for (int it = 0; it < E; ++it) tile[((uint32_t)it << tl) | tid] = r[it];
  }
  T hr[E], hi[E];
#pragma unroll
  for (int it = 0; it < E; ++it) hr[it] = hi[it] = T(0);
  for (int ch = 0; ch < A.nc; ++ch) {
    const DPChunk C = chunks[A.c0 + ch];
    if (ch) __syncthreads();  // the chunk before has been read
    for (int i = threadIdx.x; i < C.nt; i += blockDim.x) {
      const DPTermS t = terms[C.t0 + i];
      recs[i] = Rec<T>{flip_sign((T)t.w, __popcll(base & t.yz_g) & 1u), t.yz_t};
    }
    for (int i = threadIdx.x; i < C.ng; i += blockDim.x) grps[i] = groups[C.g0 + i];
    __syncthreads();
    int t = 0;
    for (int g = 0; g < C.ng; ++g) {
      const DPGroupS G = grps[g];
      const uint32_t flip = __builtin_amdgcn_readfirstlane(G.flip_t);
      const uint32_t cnt = __builtin_amdgcn_readfirstlane(G.cnt);
      const uint32_t a0 = tid ^ flip;
      V2<T> q[E];
#pragma unroll
      for (int it = 0; it < E; ++it) q[it] = tile[a0 ^ ((uint32_t)it << tl)];
      // the real-coefficient terms, then the imaginary ones
#pragma unroll
      for (int im = 0; im < 2; ++im) {
        const int end = t + (int)(im ? cnt >> 16 : cnt & 0xffffu);
        if (t == end) continue;
        T c[E];
#pragma unroll
        for (int it = 0; it < E; ++it) c[it] = T(0);
        while (t < end) {
          // a run of terms with one element pattern
          uint32_t yz = __builtin_amdgcn_readfirstlane(recs[t].yz);
          const uint32_t pat = yz >> tl;
          T d[E];
          d[0] = flip_sign(recs[t].w, __popc(tid & yz) & 1u);
          for (++t; t < end; ++t) {
            yz = __builtin_amdgcn_readfirstlane(recs[t].yz);
            if ((yz >> tl) != pat) break;
            d[0] += flip_sign(recs[t].w, __popc(tid & yz) & 1u);
          }
#pragma unroll
          for (int e = 0; e < LE; ++e) {
            const T f = (pat >> e) & 1u ? T(-1) : T(1);
#pragma unroll
            for (int j = 0; j < (1 << e); ++j) d[j | (1 << e)] = d[j] * f;
          }
#pragma unroll
          for (int it = 0; it < E; ++it) c[it] += d[it];
        }
        if (im == 0) {
#pragma unroll
          for (int it = 0; it < E; ++it) {
            hr[it] += c[it] * q[it].x;
            hi[it] += c[it] * q[it].y;
          }
        } else {
#pragma unroll
          for (int it = 0; it < E; ++it) {
            hr[it] -= c[it] * q[it].y;
            hi[it] += c[it] * q[it].x;
          }
        }
      }
    }
  }
  if constexpr (APPLY) {
    if (act) {
      const double al = alpha ? alpha[b] : 1.0;
      const uint64_t ob = b * sstride + base + dlo;
#pragma unroll
      for (int it = 0; it < E; ++it) {
        const uint64_t off = ob + run_dep(ro, L, (uint32_t)it << tl);
        V2<T> o;
        o.x = o.y = T(0);
        if (lam_in) o = lam_in[off];
        o.x = (T)(o.x + al * hr[it]);
        o.y = (T)(o.y + al * hi[it]);
        lam_out[off] = o;
      }
    }
  }
  if constexpr (ENERGY) {
    double er = 0.0, ei = 0.0;
    if (act) {
#pragma unroll
      for (int it = 0; it < E; ++it) {
        const V2<T> p = tile[((uint32_t)it << tl) | tid];
        er += (double)p.x * hr[it] + (double)p.y * hi[it];
        ei += (double)p.x * hi[it] - (double)p.y * hr[it];
      }
    }
    sum_block(er, ei);
    if (threadIdx.x == 0) {
      epart[b * estride + 2 * (A.slot0 + blk)] = er;
      epart[b * estride + 2 * (A.slot0 + blk) + 1] = ei;
    }
  }
}

template <typename T, int LE, bool ENERGY, bool APPLY>
static void launch_le(const PauliTileArgs& A, int np, const PauliTileTables& D, const void* psi, const void* lam_in,
                      void* lam_out, int n, const double* alpha, double* epart, int64_t estride, int64_t batch,
                      hipStream_t st) {
  const size_t lds = (sizeof(V2<T>) << A.k) + kPauliChunk * (sizeof(Rec<T>) + sizeof(DPGroupS));
  allow_lds((const void*)k_pauli_tile<T, LE, ENERGY, APPLY>, lds);
  const unsigned threads = std::max(64u, 1u << (A.k - LE));
  // all states at once unless they are too many threads
  const int64_t part = std::max<int64_t>(1, (kMaxLaunchThreads / threads) >> A.nblk_log);
  for (int64_t b0 = 0; b0 < batch; b0 += part) {
    const int64_t nb = std::min(part, batch - b0), o = b0 << n;
    hipLaunchKernelGGL((k_pauli_tile<T, LE, ENERGY, APPLY>), dim3((unsigned)(nb << A.nblk_log), (unsigned)np),
                       dim3(threads), lds, st, A, (const DPChunk*)D.chunks, (const DPGroupS*)D.groups,
                       (const DPTermS*)D.terms, (const uint32_t*)D.runoff, (const V2<T>*)psi + o,
                       lam_in ? (const V2<T>*)lam_in + o : nullptr, lam_out ? (V2<T>*)lam_out + o : nullptr,
                       (int64_t)1 << n, alpha ? alpha + b0 : nullptr, epart ? epart + b0 * estride : nullptr, estride);
  }
}

template <typename T>
void launch_pauli_tile(const DPPass* P, int np, const PauliTileTables& D, const void* psi, const void* lam_in,
                       void* lam_out, int n, const double* alpha, double* epart, int64_t estride, int64_t batch,
                       bool energy, bool apply, hipStream_t st) {
  PauliTileArgs A{};
  A.k = P->k;
  A.nblk_log = P->nblk_log;
  for (int q = 0; q < np; ++q) {
    PauliTileArg& a = A.p[q];
    a.L = P[q].L;
    a.runoff0 = P[q].runoff0;
    a.slot0 = P[q].slot0;
    a.c0 = P[q].c0;
    a.nc = P[q].nc;
    for (int i = 0; i < P[q].nblk_log; ++i) a.bmask |= 1ull << P[q].blk_bits[i];
  }
  // 8 amplitudes per thread; 4 where the tile would not fill a wave, 16 for
  // the complex64 tiles of 2^14.  4, 8 and 16 run alike in complex64 (1049,
  // 1032, 1036 us for a step over 10 to 18 qubits); in complex128 16 spill
  // (18-qubit energy and gradient 1095 us against 983 with 4 and 986 with 8)
  const int le = A.k < 9 ? 2 : A.k < 14 ? 3 : 4;
#define TCM_PT(LE)                                                                                                  \
  do {                                                                                                              \
    if (energy && apply)                                                                                            \
      launch_le<T, LE, true, true>(A, np, D, psi, lam_in, lam_out, n, alpha, epart, estride, batch, st);            \
    else if (energy)                                                                                                \
      launch_le<T, LE, true, false>(A, np, D, psi, lam_in, lam_out, n, alpha, epart, estride, batch, st);           \
    else                                                                                                            \
      launch_le<T, LE, false, true>(A, np, D, psi, lam_in, lam_out, n, alpha, epart, estride, batch, st);           \
  } while (0)
  if (le == 2) TCM_PT(2);
  else if (le == 3) TCM_PT(3);
  else if constexpr (sizeof(T) == 4) TCM_PT(4);
#undef TCM_PT
}

#define TCM_PT_INST(T)                                                                                               \
  template void launch_pauli_tile<T>(const DPPass*, int, const PauliTileTables&, const void*, const void*, void*,    \
                                     int, const double*, double*, int64_t, int64_t, bool, bool, hipStream_t);
TCM_PT_INST(float)
TCM_PT_INST(double)

}  // namespace tcm

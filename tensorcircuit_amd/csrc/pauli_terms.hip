// HIP kernels of libtcm for CDNA4 (gfx950), many Pauli strings of one state
// kept apart:
//  - per-term expectations  E[b][t] = w_t <psi_b|P_t|psi_b>  (fp64) behind
//    any_measurements / parameterized_local_measurements over many structures
//    at once (templates/measurements.py:18-153);
//  - weighted applications  out_b = sum_t a[b][t] w_t P_t psi_b, the
//    vector-Jacobian product of those expectations.
//
// Pauli action (index rule of ps2coo_core, quantum.py:1461-1485):
//   (P psi)[a] = (-i)^ny (-1)^popcount(a & yz) psi[a ^ flip].
// State layout: [batch][2^n] complex, qubit 0 = most significant index bit.
//
// Two ways for each, chosen by the number of strings and amplitudes (each_term,
// each_term_apply): straight from memory, a string or 16 bytes at a time, or
// by tiles of 2^k consecutive amplitudes held in LDS, 2^LE per thread at
// positions it << tl | tid, with the strings sorted by flip mask (DPGroupX,
// DPTermX): a partner whose flip stays inside the tile is an LDS read, one
// outside it a coalesced read of another tile; conj(psi) psi' is formed once
// per flip mask, and the sign of a string splits into block, thread and
// element parts.  59 strings of a 20-qubit complex64 state: 67 us from memory
// (8 bytes at a time), 25 us by tiles; applied, 76 and 30 us, bound by their
// issue of 64-bit operations and LDS reads at two waves per SIMD.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"
#include "regops.h"

namespace tcm {

namespace {

__device__ __forceinline__ uint32_t first_lane(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ double with_sign(double x, uint32_t odd) {
  return __hiloint2double(__double2hiint(x) ^ (int)(odd << 31), __double2loint(x));
}

constexpr int kRow = 66;  // a string's 64 lane values, padded off its banks

// lane values of one wave, summed four strings at a time: each 16-lane row
// takes one string (16 lanes x 4 values)
struct TermSink {
  double* buf;  // [4][kRow]
  double* acc;  // [string][wave]
  int wv, nw, lane, cnt;
  bool act;
  __device__ __forceinline__ void flush(int first) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int q = lane >> 4;
    const double* r = buf + q * kRow + (lane & 15) * 4;
    double x = (r[0] + r[1]) + (r[2] + r[3]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    x += dpp_shr<0x111>(x);
    x += dpp_shr<0x112>(x);
    x += dpp_shr<0x114>(x);
    x += dpp_shr<0x118>(x);
    if ((lane & 15) == 15 && first + q < cnt) acc[(first + q) * nw + wv] += x;
  }
  __device__ __forceinline__ void push(double x) {
    buf[(cnt & 3) * kRow + lane] = act ? x : 0.0;
    ++cnt;
    if ((cnt & 3) == 0) flush(cnt - 4);
  }
  __device__ __forceinline__ void finish() {
    if (cnt & 3) flush(cnt & ~3);
  }
};

// the tile's amplitudes flipped by `flip`: from LDS, or from another tile
template <typename T, int E>
__device__ __forceinline__ void partners(V2<T>* q, const V2<T>* tile, const V2<T>* s, uint32_t base, uint32_t flip,
                                         int k, int tl, uint32_t tid) {
  const uint32_t hi = flip >> k << k, a0 = tid ^ (flip ^ hi);
  if (hi) {
    const V2<T>* o = s + (base ^ hi);
#pragma unroll
    for (int it = 0; it < E; ++it) q[it] = o[a0 ^ ((uint32_t)it << tl)];
  } else {
#pragma unroll
    for (int it = 0; it < E; ++it) q[it] = tile[a0 ^ ((uint32_t)it << tl)];
  }
}

}  // namespace

// part[b][string][blk]: sums over the tiles blk, blk + nblk, ... of chunk
// blockIdx.y's strings.  The expectation of a Hermitian string is real: only
// Re(conj(psi) psi') of strings with an even number of Y, or Im of the odd
// ones, is summed.  grid (nblk, chunks, batch)
template <typename T, int LE>
__global__ void __launch_bounds__(512) k_pauli_terms(const DPChunk* __restrict__ chunks,
                                                     const DPGroupX* __restrict__ groups,
                                                     const DPTermX* __restrict__ terms, int n, int k, int nterms,
                                                     const V2<T>* __restrict__ psi, double* __restrict__ part) {
  constexpr int E = 1 << LE;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tl = k - LE, nw = blockDim.x >> 6, nblk = gridDim.x;
  V2<T>* tile = reinterpret_cast<V2<T>*>(smem);
  double* acc = reinterpret_cast<double*>(tile + (1 << k));
  double* buf = acc + kTermsChunk * nw;
  uint32_t* recs = reinterpret_cast<uint32_t*>(buf + 4 * kRow * nw);
  DPGroupX* grps = reinterpret_cast<DPGroupX*>(recs + kTermsChunk);
  const uint32_t tid = threadIdx.x & ((1u << tl) - 1);
  const int64_t b = blockIdx.z;
  const V2<T>* s = psi + (b << n);
  const DPChunk C = chunks[blockIdx.y];
  for (int i = threadIdx.x; i < C.nt; i += blockDim.x) recs[i] = terms[C.t0 + i].yz;
  for (int i = threadIdx.x; i < C.ng; i += blockDim.x) grps[i] = groups[C.g0 + i];
  for (int i = threadIdx.x; i < C.nt * nw; i += blockDim.x) acc[i] = 0.0;
  TermSink sink;
  sink.wv = threadIdx.x >> 6;
  sink.nw = nw;
  sink.lane = threadIdx.x & 63;
  sink.act = threadIdx.x < (1u << tl);
  sink.acc = acc;
  sink.buf = buf + sink.wv * 4 * kRow;
  const uint32_t ntiles = 1u << (n - k);
  for (uint32_t t = blockIdx.x; t < ntiles; t += nblk) {
    const uint32_t base = t << k;
    V2<T> r[E];
#pragma unroll
    for (int it = 0; it < E; ++it) r[it] = s[base + (((uint32_t)it << tl) | tid)];
    __syncthreads();  // the tile before has been read
#pragma unroll
    for (int it = 0; it < E; ++it) tile[((uint32_t)it << tl) | tid] = r[it];
    __syncthreads();
    const uint32_t me = base | tid;
    sink.cnt = 0;
    int e = 0;
    for (int g = 0; g < C.ng; ++g) {
      const uint32_t flip = first_lane(grps[g].flip), cnt = first_lane(grps[g].cnt);
      V2<T> q[E];
      partners<T, E>(q, tile, s, base, flip, k, tl, tid);
#pragma unroll
      for (int im = 0; im < 2; ++im) {
        const int end = e + (int)(im ? cnt >> 16 : cnt & 0xffffu);
        if (e == end) continue;
        double c[E];
#pragma unroll
        for (int it = 0; it < E; ++it)
          c[it] = im ? (double)r[it].y * q[it].x - (double)r[it].x * q[it].y
                     : (double)r[it].x * q[it].x + (double)r[it].y * q[it].y;
        uint32_t pat = ~0u;
        double sum = 0.0;
        for (; e < end; ++e) {
          const uint32_t yz = first_lane(recs[e]);
          const uint32_t pe = (yz >> tl) & (E - 1);
          if (pe != pat) {  // a new element pattern: sum_it (-1)^popc(it & pat) c[it]
            pat = pe;
            double v[E];
#pragma unroll
            for (int it = 0; it < E; ++it) v[it] = c[it];
#pragma unroll
            for (int l = 0; l < LE; ++l) {
              const double f = (pat >> l) & 1u ? -1.0 : 1.0;
#pragma unroll
              for (int it = 0; it < (E >> (l + 1)); ++it) v[it] = v[2 * it] + f * v[2 * it + 1];
            }
            sum = v[0];
          }
          sink.push(with_sign(sum, __popc(me & (yz & ~((uint32_t)(E - 1) << tl))) & 1u));
        }
      }
    }
    sink.finish();
  }
  __syncthreads();
  for (int i = threadIdx.x; i < C.nt; i += blockDim.x) {
    double x = 0.0;
    for (int w = 0; w < nw; ++w) x += acc[i * nw + w];
    const DPTermX tm = terms[C.t0 + i];
    part[(b * nterms + tm.idx) * nblk + blockIdx.x] = tm.w * x;
  }
}

// out[b][t] = the sum of the nblk partials of (b, t) and a zero imaginary part
// (NaN where the sum is not finite); one wave per (b, t) in turn
__global__ void __launch_bounds__(64) k_pauli_terms_sum(const double* __restrict__ part, int nblk, int64_t total,
                                                        double* __restrict__ out) {
  for (int64_t bt = blockIdx.x; bt < total; bt += gridDim.x) {
    double a = 0.0;
    for (int i = threadIdx.x; i < nblk; i += 64) a += part[bt * nblk + i];
    for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
    if (threadIdx.x == 0) {
      out[2 * bt] = a;
      out[2 * bt + 1] = a - a;
    }
  }
}

// out_b[a] = sum_t wts[b][t] w_t (P_t psi_b)[a] in fp64, stored in T; the
// blocks walk the ntiles tiles of the batch.  Strings of zero weight are left out.
template <typename T, int LE>
__global__ void __launch_bounds__(512) k_pauli_terms_apply(const DPChunk* __restrict__ chunks, int nchunks,
                                                           const DPGroupX* __restrict__ groups,
                                                           const DPTermX* __restrict__ terms, int n, int k, int nterms,
                                                           const V2<T>* __restrict__ psi, V2<T>* __restrict__ out,
                                                           const double* __restrict__ wts, int64_t ntiles) {
  constexpr int E = 1 << LE;
  struct Rec {
    double w;
    uint32_t yz, used;
  };
  extern __shared__ __align__(16) unsigned char smem[];
  const int tl = k - LE;
  V2<T>* tile = reinterpret_cast<V2<T>*>(smem);
  Rec* recs = reinterpret_cast<Rec*>(tile + (1 << k));
  DPGroupX* grps = reinterpret_cast<DPGroupX*>(recs + kTermsChunk);
  const uint32_t tid = threadIdx.x & ((1u << tl) - 1);
  for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const uint32_t base = (uint32_t)(t & (((int64_t)1 << (n - k)) - 1)) << k;
    const int64_t b = t >> (n - k);
    const V2<T>* s = psi + (b << n);
    {
      V2<T> r[E];
#pragma unroll
      for (int it = 0; it < E; ++it) r[it] = s[base + (((uint32_t)it << tl) | tid)];
      if (t != blockIdx.x) __syncthreads();  // the tile before has been read
#pragma unroll
      for (int it = 0; it < E; ++it) tile[((uint32_t)it << tl) | tid] = r[it];
    }
    double hr[E], hi[E];
#pragma unroll
    for (int it = 0; it < E; ++it) hr[it] = hi[it] = 0.0;
    for (int ch = 0; ch < nchunks; ++ch) {
      const DPChunk C = chunks[ch];
      if (ch) __syncthreads();  // the chunk before has been read
      for (int i = threadIdx.x; i < C.nt; i += blockDim.x) {
        const DPTermX tm = terms[C.t0 + i];
        const double w = tm.w * wts[b * nterms + tm.idx];
        recs[i] = Rec{with_sign(w, __popc(base & tm.yz) & 1u), tm.yz, w != 0.0 ? 1u : 0u};
      }
      for (int i = threadIdx.x; i < C.ng; i += blockDim.x) grps[i] = groups[C.g0 + i];
      __syncthreads();
      int e = 0;
      for (int g = 0; g < C.ng; ++g) {
        const uint32_t flip = first_lane(grps[g].flip), cnt = first_lane(grps[g].cnt);
        V2<T> q[E];
        partners<T, E>(q, tile, s, base, flip, k, tl, tid);
#pragma unroll
        for (int im = 0; im < 2; ++im) {
          const int end = e + (int)(im ? cnt >> 16 : cnt & 0xffffu);
          if (e == end) continue;
          double c[E];
#pragma unroll
          for (int it = 0; it < E; ++it) c[it] = 0.0;
          uint32_t any = 0;
          while (e < end) {
            // a run of strings with one element pattern
            uint32_t yz = first_lane(recs[e].yz);
            const uint32_t pat = (yz >> tl) & (E - 1);
            double d[E];
            d[0] = 0.0;
            for (; e < end; ++e) {
              yz = first_lane(recs[e].yz);
              if (((yz >> tl) & (E - 1)) != pat) break;
              if (!first_lane(recs[e].used)) continue;
              any = 1;
              d[0] += with_sign(recs[e].w, __popc(tid & yz & ~((uint32_t)(E - 1) << tl)) & 1u);
            }
#pragma unroll
            for (int l = 0; l < LE; ++l) {
              const double f = (pat >> l) & 1u ? -1.0 : 1.0;
#pragma unroll
              for (int j = 0; j < (1 << l); ++j) d[j | (1 << l)] = d[j] * f;
            }
#pragma unroll
            for (int it = 0; it < E; ++it) c[it] += d[it];
          }
          if (!any) continue;
          if (im == 0) {
#pragma unroll
            for (int it = 0; it < E; ++it) {
              hr[it] += c[it] * (double)q[it].x;
              hi[it] += c[it] * (double)q[it].y;
            }
          } else {
#pragma unroll
            for (int it = 0; it < E; ++it) {
              hr[it] -= c[it] * (double)q[it].y;
              hi[it] += c[it] * (double)q[it].x;
            }
          }
        }
      }
    }
    if (threadIdx.x < (1u << tl)) {
#pragma unroll
      for (int it = 0; it < E; ++it) {
        V2<T> o;
        o.x = (T)hr[it];
        o.y = (T)hi[it];
        out[(b << n) + base + (((uint32_t)it << tl) | tid)] = o;
      }
    }
  }
}

// part as k_pauli_terms, blocks of one string each and no tiles: both
// amplitudes from memory.  grid (nblk, nterms, batch)
template <typename T>
__global__ void __launch_bounds__(256) k_pauli_terms_each(const DPTermX* __restrict__ terms, int n, int nterms,
                                                          const V2<T>* __restrict__ psi, double* __restrict__ part) {
  __shared__ double red[4];
  const DPTermX tm = terms[blockIdx.y];
  const int64_t b = blockIdx.z;
  const V2<T>* s = psi + (b << n);
  const uint64_t N = 1ull << n;
  double x = 0.0;
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < N; i += gridDim.x * 256ull) {
    const uint32_t a = (uint32_t)i;
    const V2<T> p = s[a], q = s[a ^ tm.flip];
    const double c = tm.odd ? (double)p.y * q.x - (double)p.x * q.y : (double)p.x * q.x + (double)p.y * q.y;
    x += with_sign(c, __popc(a & tm.yz) & 1u);
  }
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  if (threadIdx.x == 0)
    part[(b * nterms + tm.idx) * gridDim.x + blockIdx.x] = tm.w * ((red[0] + red[1]) + (red[2] + red[3]));
}

namespace {
// 16 bytes of a state: one complex128 amplitude, or two of complex64, those
// at the positions of a flipped within the 16 bytes as well
template <typename T>
constexpr int kQuad = 16 / sizeof(V2<T>);
__device__ __forceinline__ void load_quad(V2<double>* q, const V2<double>* s, uint32_t a) { q[0] = s[a]; }
__device__ __forceinline__ void load_quad(V2<float>* q, const V2<float>* s, uint32_t a) {
  const float4 v = *reinterpret_cast<const float4*>(s + (a & ~1u));
  const bool odd = a & 1u;
  q[0].x = odd ? v.z : v.x;
  q[0].y = odd ? v.w : v.y;
  q[1].x = odd ? v.x : v.z;
  q[1].y = odd ? v.y : v.w;
}
__device__ __forceinline__ void store_quad(V2<double>* s, const double* re, const double* im) {
  *s = double2{re[0], im[0]};
}
__device__ __forceinline__ void store_quad(V2<float>* s, const double* re, const double* im) {
  *reinterpret_cast<float4*>(s) = float4{(float)re[0], (float)im[0], (float)re[1], (float)im[1]};
}
}  // namespace

// out as k_pauli_terms_apply, 16 bytes per thread over all strings
template <typename T>
__global__ void __launch_bounds__(256) k_pauli_terms_apply_each(const DPTermX* __restrict__ terms, int n, int nterms,
                                                                const V2<T>* __restrict__ psi,
                                                                V2<T>* __restrict__ out,
                                                                const double* __restrict__ wts, int64_t total) {
  constexpr int E = kQuad<T>;
  for (int64_t i = (blockIdx.x * 256ll + threadIdx.x) * E; i < total; i += gridDim.x * 256ll * E) {
    const int64_t b = i >> n;
    const uint32_t a = (uint32_t)(i & (((int64_t)1 << n) - 1));
    const V2<T>* s = psi + (b << n);
    const double* wb = wts + b * nterms;
    double hr[E], hi[E];
#pragma unroll
    for (int e = 0; e < E; ++e) hr[e] = hi[e] = 0.0;
    for (int t = 0; t < nterms; ++t) {
      const DPTermX tm = terms[t];
      const double w = tm.w * wb[tm.idx];
      if (w == 0.0) continue;
      V2<T> q[E];
      load_quad(q, s, a ^ tm.flip);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const double c = with_sign(w, __popc((a + e) & tm.yz) & 1u);
        hr[e] += tm.odd ? -c * (double)q[e].y : c * (double)q[e].x;
        hi[e] += tm.odd ? c * (double)q[e].x : c * (double)q[e].y;
      }
    }
    store_quad(out + i, hr, hi);
  }
}

namespace {
// 32 KiB tiles; 8 amplitudes per thread, 1 where that would not fill a wave
template <typename T>
int tile_bits(int n) { return std::min(n, sizeof(T) == 4 ? 12 : 11); }

// Without tiles, from 9 qubits (below, a tile is a wave with one amplitude per
// thread and as fast):
//  - few amplitudes and strings, where tiles are a chain of LDS reads on few CUs
//    (expectations of 60 and of 200 strings on 2^16 amplitudes, complex64: 17 and
//    17 us, 21 and 24 by tiles; of 200 on 2^18, 50 and 32 us; of 16 on 64 x 2^14,
//    22 and 17 us);
//  - one or two strings, which leave little to share (one on 8 x 2^22
//    amplitudes, complex64: 54 us, 83 by tiles; on 64 x 2^20 in complex128 176
//    and 207), four where most flips leave the tile and a state stays in cache
//    (four of four on 8 x 2^20, complex128: 52 and 80 us; two of four on 64 x
//    2^18, 111 and 59 us).
// far: flip masks that leave the tile
template <typename T>
bool each_term(int n, int nterms, int far, int64_t batch) {
  if (n < 9) return false;
  if (nterms <= 2 || (batch << n <= 1 << 18 && (batch << n) * nterms <= 1 << 24)) return true;
  return nterms <= 4 && 2 * far > nterms && (int64_t)sizeof(V2<T>) << n <= 16 << 20;
}
// Applied, for states that can be read 16 bytes at a time:
//  - up to 2^19 amplitudes (60 strings on 2^10, complex64: 18 us, 28 by tiles; on
//    8 x 2^16 28 and 38, on 64 x 2^14 50 and 39 us);
//  - one or two strings, in complex128 up to eight (two on 8 x 2^20, complex64:
//    24 and 39 us, four on 2^24 94 and 73; eight on 8 x 2^22 in complex128 537
//    and 619 us, sixteen on 2^24 542 and 540).
template <typename T>
bool each_term_apply(int n, int nterms, int64_t batch, const void* psi, const void* out) {
  if (n < 9 || (((uintptr_t)psi | (uintptr_t)out) & 15)) return false;
  return nterms <= (sizeof(T) == 4 ? 2 : 8) || batch << n <= 1 << 19;
}
}  // namespace

int pauli_terms_far(uint32_t flip, int n, bool c64) { return flip >> (c64 ? tile_bits<float>(n) : tile_bits<double>(n)) ? 1 : 0; }

int pauli_terms_blocks(int n, bool c64) { return 1 << std::min(n - (c64 ? tile_bits<float>(n) : tile_bits<double>(n)), 10); }

template <typename T>
void launch_pauli_terms(const PauliTermTables& D, int nchunks, int nterms, const int* far, int n, const void* psi,
                        int64_t batch, double* part, double* out, hipStream_t st) {
  const int k = tile_bits<T>(n), nblk = pauli_terms_blocks(n, sizeof(T) == 4);
  auto go = [&](auto kern, int le) {
    const unsigned threads = std::max(64u, 1u << (k - le)), nw = threads / 64;
    const size_t lds = (sizeof(V2<T>) << k) + (size_t)nw * 8 * (kTermsChunk + 4 * kRow) +
                       kTermsChunk * (sizeof(uint32_t) + sizeof(DPGroupX));
    hipLaunchKernelGGL(kern, dim3((unsigned)nblk, (unsigned)nchunks, (unsigned)batch), dim3(threads), lds, st,
                       (const DPChunk*)D.chunks, (const DPGroupX*)D.groups, (const DPTermX*)D.terms, n, k, nterms,
                       (const V2<T>*)psi, part);
  };
  if (each_term<T>(n, nterms, far[sizeof(T) == 8], batch))
    hipLaunchKernelGGL(k_pauli_terms_each<T>, dim3((unsigned)nblk, (unsigned)nterms, (unsigned)batch), dim3(256), 0, st,
                       (const DPTermX*)D.terms, n, nterms, (const V2<T>*)psi, part);
  else if (k >= 9) go(k_pauli_terms<T, 3>, 3);
  else go(k_pauli_terms<T, 0>, 0);
  const int64_t total = batch * nterms;
  hipLaunchKernelGGL(k_pauli_terms_sum, dim3((unsigned)std::min(total, kMaxLaunchThreads / 64)), dim3(64), 0, st,
                     (const double*)part, nblk, total, out);
}

template <typename T>
void launch_pauli_terms_apply(const PauliTermTables& D, int nchunks, int nterms, int n, const void* psi, void* out,
                              const double* weights, int64_t batch, hipStream_t st) {
  const int k = tile_bits<T>(n);
  const size_t lds = (sizeof(V2<T>) << k) + kTermsChunk * (16 + sizeof(DPGroupX));
  auto go = [&](auto kern, int le) {
    const int64_t ntiles = batch << (n - k);
    hipLaunchKernelGGL(kern, dim3((unsigned)std::min<int64_t>(ntiles, 1 << 20)), dim3(std::max(64u, 1u << (k - le))),
                       lds, st, (const DPChunk*)D.chunks, nchunks, (const DPGroupX*)D.groups, (const DPTermX*)D.terms,
                       n, k, nterms, (const V2<T>*)psi, (V2<T>*)out, weights, ntiles);
  };
  const int64_t total = batch << n;
  if (each_term_apply<T>(n, nterms, batch, psi, out)) {
    const int64_t blocks = std::min<int64_t>(std::max<int64_t>(total / (256 * kQuad<T>), 1), 65536);
    hipLaunchKernelGGL(k_pauli_terms_apply_each<T>, dim3((unsigned)blocks), dim3(256), 0, st, (const DPTermX*)D.terms, n,
                       nterms, (const V2<T>*)psi, (V2<T>*)out, weights, total);
  } else if (k >= 9) {
    go(k_pauli_terms_apply<T, 3>, 3);
  } else {
    go(k_pauli_terms_apply<T, 0>, 0);
  }
}

#define TCM_TERMS_INST(T)                                                                                           \
  template void launch_pauli_terms<T>(const PauliTermTables&, int, int, const int*, int, const void*, int64_t,     \
                                      double*, double*, hipStream_t);                                               \
  template void launch_pauli_terms_apply<T>(const PauliTermTables&, int, int, int, const void*, void*,              \
                                            const double*, int64_t, hipStream_t);
TCM_TERMS_INST(float)
TCM_TERMS_INST(double)

}  // namespace tcm

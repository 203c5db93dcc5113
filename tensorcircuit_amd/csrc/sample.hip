// HIP kernels of libtcm for CDNA4 (gfx950): draws from |psi|^2 or a
// probability vector by inverse CDF (backend.probability_sample,
// abstract_backend.py:1124-1157).
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace tcm {

namespace {

// weight of index i: |psi_i|^2 of a state (PROB false) or p_i (PROB true)
template <typename T, bool PROB>
__device__ __forceinline__ double weight_at(const void* src, int64_t i) {
  if constexpr (PROB) {
    return (double)static_cast<const T*>(src)[i];
  } else {
    const V2<T> x = static_cast<const V2<T>*>(src)[i];
    return (double)x.x * x.x + (double)x.y * x.y;
  }
}

// inclusive prefix sum over each group of 16 lanes
__device__ __forceinline__ double scan16(double x, int l16) {
  for (int off = 1; off < 16; off <<= 1) {
    const double v = __shfl_up(x, off, 16);
    if (l16 >= off) x += v;
  }
  return x;
}

}  // namespace

// fp64 sums of the weights over chunks of 2^cl indices (cum[b][c + 1]) and,
// inside a chunk, inclusive prefix sums over its stretches of 2^sl
// (sub[b][c][..]): what a draw needs to read 64 weights instead of 1024.
// Bound by reading the state.  grid (nchunks, batch), 256 threads
template <typename T, bool PROB>
__global__ void __launch_bounds__(256) k_sample_sums(const void* __restrict__ src, int64_t sstride, int cl, int sl,
                                                     int64_t nchunks, double* __restrict__ cum,
                                                     double* __restrict__ sub) {
  __shared__ double tot[16];
  const int64_t c = blockIdx.x, b = blockIdx.y;
  const int64_t off = b * sstride + (c << cl);
  const int len = 1 << cl, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double a[4];
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int i = it * 256 + threadIdx.x;
    a[it] = i < len ? weight_at<T, PROB>(src, off + i) : 0.0;
  }
  // the four wave sums together: halves of the wave keep two values each,
  // then quarters one (7 exchanges instead of 24)
  const bool hi = lane & 32, odd = lane & 16;
  double k0 = hi ? a[2] : a[0], k1 = hi ? a[3] : a[1];
  k0 += __shfl_xor(hi ? a[0] : a[2], 32, 64);
  k1 += __shfl_xor(hi ? a[1] : a[3], 32, 64);
  double x = odd ? k1 : k0;
  x += __shfl_xor(odd ? k0 : k1, 16, 64);
  for (int o = 8; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  if ((lane & 15) == 0) tot[((lane >> 5) * 2 + ((lane >> 4) & 1)) * 4 + w] = x;
  __syncthreads();
  if (threadIdx.x < 16) {
    const int nsub = 1 << (cl - sl);
    const double s = scan16(tot[threadIdx.x], threadIdx.x);
    if ((int)threadIdx.x < nsub) sub[(b * nchunks + c) * nsub + threadIdx.x] = s;
    if ((int)threadIdx.x == nsub - 1) cum[b * (nchunks + 1) + c + 1] = s;
    if (c == 0 && threadIdx.x == 0) cum[b * (nchunks + 1)] = 0.0;
  }
}

// In-place inclusive prefix sums of cum[b][1 .. nchunks]; one block per batch
// item, 4 NT sums at a time through LDS so that memory is read and written in
// order (a contiguous range per thread: 32 us for 16384 sums; this: 11 us).
// A wave where a batch item has up to 256 sums (one draw from each of 4096
// vectors of 14 qubits: 123 us with 1024 threads, 100 us), none where it has one
// (of 6 qubits: 41 us with the scan, 17.5 us).
template <int NT>
__global__ void __launch_bounds__(NT) k_sample_scan(double* __restrict__ cum, int64_t nchunks) {
  __shared__ double buf[4 * NT + NT];
  __shared__ double wt[NT / 64];
  __shared__ double last;
  double* c = cum + blockIdx.x * (nchunks + 1) + 1;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  auto at = [](int i) { return i + (i >> 2); };
  double carry = 0.0, nx[4];
  auto fetch = [&](int64_t base) {  // the next ones, while these are summed
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t i = base + q * NT + t;
      nx[q] = i < nchunks ? c[i] : 0.0;
    }
  };
  fetch(0);
  for (int64_t base = 0; base < nchunks; base += 4 * NT) {
#pragma unroll
    for (int q = 0; q < 4; ++q) buf[at(q * NT + t)] = nx[q];
    fetch(base + 4 * NT);
    __syncthreads();
    double v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = buf[at(4 * t + q)];
    const double s = (v[0] + v[1]) + (v[2] + v[3]);
    double incl = s;
    for (int off = 1; off < 64; off <<= 1) {
      const double u = __shfl_up(incl, off, 64);
      if (lane >= off) incl += u;
    }
    if (lane == 63) wt[w] = incl;
    __syncthreads();
    double run = carry;
    for (int i = 0; i < w; ++i) run += wt[i];
    run += incl - s;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      run += v[q];
      buf[at(4 * t + q)] = run;
    }
    if (t == NT - 1) last = run;
    __syncthreads();
    carry = last;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = q * NT + t;
      if (base + i < nchunks) c[base + i] = buf[at(i)];
    }
    __syncthreads();
  }
}

// 16 lanes per draw: r = total (1 - u); the drawn index is the smallest i
// whose inclusive prefix sum reaches r (searchsorted, side left): 16-ary
// search over the chunk sums, then the chunk's 16 stretch sums, then the 64
// weights of a stretch, 4 per lane -- about 4 + 1 + 1 dependent reads and 0.7
// KiB a draw.  (A wave per draw, a binary search and a running scan of the
// chunk: 14 + 16 dependent reads and up to 8 KiB; 187 us for 100000 draws
// from 24 qubits, this 20 us.)
// Tree scans round in another order at every lane, so that a running sum can
// grow by a unit over entries of zero weight, and r fall in between (the
// total, for u = 0, did in one of five distributions that end in zeros).  An
// index of probability zero is not drawn then: an empty chunk or stretch is
// left for the last one of nonzero weight before it, and only indices of
// nonzero weight are taken (r = 0 takes index 0).  grid (ceil(shots / 16), batch)
template <typename T, bool PROB>
__global__ void __launch_bounds__(256) k_sample_draw(const void* __restrict__ src, int64_t sstride, int cl, int sl,
                                                     int64_t nchunks, const double* __restrict__ cum,
                                                     const double* __restrict__ sub, const double* __restrict__ u,
                                                     int64_t shots, int64_t* __restrict__ out) {
  const int l = threadIdx.x & 15, shift = (threadIdx.x & 48);
  const int64_t s = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
  const int64_t b = blockIdx.y;
  const bool live = s < shots;
  auto mask16 = [&](bool x) { return (uint32_t)(__ballot(x) >> shift) & 0xffffu; };
  const double* c = cum + b * (nchunks + 1);
  const double r = c[nchunks] * (1.0 - u[b * shots + (live ? s : shots - 1)]);
  int64_t lo = 0;
  for (int64_t rem = nchunks; rem > 1;) {
    const int64_t step = rem >= 16 ? rem >> 4 : 1;
    const int segs = rem >= 16 ? 16 : (int)rem;
    const uint32_t m = mask16(l < segs && c[lo + (l < segs ? l + 1 : 1) * step] >= r);
    lo += (m ? __ffs(m) - 1 : segs - 1) * step;
    rem = step;
  }
  const int nsub = 1 << (cl - sl);
  double c0, sp;
  uint32_t m, grows;
  auto read_sums = [&] {
    c0 = c[lo];
    sp = l < nsub ? sub[(b * nchunks + lo) * nsub + l] : 0.0;
    const double before = __shfl_up(sp, 1, 16);
    m = mask16(l < nsub && c0 + sp >= r);
    // rounding left r just above the chunk's last sum: its last stretch of
    // nonzero weight (and, below, the last index of it)
    grows = mask16(l < nsub && sp > (l ? before : 0.0));
  };
  read_sums();
  // the rare steps back are left to branches of the whole wave
  if (__any(!m && !grows)) {  // an empty chunk: the last one of nonzero weight before
    uint32_t some = m | grows;
    for (int64_t e = lo; e > 0 && !some; e -= 16) {
      some = mask16(e > l && sub[(b * nchunks + (e > l ? e - 1 - l : 0)) * nsub + nsub - 1] > 0.0);
      if (some) lo = e - __ffs(some);
    }
    read_sums();
  }
  int k = m ? __ffs(m) - 1 : grows ? 31 - __clz(grows) : 0;
  // 2^sl weights, `per` consecutive ones per lane
  const int len = 1 << sl, per = len >= 16 ? len >> 4 : 1;
  double p[4], acc, run;
  bool some[4];  // which of them are not zero
  uint32_t nz;   // in which lanes
  auto read_weights = [&] {
    const double prefix = __shfl(sp, k > 0 ? k - 1 : 0, 16);
    run = c0 + (k > 0 ? prefix : 0.0);
    const int64_t first = b * sstride + (lo << cl) + ((int64_t)k << sl);
    double x[4];  // all four loads in flight
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = weight_at<T, PROB>(src, first + (j < per && l * per + j < len ? l * per + j : 0));
    acc = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j >= per || l * per + j >= len) x[j] = 0.0;
      acc += x[j];
      p[j] = acc;
      some[j] = x[j] > 0.0;
    }
    nz = mask16(some[0] || some[1] || some[2] || some[3]);
  };
  read_weights();
  while (__any(!nz && k > 0 && r > 0.0)) {  // an empty stretch: the one before
    if (!nz && k > 0 && r > 0.0) --k;
    read_weights();
  }
  const bool all = !(r > 0.0);
  const double excl = scan16(acc, l) - acc;
  int hit = -1;
#pragma unroll
  for (int j = 3; j >= 0; --j) {
    const int i = l * per + j;
    if (j < per && i < len && (some[j] || all) && run + (excl + p[j]) >= r) hit = i;
  }
  m = mask16(hit >= 0);
  const int lastnz = l * per + (some[3] ? 3 : some[2] ? 2 : some[1] ? 1 : 0);
  const int from = m ? __ffs(m) - 1 : nz ? 31 - __clz(nz) : 0;
  const int found = __shfl(m ? hit : nz ? lastnz : 0, from, 16);
  if (live && l == 0) out[b * shots + s] = (lo << cl) + ((int64_t)k << sl) + found;
}

// chunks of up to 2^10 indices, stretches of up to 2^6; cum: batch x
// (nchunks + 1) sums, then batch x nchunks x 16 stretch sums
template <typename T>
void launch_sample(const void* src, bool prob, int n, int64_t batch, const double* u, int64_t shots, int64_t* out,
                   double* cum, hipStream_t st) {
  const int cl = n < kSampleChunkLog ? n : kSampleChunkLog, sl = n < kSampleSubLog ? n : kSampleSubLog;
  const int64_t nchunks = 1ll << (n - cl);
  const int64_t sstride = 1ll << n;
  double* sub = cum + batch * (nchunks + 1);
  const dim3 gc((unsigned)nchunks, (unsigned)batch), gd((unsigned)((shots + 15) / 16), (unsigned)batch);
  if (prob) hipLaunchKernelGGL((k_sample_sums<T, true>), gc, dim3(256), 0, st, src, sstride, cl, sl, nchunks, cum, sub);
  else hipLaunchKernelGGL((k_sample_sums<T, false>), gc, dim3(256), 0, st, src, sstride, cl, sl, nchunks, cum, sub);
  if (nchunks > 256) hipLaunchKernelGGL(k_sample_scan<1024>, dim3((unsigned)batch), dim3(1024), 0, st, cum, nchunks);
  else if (nchunks > 1) hipLaunchKernelGGL(k_sample_scan<64>, dim3((unsigned)batch), dim3(64), 0, st, cum, nchunks);
  if (prob)
    hipLaunchKernelGGL((k_sample_draw<T, true>), gd, dim3(256), 0, st, src, sstride, cl, sl, nchunks,
                       (const double*)cum, (const double*)sub, u, shots, out);
  else
    hipLaunchKernelGGL((k_sample_draw<T, false>), gd, dim3(256), 0, st, src, sstride, cl, sl, nchunks,
                       (const double*)cum, (const double*)sub, u, shots, out);
}

#define TCM_SAMPLE_INST(T)                                                                                          \
  template void launch_sample<T>(const void*, bool, int, int64_t, const double*, int64_t, int64_t*, double*,        \
                                 hipStream_t);
TCM_SAMPLE_INST(float)
TCM_SAMPLE_INST(double)

}  // namespace tcm

// HIP kernels of libtcm for CDNA4 (gfx950): sparse matrices in CSR form --
// <psi|A|psi> (sparse_expectation, templates/measurements.py:177-191), A x,
// and conj(g) A x + g A^dagger x, the vector-Jacobian product of the
// expectation.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"

namespace tcm {

namespace {

enum CsrMode { CSR_MATVEC, CSR_EXPECT, CSR_VJP };

// lanes per row: a power of two near a quarter of the mean row length, so
// that a row of the mean length is one step of four entries per lane
__device__ __forceinline__ int lanes_per_row(const int64_t* rowptr, int n) {
  const int64_t mean = rowptr[(int64_t)1 << n] >> n;
  int g = 1;
  while (g < 64 && 4 * g < mean) g <<= 1;
  return __builtin_amdgcn_readfirstlane(g);
}

// sum over the row's entries of vals_k x_{cols_k} in fp64, in every lane of
// its group of g lanes (q = lane within the group); all lanes of the wave
// call it, with an empty range where there is no row
template <typename T>
__device__ __forceinline__ void row_dot(int64_t k0, int64_t k1, const int64_t* __restrict__ cols,
                                        const V2<T>* __restrict__ vals, const V2<T>* __restrict__ x, int g, int q,
                                        double& hr, double& hi) {
  hr = hi = 0.0;
  for (int64_t k = k0 + q; k < k1; k += 4 * g) {
    int64_t c[4];
    V2<T> v[4], p[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t e = k + (int64_t)u * g;
      if (e < k1) {
        c[u] = cols[e];
        v[u] = vals[e];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k + (int64_t)u * g < k1) p[u] = x[c[u]];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (k + (int64_t)u * g >= k1) break;
      hr += (double)v[u].x * p[u].x - (double)v[u].y * p[u].y;
      hi += (double)v[u].x * p[u].y + (double)v[u].y * p[u].x;
    }
  }
  for (int off = g >> 1; off > 0; off >>= 1) {
    hr += __shfl_xor(hr, off, 64);
    hi += __shfl_xor(hi, off, 64);
  }
}

}  // namespace

// One group of 1 to 64 lanes per row (lanes_per_row), rows of a wave next to
// each other, so that the wave's loads of columns and values are one
// contiguous stretch; bound by reading the matrix (16 or 24 bytes an entry).
// One thread per row read its own stretch 8 bytes at a time, a cache line per
// lane: 187 us for the 5 million entries of an 18-qubit Ising matrix in
// complex64; this: 24 us (3.6 TB/s).  Entries past a lane's last are not loaded:
// read again, they cost rows of three entries a third more.
// MATVEC: y_b = A x_b.  EXPECT: partial sums of conj(x) A x.  VJP: y_b =
// conj(g_b) A x_b + g_b A^dagger x_b, the second product from the CSR form of
// A^dagger (drowptr, ...), or 2 Re(g_b) A x_b where that is null (A = A^dagger).
template <typename T, int MODE>
__global__ void __launch_bounds__(256) k_csr(const int64_t* __restrict__ rowptr, const int64_t* __restrict__ cols,
                                             const V2<T>* __restrict__ vals, const int64_t* __restrict__ drowptr,
                                             const int64_t* __restrict__ dcols, const V2<T>* __restrict__ dvals,
                                             const V2<T>* __restrict__ x, const V2<T>* __restrict__ gs,
                                             V2<T>* __restrict__ y, int n, int64_t total,
                                             double* __restrict__ part) {
  const int g = lanes_per_row(rowptr, n);
  const int lane = threadIdx.x & 63, q = lane & (g - 1), per = 64 / g;
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
  double er = 0.0, ei = 0.0;
  for (int64_t i0 = wave * per; i0 < total; i0 += nwaves * per) {
    const int64_t i = i0 + lane / g;
    const bool have = i < total;
    const int64_t b = have ? i >> n : 0, r = have ? i - (b << n) : 0;
    const V2<T>* xb = x + (b << n);
    double hr, hi;
    row_dot<T>(have ? rowptr[r] : 0, have ? rowptr[r + 1] : 0, cols, vals, xb, g, q, hr, hi);
    if constexpr (MODE == CSR_EXPECT) {
      if (have && q == 0) {
        const V2<T> p = xb[r];
        er += (double)p.x * hr + (double)p.y * hi;
        ei += (double)p.x * hi - (double)p.y * hr;
      }
    }
    if constexpr (MODE == CSR_VJP) {
      const V2<T> gb = gs[b];
      if (drowptr) {
        double dr, di;
        row_dot<T>(have ? drowptr[r] : 0, have ? drowptr[r + 1] : 0, dcols, dvals, xb, g, q, dr, di);
        const double a = (double)gb.x * hr + (double)gb.y * hi, c = (double)gb.x * hi - (double)gb.y * hr;
        hr = a + ((double)gb.x * dr - (double)gb.y * di);
        hi = c + ((double)gb.x * di + (double)gb.y * dr);
      } else {
        // the imaginary parts cancel; one that is not finite leaves NaN
        const double a = 2.0 * (double)gb.x + ((double)gb.y - (double)gb.y);
        hr *= a;
        hi *= a;
      }
    }
    if constexpr (MODE != CSR_EXPECT) {
      if (have && q == 0) {
        V2<T> o;
        o.x = (T)hr;
        o.y = (T)hi;
        y[i] = o;
      }
    }
  }
  if constexpr (MODE == CSR_EXPECT) {
    __shared__ double red[2][4];
    for (int off = 32; off > 0; off >>= 1) {
      er += __shfl_xor(er, off, 64);
      ei += __shfl_xor(ei, off, 64);
    }
    if (lane == 0) {
      red[0][threadIdx.x >> 6] = er;
      red[1][threadIdx.x >> 6] = ei;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      part[2 * blockIdx.x] = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
      part[2 * blockIdx.x + 1] = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    }
  }
}

namespace {
// an expectation: up to 8 blocks per CU, at least 16 lanes per row
int csr_blocks(int64_t total) { return (int)std::max<int64_t>(1, std::min<int64_t>(kCsrBlocks, total / 16)); }
// a product: a lane per row in blocks that come and go (33 products with 2^18
// rows of three entries, complex64: 84 us with 2048 blocks that loop, 53 us)
int product_blocks(int64_t total) {
  return (int)std::max<int64_t>(csr_blocks(total), std::min<int64_t>(65536, total / 256));
}
}  // namespace

template <typename T>
void launch_csr_matvec(const int64_t* rowptr, const int64_t* cols, const void* vals, const void* x, void* y,
                       int n, int64_t batch, hipStream_t st) {
  hipLaunchKernelGGL((k_csr<T, CSR_MATVEC>), dim3(product_blocks(batch << n)), dim3(256), 0, st, rowptr, cols,
                     (const V2<T>*)vals, nullptr, nullptr, nullptr, (const V2<T>*)x, nullptr, (V2<T>*)y, n,
                     batch << n, nullptr);
}

template <typename T>
void launch_csr_vjp(const int64_t* rowptr, const int64_t* cols, const void* vals, const int64_t* drowptr,
                    const int64_t* dcols, const void* dvals, const void* x, const void* g, void* y, int n,
                    int64_t batch, hipStream_t st) {
  hipLaunchKernelGGL((k_csr<T, CSR_VJP>), dim3(product_blocks(batch << n)), dim3(256), 0, st, rowptr, cols,
                     (const V2<T>*)vals, drowptr, dcols, (const V2<T>*)dvals, (const V2<T>*)x, (const V2<T>*)g,
                     (V2<T>*)y, n, batch << n, nullptr);
}

template <typename T>
void launch_csr_expect(const int64_t* rowptr, const int64_t* cols, const void* vals, const void* psi, int n,
                       double* part, double* out, hipStream_t st) {
  const int nblk = csr_blocks((int64_t)1 << n);
  hipLaunchKernelGGL((k_csr<T, CSR_EXPECT>), dim3(nblk), dim3(256), 0, st, rowptr, cols, (const V2<T>*)vals, nullptr,
                     nullptr, nullptr, (const V2<T>*)psi, nullptr, nullptr, n, (int64_t)1 << n, part);
  launch_sum_slots(part, (int64_t)2 * nblk, nblk, 2, out, 1, st);
}

#define TCM_CSR_INST(T)                                                                                              \
  template void launch_csr_matvec<T>(const int64_t*, const int64_t*, const void*, const void*, void*, int, int64_t,  \
                                     hipStream_t);                                                          \
  template void launch_csr_vjp<T>(const int64_t*, const int64_t*, const void*, const int64_t*, const int64_t*,       \
                                  const void*, const void*, const void*, void*, int, int64_t, hipStream_t);          \
  template void launch_csr_expect<T>(const int64_t*, const int64_t*, const void*, const void*, int, double*,         \
                                     double*, hipStream_t);
TCM_CSR_INST(float)
TCM_CSR_INST(double)

}  // namespace tcm

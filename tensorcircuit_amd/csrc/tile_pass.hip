// HIP kernels of libtcm for CDNA4 (gfx950): table-driven tile passes, forward,
// adjoint and several programs in one launch -- every pass that is not
// compiled (programs built without opts.jit, tiles of less than a wave).
//
// A tile of 2^k amplitudes (k tile bits) is staged in LDS; segments (register
// groups) of 2^4 amplitudes per thread apply runs of gates, exchanged through
// the tile between segments, and the tile is written back: one read and one
// write of the state for all gates of the pass.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "regops.h"

namespace tcm {

namespace {

constexpr int kR = kTileSlots, kE = 1 << kR;
// a lane row of the gradient buffer: 64 partials, padded off its banks
template <typename T>
constexpr int kGRow = sizeof(T) == 4 ? 68 : 66;

// LDS swizzle: the low 5 element bits XOR the higher 5-bit fields (linear
// over XOR), so that the lanes of a group exchange meet few bank conflicts
__device__ __forceinline__ uint32_t swz5(uint32_t t) { return t ^ (((t >> 5) ^ (t >> 10)) & 0x1Fu); }

// no permutation at the end of a segment (the second word's bits 8 ..)
constexpr uint32_t kPermNone = 0x08421u;

__device__ __forceinline__ uint32_t uni(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }

// block index -> the index bits outside the tile
__device__ __forceinline__ uint64_t deposit(uint64_t blk, uint64_t m, int nbl) {
  uint64_t base = 0;
  for (int i = 0; i < nbl; ++i) {
    const uint64_t low = m & (~m + 1);
    if ((blk >> i) & 1) base |= low;
    m ^= low;
  }
  return base;
}

// LDS of one block, carved from the dynamic allocation
template <typename T>
struct Lds {
  A2<T>* tile;     // 2^k
  T* mat;          // kStageMat
  uint32_t* blob;  // kStageBlob words: segments, ops, members, gradient list, counts
  double* red;     // adjoint: [kStageGrad][waves]
  T* grad;         // adjoint: [waves][4][kGRow]
  __device__ __forceinline__ Lds(unsigned char* p, int k, int nw) {
    tile = reinterpret_cast<A2<T>*>(p);
    mat = reinterpret_cast<T*>(tile + (1 << k));
    blob = reinterpret_cast<uint32_t*>(mat + kStageMat);
    red = reinterpret_cast<double*>(blob + kStageBlob);
    grad = reinterpret_cast<T*>(red + kStageGrad * nw);
  }
};

// Stage one chunk's tables: its words, and the matrix entries it reads,
// gathered from the item's table or the constants.  Four loads in flight per
// thread; `between` issues other loads before the first wait.
template <typename T, typename F>
__device__ __forceinline__ void stage(const Lds<T>& S, const uint32_t* __restrict__ blob,
                                      const int32_t* __restrict__ msrc, const T* mt, const T* __restrict__ ct,
                                      F between) {
  const int nt = blockDim.x, t0 = threadIdx.x;
  auto entry = [&](int32_t s) { return s >= 0 ? mt[s] : s == kStageZero ? T(0) : ct[-s - 1]; };
  int32_t ms[4];
  uint32_t bw[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = u * nt + t0;
    ms[u] = i < kStageMat ? msrc[i] : kStageNone;
    bw[u] = i < kStageBlob ? blob[i] : 0u;
  }
  between();
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int i = u * nt + t0;
    if (ms[u] != kStageNone) S.mat[i] = entry(ms[u]);
    if (i < kStageBlob) S.blob[i] = bw[u];
  }
  for (int i = 4 * nt + t0; i < kStageMat; i += nt) {  // blocks of one wave
    const int32_t s = msrc[i];
    if (s != kStageNone) S.mat[i] = entry(s);
  }
}
static_assert(kStageBlob <= 4 * 64, "a block of one wave stages the words in four loads");

// N matrix entries from LDS (N a multiple of 4, 16-byte aligned)
template <typename T, int N>
__device__ __forceinline__ void load_mat(T* m, const T* s) {
  typedef T v4 __attribute__((ext_vector_type(4)));
  const v4* p = reinterpret_cast<const v4*>(s);
#pragma unroll
  for (int i = 0; i < N / 4; ++i) {
    const v4 x = p[i];
    m[4 * i] = x.x;
    m[4 * i + 1] = x.y;
    m[4 * i + 2] = x.z;
    m[4 * i + 3] = x.w;
  }
}

// f(0), ..., f(N - 1) with compile-time indices
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (N > 0) {
    each<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// Exchange two amplitudes in place.  Written as plain assignments the swaps
// become moves of every amplitude at the end of the branch.  TAG tells the
// statements of different branches apart: alike, they are merged into one
// that works on indexed memory.
template <int TAG>
__device__ __forceinline__ void swap_reg(int& a, int& b) {
  asm("v_swap_b32 %0, %1 ; %2" : "+v"(a), "+v"(b) : "n"(TAG));
}
template <int TAG>
__device__ __forceinline__ void swap_reg(float& a, float& b) {
  asm("v_swap_b32 %0, %1 ; %2" : "+v"(a), "+v"(b) : "n"(TAG));
}
template <int TAG>
__device__ __forceinline__ void swap_reg(double& a, double& b) {
  int al = __double2loint(a), ah = __double2hiint(a), bl = __double2loint(b), bh = __double2hiint(b);
  swap_reg<TAG>(al, bl);
  swap_reg<TAG>(ah, bh);
  a = __hiloint2double(ah, al);
  b = __hiloint2double(bh, bl);
}
template <int TAG, typename T>
__device__ __forceinline__ void swap2(A2<T>& a, A2<T>& b) {
  swap_reg<TAG>(a.x, b.x);
  swap_reg<TAG>(a.y, b.y);
}
template <typename T, int S>
__device__ __forceinline__ void perm_x1(A2<T>* v) {
  each<kE>([&](auto j) {
    if constexpr (!(j & (1 << S))) swap2<j + 64 * S, T>(v[j], v[j | (1 << S)]);
  });
}
template <typename T, int S0, int S1>
__device__ __forceinline__ void perm_cx(A2<T>* v) {
  each<kE>([&](auto j) {
    if constexpr ((j & (1 << S0)) && !(j & (1 << S1))) swap2<j + 64 * S0 + 256 * S1, T>(v[j], v[j | (1 << S1)]);
  });
}
template <typename T, int S0, int S1>
__device__ __forceinline__ void perm_swap(A2<T>* v) {
  each<kE>([&](auto j) {
    if constexpr ((j & (1 << S0)) && !(j & (1 << S1)))
      swap2<j + 64 * S0 + 256 * S1, T>(v[j], v[(j ^ (1 << S0)) | (1 << S1)]);
  });
}

// x = c x + a, in x's own register (left to itself the compiler accumulates
// into a's, and moves the result at the end of the branch)
__device__ __forceinline__ void fused(float& x, float c, float a) {
  asm("v_fma_f32 %0, %1, %0, %2" : "+v"(x) : "v"(c), "v"(a));
}
__device__ __forceinline__ void fused(double& x, double c, double a) {
  asm("v_fma_f64 %0, %1, %0, %2" : "+v"(x) : "v"(c), "v"(a));
}

// sum over the wave, in every lane
__device__ __forceinline__ double wave_all(double x) {
  for (int off = 1; off < 64; off <<= 1) x += __shfl_xor(x, off, 64);
  return x;
}

// (x, y) -> (c x - s y, s x + c y), the products with c fused: near the
// identity, where variational angles are, each result is rounded once at
// full size.  (Three shears cost three quarters of this, but round three
// times a pair: gradients of a 17-qubit, 8-layer circuit were off by 2.4e-6
// instead of 2.0e-6.)
template <typename T>
__device__ __forceinline__ void turn(T& x, T& y, T c, T s) {
  const T a = -s * y, b = s * x;
  fused(x, c, a);
  fused(y, c, b);
}
// ry turns the real and the imaginary parts of a pair alike, rx the pairs
// (x.re, y.im) by -angle and (x.im, y.re) by +angle
template <typename T, int S>
__device__ __forceinline__ void ap_ry(A2<T>* v, T c, T s) {
#pragma unroll
  for (int j = 0; j < kE; ++j) {
    if (j & (1 << S)) continue;
    turn(v[j].x, v[j | (1 << S)].x, c, s);
    turn(v[j].y, v[j | (1 << S)].y, c, s);
  }
}
template <typename T, int S>
__device__ __forceinline__ void ap_rx(A2<T>* v, T c, T s) {
#pragma unroll
  for (int j = 0; j < kE; ++j) {
    if (j & (1 << S)) continue;
    turn(v[j].x, v[j | (1 << S)].y, c, -s);
    turn(v[j].y, v[j | (1 << S)].x, c, s);
  }
}

// fields of a macro op (layout: tcm_internal.h)
struct Macro {
  uint32_t ry, rx, cx, rare, s0, s1, dg, gry, grx, gen, nmem, mem0, gm;
  const uint32_t m0;
  __device__ __forceinline__ explicit Macro(uint4 w) : m0(uni(w.z) & 0xffffu) {
    const uint32_t a = uni(w.x), b = uni(w.y), c = uni(w.z);
    ry = a & 15u;
    rx = (a >> 4) & 15u;
    cx = (a >> 8) & 0xfffu;
    rare = (a >> 20) & 15u;
    s0 = (a >> 24) & 3u;
    s1 = (a >> 26) & 3u;
    dg = (a >> 28) & 1u;
    gry = b & 15u;
    grx = (b >> 4) & 15u;
    gen = (b >> 8) & 15u;
    nmem = (b >> 12) & 0xffu;
    mem0 = (b >> 20) & 0xffu;
    gm = c >> 16;
  }
};

// Every op of a macro op is a branch around straight-line code that changes
// the amplitudes in place.  As the cases of a switch, whose many edges meet in
// one block, the same code cost 16 to 48 register moves per op and spilled.
// `grad(s)` runs before the inverse of slot s's rotation.
template <typename T, bool DAG, typename G>
__device__ __forceinline__ void rys(uint32_t mask, const T*& m, A2<T>* v, A2<T>* w, G grad) {
  each<kR>([&](auto s) {
    if (mask & (1u << s)) {
      T q[4];  // c, -s, s, c
      load_mat<T, 4>(q, m);
      m += 4;
      grad(s);
      const T sn = DAG ? -q[2] : q[2];
      ap_ry<T, s>(v, q[0], sn);
      if constexpr (DAG) ap_ry<T, s>(w, q[0], sn);
    }
  });
}
template <typename T, bool DAG, typename G>
__device__ __forceinline__ void rxs(uint32_t mask, const T*& m, A2<T>* v, A2<T>* w, G grad) {
  each<kR>([&](auto s) {
    if (mask & (1u << s)) {
      T q[4];  // c, 0, 0, -s (the matrix's first row)
      load_mat<T, 4>(q, m);
      m += 4;
      grad(s);
      const T sn = DAG ? q[3] : -q[3];
      ap_rx<T, s>(v, q[0], sn);
      if constexpr (DAG) ap_rx<T, s>(w, q[0], sn);
    }
  });
}
// CX i of the fixed order: controls 3..0, for each the other slots 3..0 (the
// adjoint runs the order backwards)
template <typename T, bool DAG>
__device__ __forceinline__ void cnots(uint32_t mask, A2<T>* v, A2<T>* w) {
  each<12>([&](auto i) {
    if (mask & (1u << i)) {
      constexpr int q = DAG ? 11 - i : i, c = 3 - q / 3, k = 3 - q % 3, t = k > c ? k : k - 1;
      perm_cx<T, c, t>(v);
      if constexpr (DAG) perm_cx<T, c, t>(w);
    }
  });
}
template <typename T, bool DAG>
__device__ __forceinline__ void diagonal(const T*& m, A2<T>* v, A2<T>* w) {
  // two entries at a time: 32 held at once would spill
#pragma unroll
  for (int j = 0; j < kE; j += 2) {
    T d[4];
    load_mat<T, 4>(d, m + 2 * j);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const T dr = d[2 * q], di = DAG ? -d[2 * q + 1] : d[2 * q + 1];
      A2<T> x = v[j + q];
      v[j + q] = ma<T>(dr * x.x - di * x.y, dr * x.y + di * x.x);
      if constexpr (DAG) {
        x = w[j + q];
        w[j + q] = ma<T>(dr * x.x - di * x.y, dr * x.y + di * x.x);
      }
    }
  }
  m += 2 * kE;
}
// The ops that come alone (U2 only in FULL kernels); two-slot ones have s0 >
// s1.  The slots are tested as bits of an opaque mask: tests of one value
// would be made a switch, and its cases merged as above.
template <typename T, bool DAG, bool FULL>
__device__ __forceinline__ void rare_op(const Macro& M, const T* m, A2<T>* v, A2<T>* w) {
  uint32_t one = 1u << M.s0, two = 1u << (M.s0 * (M.s0 - 1) / 2 + M.s1), kind = 1u << (M.rare - 1);
  asm volatile("" : "+s"(one), "+s"(two), "+s"(kind));
  if (kind & (1u << OK_R1)) {
    T q[4];
    load_mat<T, 4>(q, m);
    each<kR>([&](auto s) {
      if (one & (1u << s)) {
        ap_r1<T, kR, s, DAG>(v, q);
        if constexpr (DAG) ap_r1<T, kR, s, DAG>(w, q);
      }
    });
  }
  if (kind & (1u << OK_U1)) {
    T q[8];
    load_mat<T, 8>(q, m);
    each<kR>([&](auto s) {
      if (one & (1u << s)) {
        ap_u1<T, kR, s, DAG>(v, q);
        if constexpr (DAG) ap_u1<T, kR, s, DAG>(w, q);
      }
    });
  }
  if (kind & (1u << OK_X1)) {
    each<kR>([&](auto s) {
      if (one & (1u << s)) {
        perm_x1<T, s>(v);
        if constexpr (DAG) perm_x1<T, s>(w);
      }
    });
  }
  if (kind & (1u << OK_SWAP)) {
    each<kR>([&](auto a) {
      each<a>([&](auto b) {
        if (two & (1u << (a * (a - 1) / 2 + b))) {
          perm_swap<T, a, b>(v);
          if constexpr (DAG) perm_swap<T, a, b>(w);
        }
      });
    });
  }
  if (kind & (1u << OK_CZ)) {
    each<kR>([&](auto a) {
      each<a>([&](auto b) {
        if (two & (1u << (a * (a - 1) / 2 + b))) {
          ap_cz<T, kR, a, b>(v);
          if constexpr (DAG) ap_cz<T, kR, a, b>(w);
        }
      });
    });
  }
  if constexpr (FULL) {
    if (kind & (1u << OK_U2)) {
      T q[32];
      load_mat<T, 32>(q, m);
      each<kR>([&](auto a) {
        each<a>([&](auto b) {
          if (two & (1u << (a * (a - 1) / 2 + b))) {
            ap_u2<T, kR, a, b, DAG>(v, q);
            if constexpr (DAG) ap_u2<T, kR, a, b, DAG>(w, q);
          }
        });
      });
    }
  }
}

// Addresses of a segment: the thread's tile position has zeros at the four
// slot positions; register j adds the masks of its set bits.  `perm` (second
// segment word) folds the segment's last permutation gates (X, CX, SWAP) into
// the addresses it is written to: register bit s goes to the slots of a
// 4-bit mask, all of them shifted by a constant.
struct SegAddr {
  uint32_t a0;
  uint32_t e[kR];
  __device__ __forceinline__ SegAddr(uint32_t word, uint32_t tid) {
    uint32_t x = tid;
#pragma unroll
    for (int i = 0; i < kR; ++i) {  // sorted slot positions, ascending
      const uint32_t p = (word >> (16 + 4 * i)) & 15u;
      x = ((x >> p) << (p + 1)) | (x & ((1u << p) - 1u));
    }
    a0 = swz5(x);
#pragma unroll
    for (int s = 0; s < kR; ++s) e[s] = swz5(1u << ((word >> (4 * s)) & 15u));
  }
  __device__ __forceinline__ uint32_t slots(uint32_t m) const {
    return ((m & 1u) ? e[0] : 0u) ^ ((m & 2u) ? e[1] : 0u) ^ ((m & 4u) ? e[2] : 0u) ^ ((m & 8u) ? e[3] : 0u);
  }
  __device__ __forceinline__ SegAddr permuted(uint32_t perm) const {
    SegAddr w = *this;
    w.a0 = a0 ^ slots((perm >> 24) & 15u);
    asm volatile("" : "+v"(w.a0));  // formed here, not held through the ops
#pragma unroll
    for (int s = 0; s < kR; ++s) w.e[s] = slots((perm >> (8 + 4 * s)) & 15u);
    return w;
  }
  __device__ __forceinline__ uint32_t at(int j) const { return a0 ^ slots((uint32_t)j); }
};

// Body of one forward pass over tile `blk`: s_in -> s_out (the same state,
// or the input of a run's first pass), |0..0> instead of s_in when zinit.
// Waves past the tile's threads (a smaller tile than the block) only stage
// and meet the barriers; lanes past them in the last wave repeat the tile's
// lanes and store nothing.
template <typename T, bool FULL>
__device__ __forceinline__ void fwd_tile(const TilePassArg& A, const uint32_t* __restrict__ blob,
                                         const int32_t* __restrict__ msrc, const uint32_t* __restrict__ runoff,
                                         const T* mt, const T* __restrict__ ct, const A2<T>* s_in, A2<T>* s_out,
                                         A2<T>* __restrict__ ck, uint64_t base, bool zinit, unsigned char* smem) {
  const int tl = A.k - kR, L = A.L;
  const uint32_t nthr = 1u << tl;
  const uint32_t tid = threadIdx.x & (nthr - 1);
  const bool act = threadIdx.x < nthr;
  const bool live = uni(threadIdx.x) < std::max(64u, nthr);  // per wave
  const Lds<T> S(smem, A.k, 0);
  const uint32_t* ro = runoff + A.runoff0;
  uint32_t dlo = run_dep(ro, L, tid);
  {
    A2<T> r[kE];
    stage<T>(S, blob + (int64_t)A.chunk0 * kStageBlob, msrc + (int64_t)A.chunk0 * kStageMat, mt, ct, [&] {
      if (zinit) {
#pragma unroll
        for (int it = 0; it < kE; ++it) r[it] = ma<T>(T(0), T(0));
        if ((base | dlo) == 0) r[0].x = T(1);
      } else if (live) {
#pragma unroll
        for (int it = 0; it < kE; ++it) r[it] = s_in[base + run_dep(ro, L, (uint32_t)it << tl) + dlo];
      }
    });
    if (live) {
#pragma unroll
      for (int it = 0; it < kE; ++it) S.tile[swz5(((uint32_t)it << tl) | tid)] = r[it];
    }
  }
  __syncthreads();
  for (int ch = 0; ch < A.nchunk; ++ch) {
    if (ch) {
      stage<T>(S, blob + (int64_t)(A.chunk0 + ch) * kStageBlob, msrc + (int64_t)(A.chunk0 + ch) * kStageMat, mt, ct,
               [] {});
      __syncthreads();
    }
    const uint2* segs = reinterpret_cast<const uint2*>(S.blob);
    const uint4* ops = reinterpret_cast<const uint4*>(S.blob + kStageOps);
    const int nseg = uni(S.blob[kStageCount]);
    int o = 0;
    for (int g = 0; g < nseg; ++g) {
      if (live) {
        const uint2 sw = segs[g];
        const uint32_t perm = uni(sw.y);
        const SegAddr G(uni(sw.x), tid);
        const int end = o + (int)(perm & 0xffu);
        A2<T> v[kE];
#pragma unroll
        for (int j = 0; j < kE; ++j) v[j] = S.tile[G.at(j)];
        for (; o < end; ++o) {
          const Macro M(ops[o]);
          const T* m = S.mat + M.m0;
          if (M.ry) rys<T, false>(M.ry, m, v, v, [](auto) {});
          if (M.rx) rxs<T, false>(M.rx, m, v, v, [](auto) {});
          if (M.dg) diagonal<T, false>(m, v, v);
          if (M.cx) cnots<T, false>(M.cx, v, v);
          if (M.rare) rare_op<T, false, FULL>(M, m, v, v);
        }
        const SegAddr W = G.permuted(perm);
#pragma unroll
        for (int j = 0; j < kE; ++j) S.tile[W.at(j)] = v[j];
      }
      __syncthreads();
    }
  }
  if (!act) return;
#pragma unroll
  for (int it = 0; it < kE; ++it) {
    const uint32_t ah = (uint32_t)it << tl;
    const A2<T> x = S.tile[swz5(ah | tid)];
    const uint64_t off = base + run_dep(ro, L, ah) + dlo;
    s_out[off] = x;
    if (ck) ck[off] = x;
  }
}

}  // namespace

// One tile per block, 16 amplitudes per thread.  The kernels that read op by
// op from device tables and switched on each op were bound by neither HBM nor
// arithmetic: by one cold scalar load after another (op, then matrix), the
// moves at the end of the switch, and a fp64 wave sum per gradient.  Here a
// pass's tables are gathered into LDS by all threads while the tile's loads
// are in flight, ops come several to a dispatch, the permutation gates that
// end a segment are folded into its addresses, and gradients are summed four
// at a time.  Chunks of 24 macro ops keep four blocks per CU beside a 32 KiB
// tile.  Measured, complex64: a 12-qubit 4-layer circuit 63 -> 31 us forward
// and 160 -> 76 us adjoint (one wave per SIMD: bound by the issue of one
// wave's instructions, about 8 per gate's multiply-add); 33 x 17 qubits, 8
// layers 492 -> 259 us forward (5 passes) and 1484 -> 590 us adjoint (8 -> 5
// passes), 0.50 and 0.70 of VALU issue, 1.1 TB/s.
template <typename T, bool FULL>
__global__ void __launch_bounds__(sizeof(T) == 4 ? 1024 : 512) k_tile_fwd(
    TilePassArg A, const uint32_t* __restrict__ blob, const int32_t* __restrict__ msrc,
    const uint32_t* __restrict__ runoff, const T* __restrict__ mtab, int64_t mstride, const T* __restrict__ ct,
    const A2<T>* st_in, A2<T>* st_out, int64_t sstride, A2<T>* __restrict__ ckout, int zinit) {
  extern __shared__ __align__(32) unsigned char smem[];
  const uint64_t blk = blockIdx.x & ((1ull << A.nblk_log) - 1);
  const uint64_t b = (uint64_t)blockIdx.x >> A.nblk_log;
  fwd_tile<T, FULL>(A, blob, msrc, runoff, mtab + b * mstride, ct, st_in + b * sstride, st_out + b * sstride,
                    ckout ? ckout + b * sstride : nullptr, deposit(blk, A.bmask, A.nblk_log), zinit != 0, smem);
}

// Several programs' passes in one launch (circuits of different qubit
// counts): block -> job by the prefix of the jobs' block counts.
template <typename T>
__global__ void __launch_bounds__(sizeof(T) == 4 ? 1024 : 512) k_tile_fwd_multi(MultiJobs J) {
  extern __shared__ __align__(32) unsigned char smem[];
  int j = 0;
  while (j + 1 < J.njobs && (int64_t)blockIdx.x >= J.job[j + 1].block0) ++j;
  j = __builtin_amdgcn_readfirstlane(j);  // block-uniform
  const MultiJob& Q = J.job[j];
  const uint64_t lb = (uint64_t)blockIdx.x - Q.block0;
  const uint64_t blk = lb & ((1ull << Q.pass.nblk_log) - 1);
  const uint64_t b = lb >> Q.pass.nblk_log;
  A2<T>* s = (A2<T>*)Q.state + b * Q.sstride;
  const T* mt = (const T*)Q.mtab + b * Q.mstride;
  const uint64_t base = deposit(blk, Q.pass.bmask, Q.pass.nblk_log);
  if (Q.pass.full)
    fwd_tile<T, true>(Q.pass, (const uint32_t*)Q.blob, (const int32_t*)Q.msrc, (const uint32_t*)Q.runoff, mt,
                      (const T*)Q.ctab, s, s, nullptr, base, Q.zinit != 0, smem);
  else
    fwd_tile<T, false>(Q.pass, (const uint32_t*)Q.blob, (const int32_t*)Q.msrc, (const uint32_t*)Q.runoff, mt,
                       (const T*)Q.ctab, s, s, nullptr, base, Q.zinit != 0, smem);
}

namespace {

// Gradient partials of one wave.  A trainable gate leaves one value per
// lane; four gates are collected in LDS ([gate][lane]) and summed together,
// each 16-lane row taking one gate (16 lanes x 4 values, fp64): a quarter of
// the cross-lane steps of one wave sum per gate.
template <typename T>
struct GradSink {
  T* buf;
  double* red;  // [gate of the chunk][wave]
  int wv, nw, lane, cnt;
  bool act;
  __device__ __forceinline__ void flush(int first) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int q = lane >> 4;
    const T* r = buf + q * kGRow<T> + (lane & 15) * 4;
    double x = ((double)r[0] + (double)r[1]) + ((double)r[2] + (double)r[3]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    x += dpp_shr<0x111>(x);
    x += dpp_shr<0x112>(x);
    x += dpp_shr<0x114>(x);
    x += dpp_shr<0x118>(x);
    if ((lane & 15) == 15 && first + q < cnt) red[(first + q) * nw + wv] = x;
  }
  __device__ __forceinline__ void push(T x) {
    buf[(cnt & 3) * kGRow<T> + lane] = act ? x : T(0);
    ++cnt;
    if ((cnt & 3) == 0) flush(cnt - 4);
  }
  __device__ __forceinline__ void finish() {
    if (cnt & 3) flush(cnt & ~3);
  }
};

// Im <l|G|p> of a trainable gate on the registers
template <typename T, bool FULL>
__device__ __forceinline__ T grad_staged(const A2<T>* p, const A2<T>* l, int gen, int s0, int s1, const T* gm) {
  T a = 0;
  switch (gen) {
    case GN_X: TCM_SW1(kR, s0, a = (g_x<T, kR, S_>(p, l))) break;
    case GN_Y: TCM_SW1(kR, s0, a = (g_y<T, kR, S_>(p, l))) break;
    case GN_Z: TCM_SW1(kR, s0, a = (g_z<T, kR, S_>(p, l))) break;
    case GN_P1: TCM_SW1(kR, s0, a = (g_p1<T, kR, S_>(p, l))) break;
    case GN_XX: TCM_SW2(kR, s0, s1, a = (g_xx<T, kR, A_, B_>(p, l))) break;
    case GN_YY: TCM_SW2(kR, s0, s1, a = (g_yy<T, kR, A_, B_>(p, l))) break;
    case GN_ZZ: TCM_SW2(kR, s0, s1, a = (g_zz<T, kR, A_, B_>(p, l))) break;
    case GN_M1: {
      T m[8];
      load_mat<T, 8>(m, gm);
      TCM_SW1(kR, s0, a = (g_m1<T, kR, S_>(p, l, m)))
    } break;
    case GN_M2:
      if constexpr (FULL) {
        T m[32];
        load_mat<T, 32>(m, gm);
        TCM_SW2(kR, s0, s1, a = (g_m2<T, kR, A_, B_>(p, l, m)))
      }
      break;
    default: break;
  }
  return a;
}

// partials of the diagonal gates merged into one op, from im[j] =
// Im(conj(l_j) p_j): the four Z sums share one butterfly
template <typename T>
__device__ __forceinline__ void grad_members(const A2<T>* p, const A2<T>* l, const uint32_t* mems, int n,
                                             GradSink<T>& sink) {
  T im[kE];
#pragma unroll
  for (int j = 0; j < kE; ++j) im[j] = imcj<T>(l[j], p[j]);
  T z[kR], v[kE];
#pragma unroll
  for (int j = 0; j < kE; ++j) v[j] = im[j];
#pragma unroll
  for (int s = 0; s < kR; ++s) {
    z[s] = T(0);
#pragma unroll
    for (int j = 0; j < (kE >> s); j += 2) {
      z[s] += v[j] - v[j + 1];
      v[j >> 1] = v[j] + v[j + 1];
    }
  }
  for (int q = 0; q < n; ++q) {
    const uint32_t w = uni(mems[q]);
    const int s0 = (w >> 4) & 7, s1 = (w >> 7) & 7;
    T a = T(0);
    switch (w & 15u) {
      case GN_Z: a = s0 == 0 ? z[0] : s0 == 1 ? z[1] : s0 == 2 ? z[2] : z[3]; break;
      case GN_P1: TCM_SW1(kR, s0, a = (gm_p1<T, kR, S_>(im))) break;
      case GN_ZZ: TCM_SW2(kR, s0, s1, a = (gm_zz<T, kR, A_, B_>(im))) break;
      default: break;
    }
    sink.push(a);
  }
}

}  // namespace

// Reverse sweep over one pass.  psi/lambda are read from psi_in/lam_in, gates
// are undone in reverse order (the tables are in processing order), gradient
// partials of the pass's trainable gates are reduced per tile into
// part[b][gloc][blk], and the tiles are written to psi_out (nullable: a
// checkpoint replaces it, or it is not read again) and lam_out (nullable).
// psi and lambda pass through one LDS tile, one after the other: twice the
// amplitudes per tile that two tiles would hold at the same number of blocks
// per CU, and with that fewer passes (5 instead of 8 on 17 qubits).
template <typename T, bool FULL>
__global__ void __launch_bounds__(sizeof(T) == 4 ? 1024 : 512) k_tile_adj(
    TilePassArg A, const uint32_t* __restrict__ blob, const int32_t* __restrict__ msrc,
    const uint32_t* __restrict__ runoff, const T* __restrict__ mtab, int64_t mstride, const T* __restrict__ ct,
    const A2<T>* psi_in, A2<T>* psi_out, const A2<T>* lam_in, A2<T>* lam_out, int64_t sstride,
    double* __restrict__ part, int64_t pstride, const double* __restrict__ epart, int eslots) {
  extern __shared__ __align__(32) unsigned char smem[];
  const int tl = A.k - kR, L = A.L, nbl = A.nblk_log;
  const uint32_t nthr = 1u << tl;
  const uint32_t tid = threadIdx.x & (nthr - 1);
  const int nw = blockDim.x >> 6;
  const Lds<T> S(smem, A.k, nw);
  const uint64_t blk = blockIdx.x & ((1ull << nbl) - 1);
  const uint64_t b = (uint64_t)blockIdx.x >> nbl;
  const uint64_t base = b * sstride + deposit(blk, A.bmask, nbl);
  const T* mt = mtab + b * mstride;
  const uint32_t* ro = runoff + A.runoff0;
  const uint32_t dlo = run_dep(ro, L, tid);
  GradSink<T> sink;
  sink.wv = threadIdx.x >> 6;
  sink.nw = nw;
  sink.lane = threadIdx.x & 63;
  sink.buf = S.grad + sink.wv * 4 * kGRow<T>;
  sink.red = S.red;
  sink.act = threadIdx.x < nthr;
  A2<T> p[kE], l[kE];
  stage<T>(S, blob + (int64_t)A.chunk0 * kStageBlob, msrc + (int64_t)A.chunk0 * kStageMat, mt, ct, [&] {
#pragma unroll
    for (int it = 0; it < kE; ++it) p[it] = psi_in[base + run_dep(ro, L, (uint32_t)it << tl) + dlo];
#pragma unroll
    for (int it = 0; it < kE; ++it) l[it] = lam_in[base + run_dep(ro, L, (uint32_t)it << tl) + dlo];
    // lambda = H psi of the first pass becomes (H - E) psi: <psi|G|psi> is real
    // for every generator, so no gradient changes, but where the energy is
    // large beside its spread, as near the end of a variational run, lambda
    // loses most of its length and the roundings on it theirs (hea gradients
    // against 64 bits, rms over 24 seeds: 12 qubits 1.12e-6 -> 0.65e-6, 16
    // qubits 1.68e-6 -> 0.84e-6), at no measurable time
    if (epart) {
      double e = 0.0;
      for (int s = (int)(threadIdx.x & 63); s < eslots; s += 64) e += epart[((int64_t)b * eslots + s) * 2];
      const T es = (T)wave_all(e);
#pragma unroll
      for (int it = 0; it < kE; ++it) {
        l[it].x -= es * p[it].x;
        l[it].y -= es * p[it].y;
      }
    }
  });
  // p and l start in the tile's own order; then (prev, prev_perm) is their layout
  bool flat = true;
  uint32_t prev = 0, prev_perm = 0;
  // (`t`: the addresses are formed where they are used, not held in registers
  // beside the 64 of p and l)
  auto put = [&](const A2<T>* v) {
    uint32_t t = tid;
    asm volatile("" : "+v"(t));
    if (flat) {
#pragma unroll
      for (int it = 0; it < kE; ++it) S.tile[swz5(((uint32_t)it << tl) | t)] = v[it];
    } else {
      const SegAddr G = SegAddr(prev, t).permuted(prev_perm);
#pragma unroll
      for (int j = 0; j < kE; ++j) S.tile[G.at(j)] = v[j];
    }
  };
  auto get = [&](A2<T>* v, uint32_t word) {
    uint32_t t = tid;
    asm volatile("" : "+v"(t));
    const SegAddr G(word, t);
#pragma unroll
    for (int j = 0; j < kE; ++j) v[j] = S.tile[G.at(j)];
  };
  for (int ch = 0; ch < A.nchunk; ++ch) {
    if (ch) {
      __syncthreads();  // the chunk before (and its sums) have been read
      stage<T>(S, blob + (int64_t)(A.chunk0 + ch) * kStageBlob, msrc + (int64_t)(A.chunk0 + ch) * kStageMat, mt, ct,
               [] {});
    }
    __syncthreads();
    const uint2* segs = reinterpret_cast<const uint2*>(S.blob);
    const uint4* ops = reinterpret_cast<const uint4*>(S.blob + kStageOps);
    const uint32_t* mems = S.blob + kStageMems;
    const int nseg = uni(S.blob[kStageCount]);
    sink.cnt = 0;
    int o = 0;
    for (int g = 0; g < nseg; ++g) {
      const uint2 sw = segs[g];
      const uint32_t word = uni(sw.x), perm = uni(sw.y);
      const int end = o + (int)(perm & 0xffu);
      if (flat || word != prev || (prev_perm >> 8) != kPermNone) {
        put(p);
        __syncthreads();
        get(p, word);
        __syncthreads();
        put(l);
        __syncthreads();
        get(l, word);
        __syncthreads();
        flat = false;
        prev = word;
      }
      prev_perm = perm;
      for (; o < end; ++o) {
        const Macro M(ops[o]);
        const T* m = S.mat + M.m0;
        if (M.cx) cnots<T, true>(M.cx, p, l);
        if (M.nmem) grad_members<T>(p, l, mems + M.mem0, (int)M.nmem, sink);
        if (M.dg) diagonal<T, true>(m, p, l);
        if (M.rx) rxs<T, true>(M.rx, m, p, l, [&](auto s) {
          if (M.grx & (1u << s)) sink.push(g_x<T, kR, s>(p, l));
        });
        if (M.ry) rys<T, true>(M.ry, m, p, l, [&](auto s) {
          if (M.gry & (1u << s)) sink.push(g_y<T, kR, s>(p, l));
        });
        if (M.rare) {
          if (M.gen) sink.push(grad_staged<T, FULL>(p, l, (int)M.gen, (int)M.s0, (int)M.s1, S.mat + M.gm));
          rare_op<T, true, FULL>(M, m, p, l);
        }
      }
    }
    sink.finish();
    const int ng = uni(S.blob[kStageCount + 1]);
    if (ng) {
      __syncthreads();
      for (int e = threadIdx.x; e < ng; e += blockDim.x) {
        double s = 0.0;
        for (int w = 0; w < nw; ++w) s += S.red[e * nw + w];
        part[b * pstride + ((int64_t)S.blob[kStageGl + e] << nbl) + blk] = s;
      }
    }
  }
  __syncthreads();
  auto store = [&](const A2<T>* v, A2<T>* out) {
    put(v);
    __syncthreads();
    if (sink.act) {
#pragma unroll
      for (int it = 0; it < kE; ++it) {
        const uint32_t ah = (uint32_t)it << tl;
        out[base + run_dep(ro, L, ah) + dlo] = S.tile[swz5(ah | tid)];
      }
    }
  };
  if (psi_out) {
    store(p, psi_out);
    __syncthreads();
  }
  if (lam_out) store(l, lam_out);
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
namespace {

template <typename T>
size_t lds_fwd(int k) { return (sizeof(A2<T>) << k) + kStageMat * sizeof(T) + kStageBlob * 4; }
template <typename T>
size_t lds_adj(int k, int nw) {
  return lds_fwd<T>(k) + (size_t)nw * (kStageGrad * sizeof(double) + 4 * kGRow<T> * sizeof(T));
}

unsigned threads_of(const DPass& P) { return std::max(64u, 1u << (P.k - kR)); }

// launch(b0, nb) for batch items b0 .. b0 + nb - 1, all at once unless they
// are too many threads
template <typename F>
void batch_parts(const DPass& P, int64_t batch, F launch) {
  const int64_t part = std::max<int64_t>(1, (kMaxLaunchThreads / threads_of(P)) >> P.nblk_log);
  for (int64_t b0 = 0; b0 < batch; b0 += part) launch(b0, std::min(part, batch - b0));
}

}  // namespace

TilePassArg tile_pass_arg(const DPass& P) {
  TilePassArg A{};
  A.k = P.k;
  A.L = P.L;
  A.nblk_log = P.nblk_log;
  A.runoff0 = P.runoff0;
  A.chunk0 = P.chunk0;
  A.nchunk = P.nchunk;
  A.full = P.full;
  for (int i = 0; i < P.nblk_log; ++i) A.bmask |= 1ull << P.blk_bits[i];
  return A;
}

template <typename T>
void launch_tile_fwd(const Sched& S, const DeviceTables& D, int pi, const void* mtab, const void* ctab,
                     const void* in, void* out, int64_t batch, int n, void* ckout, bool zinit, hipStream_t st) {
  const DPass& P = S.dpass[pi];
  const size_t lds = lds_fwd<T>(P.k);
  auto go = [&](auto kern) {
    allow_lds((const void*)kern, lds);
    batch_parts(P, batch, [&](int64_t b0, int64_t nb) {
      const int64_t o = b0 << n;
      hipLaunchKernelGGL(kern, dim3((unsigned)(nb << P.nblk_log)), dim3(threads_of(P)), lds, st, tile_pass_arg(P),
                         (const uint32_t*)D.blob, (const int32_t*)D.msrc, (const uint32_t*)D.runoff,
                         (const T*)mtab + b0 * S.mtab_size, (int64_t)S.mtab_size, (const T*)ctab,
                         zinit ? nullptr : (const A2<T>*)in + o, (A2<T>*)out + o, (int64_t)1 << n,
                         ckout ? (A2<T>*)ckout + o : nullptr, zinit ? 1 : 0);
    });
  };
  if (P.full) go(k_tile_fwd<T, true>);
  else go(k_tile_fwd<T, false>);
}

template <typename T>
void launch_tile_fwd_multi(const MultiJobs& J, int64_t blocks, int threads, int k, hipStream_t st) {
  const size_t lds = lds_fwd<T>(k);
  allow_lds((const void*)k_tile_fwd_multi<T>, lds);
  hipLaunchKernelGGL((k_tile_fwd_multi<T>), dim3((unsigned)blocks), dim3((unsigned)threads), lds, st, J);
}

template <typename T>
void launch_tile_adj(const Sched& S, const DeviceTables& D, int pi, const void* mtab, const void* ctab,
                     const void* psi_in, void* psi_out, const void* lam_in, void* lam_out, int64_t batch, int n,
                     double* part, int64_t pstride, hipStream_t st, const double* epart, int eslots) {
  const DPass& P = S.dpass[pi];
  const unsigned thr = threads_of(P);
  const size_t lds = lds_adj<T>(P.k, (int)(thr / 64));
  auto go = [&](auto kern) {
    allow_lds((const void*)kern, lds);
    batch_parts(P, batch, [&](int64_t b0, int64_t nb) {
      const int64_t o = b0 << n;
      hipLaunchKernelGGL(kern, dim3((unsigned)(nb << P.nblk_log)), dim3(thr), lds, st, tile_pass_arg(P),
                         (const uint32_t*)D.blob, (const int32_t*)D.msrc, (const uint32_t*)D.runoff,
                         (const T*)mtab + b0 * S.mtab_size, (int64_t)S.mtab_size, (const T*)ctab,
                         (const A2<T>*)psi_in + o, psi_out ? (A2<T>*)psi_out + o : nullptr, (const A2<T>*)lam_in + o,
                         lam_out ? (A2<T>*)lam_out + o : nullptr, (int64_t)1 << n, part + b0 * pstride, pstride,
                         epart ? epart + 2 * b0 * eslots : nullptr, eslots);
    });
  };
  if (P.full) go(k_tile_adj<T, true>);
  else go(k_tile_adj<T, false>);
}

#define TCM_TP_INST(T)                                                                                              \
  template void launch_tile_fwd<T>(const Sched&, const DeviceTables&, int, const void*, const void*, const void*,   \
                                   void*, int64_t, int, void*, bool, hipStream_t);                                  \
  template void launch_tile_fwd_multi<T>(const MultiJobs&, int64_t, int, int, hipStream_t);                         \
  template void launch_tile_adj<T>(const Sched&, const DeviceTables&, int, const void*, const void*, const void*,   \
                                   void*, const void*, void*, int64_t, int, double*, int64_t, hipStream_t,    \
                                   const double*, int);
TCM_TP_INST(float)
TCM_TP_INST(double)

}  // namespace tcm

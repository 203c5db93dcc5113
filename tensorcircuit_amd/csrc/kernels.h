// Declarations shared by kernels.hip (device code + launchers) and
// engine.cpp (the C ABI).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "tcm_internal.h"

namespace tcm {

template <typename T>
struct V2T;
template <>
struct V2T<float> {
  using type = float2;
};
template <>
struct V2T<double> {
  using type = double2;
};
template <typename T>
using V2 = typename V2T<T>::type;

// Pauli-sum device descriptors
struct DPGroup {
  uint64_t flip;   // X/Y positions (index bits)
  int32_t t0, nt;  // terms
  int32_t slot0;   // first energy-partial slot of this group
  int32_t nblk;    // blocks launched (= slots used)
};
struct DPTerm {
  uint64_t yz;     // Y/Z positions (index bits)
  int32_t ny;      // number of Y factors
  int32_t pad;
  double w;        // weight
};

// LDS-tiled Pauli passes: every term whose X/Y positions lie in the tile is
// evaluated from one read of psi
struct DPPass {
  int32_t k, L, nblk_log, runoff0;
  int32_t g0, ng;      // groups of this pass
  int32_t nthr_log;    // threads per block (log2)
  int32_t slot0;       // first energy-partial slot
  int32_t c0, nc;      // chunks of its sorted terms (the kernel that is not compiled)
  int32_t blk_bits[32];
};
// Pauli strings kept apart (pauli_terms.hip), sorted by (flip mask, odd
// number of Y, yz): `idx` is the string's place in the caller's order, w holds
// the sign of (-i)^ny, `cnt` counts the group's strings with an even (low
// half) and an odd (high half) number of Y
struct DPTermX {
  double w;
  uint32_t yz, idx;
  uint32_t flip, odd;  // its group's
};
struct DPGroupX {
  uint32_t flip, cnt;
};
// strings a block of k_pauli_terms takes (DPChunk): 32 and not 128, so that a
// state of few tiles has blocks enough (59 strings, 20 qubits: 24 us, not 28)
constexpr int kTermsChunk = 32;
struct PauliTermTables {
  const void *chunks, *groups, *terms;
};

struct DPGroupT {
  uint32_t flip_t;     // tile-local X/Y mask
  int32_t t0, nt, pad;
};
struct DPTermT {
  uint64_t yz_g;       // Y/Z positions outside the tile (global bits)
  uint32_t yz_t;       // Y/Z positions inside the tile (tile-local bits)
  int32_t ny;
  double w;
};
// the same for k_pauli_tile: w holds the sign of (-i)^ny, `cnt` counts the
// group's terms with a real (low half) and an imaginary (high half)
// coefficient; terms are sorted by (group, imaginary, yz_t), so that those
// with the same high tile bits follow each other for any thread count
struct DPTermS {
  double w;
  uint64_t yz_g;
  uint32_t yz_t, pad;
};
struct DPGroupS {
  uint32_t flip_t, cnt;
};
// what is staged in LDS at a time: at most kPauliChunk terms (and as many
// groups; a group of more terms is continued in the next chunk)
struct DPChunk {
  int32_t g0, ng, t0, nt;
};
constexpr int kPauliChunk = 256;
struct PauliTileArg {
  int32_t L, runoff0, slot0, c0, nc, pad;
  uint64_t bmask;      // index bits outside the tile
};
constexpr int kPauliPasses = 16;  // passes of one launch
struct PauliTileArgs {
  int32_t k, nblk_log;  // the same for all passes of a schedule
  PauliTileArg p[kPauliPasses];
};
struct PauliTileTables {
  const void *chunks, *groups, *terms, *runoff;
};

// one table-driven tile pass, by value
struct TilePassArg {
  int32_t k, L, nblk_log, runoff0, chunk0, nchunk, full, pad;
  uint64_t bmask;      // index bits outside the tile
};
// one program's pass inside a multi-program launch (passed by value)
struct MultiJob {
  const void *blob, *msrc, *runoff, *ctab, *mtab;
  void* state;
  int64_t mstride, sstride;
  int64_t block0;   // first block of this job in the launch
  TilePassArg pass;
  int32_t zinit, pad;
};
constexpr int kMaxMultiJobs = 24;
struct MultiJobs {
  int32_t njobs, pad;
  MultiJob job[kMaxMultiJobs];
};

// device copies of one schedule's descriptors (owned by the program)
struct DeviceTables {
  void* dpass = nullptr;
  void* dop = nullptr;
  void* ukbits = nullptr;
  void* runoff = nullptr;
  void* blob = nullptr;
  void* msrc = nullptr;
  void* recipes = nullptr;
  void* factors = nullptr;
  void* gop_list = nullptr;
  void* gop_sum = nullptr;
  // program-wide (shared by both schedules of a dtype, owned by mode 0)
  void* ctab = nullptr;    // constant matrices in T
  void* p_ptr = nullptr;
  void* p_gops = nullptr;
  void* gfac = nullptr;
  // pass compiler: loaded modules and kernel handles (hipModule_t / hipFunction_t)
  std::vector<void*> jit_mod;
  std::vector<void*> jit_fn;
};

// kernels that need more than 64 KiB of dynamic LDS opt in once per device
void allow_lds(const void* kern, size_t bytes);

// launch compiled pass kernels (jit.cpp)
int jit_load(const Sched& S, DeviceTables& D);
// zinit: the pass starts from |0..0> instead of reading `src` (`state` or others)
int jit_launch_fwd(const Sched& S, const DeviceTables& D, int pi, int dt, const void* mtab, const void* ctab,
                   const void* src, void* state, int64_t batch, int n, void* ckout, hipStream_t st, int zinit = 0);
int jit_launch_adj(const Sched& S, const DeviceTables& D, int pi, int dt, const void* mtab, const void* ctab,
                   const void* psi_in, void* psi_out, const void* lam_in, void* lam_out, int64_t batch, int n,
                   double* part, int64_t pstride, hipStream_t st);

// most threads of a launch whose blocks are one per tile or parameter set: one
// of 2^32 or more is cut short without an error
constexpr int64_t kMaxLaunchThreads = 1ll << 31;

// matrix tables of up to kMaxPrepJobs schedules in one launch, and of at most
// kMaxPrepItems batch items (of at most 256 threads each)
constexpr int kMaxPrepJobs = 16;
constexpr int64_t kMaxPrepItems = kMaxLaunchThreads / 256;
struct PrepJob {
  const void *rec, *fac, *params, *ctab;
  void* mtab;
  int64_t pstride, mstride, block0, batch;
  int32_t nrec, first_dg, dg_log, wlog;
};
struct PrepJobs {
  int32_t njobs = 0, widest = 0;
  int64_t items = 0;
  PrepJob job[kMaxPrepJobs];
};
// adds a job; launches the jobs at either limit
template <typename T>
void add_prep(PrepJobs& J, const Sched& S, const DeviceTables& D, const void* ctab, const void* params,
              int64_t pstride, void* mtab, int64_t batch, hipStream_t st);
template <typename T>
void launch_prep(PrepJobs& J, hipStream_t st);
template <typename T>
void launch_init_zero(void* state, int n, int64_t batch, hipStream_t st);
template <typename T>
void launch_copy(void* dst, const void* src, int64_t total, hipStream_t st);
template <typename T, bool DAG>
void launch_plain_gate(const DOp& op, const int32_t* ukbits_dev, const void* mtab, int64_t mstride,
                       const void* ctab, void* state, int n, int64_t batch, hipStream_t st);
// table-driven tile passes (tile_pass.hip); in: the state read, or with zinit
// nothing (the pass starts from |0..0>)
TilePassArg tile_pass_arg(const DPass& P);
template <typename T>
void launch_tile_fwd(const Sched& S, const DeviceTables& D, int pi, const void* mtab, const void* ctab,
                     const void* in, void* out, int64_t batch, int n, void* ckout, bool zinit, hipStream_t st);
// epart: energy partials [batch][eslots] (re, im), at most kMaxShiftSlots; the
// pass then starts from lambda - E psi
constexpr int kMaxShiftSlots = 1024;
template <typename T>
void launch_tile_adj(const Sched& S, const DeviceTables& D, int pi, const void* mtab, const void* ctab,
                     const void* psi_in, void* psi_out, const void* lam_in, void* lam_out, int64_t batch, int n,
                     double* part, int64_t pstride, hipStream_t st, const double* epart, int eslots);
// k: the largest tile of the jobs
template <typename T>
void launch_tile_fwd_multi(const MultiJobs& J, int64_t blocks, int threads, int k, hipStream_t st);
template <typename T>
void launch_plain_adj(const DOp& op, const void* mtab, int64_t mstride, const void* ctab, const void* psi_in,
                      void* psi_out, const void* lam_in, void* lam_out, int64_t batch, int n, int slots, double* part,
                      int64_t pstride, hipStream_t st);
template <typename T>
void launch_plain_adj_uk(const DOp& op, const int32_t* ukbits_dev, const void* ctab, void* psi, void* lam,
                         int64_t batch, int n, hipStream_t st);
template <typename T>
void launch_pauli(const DPGroup& G, const DPTerm* terms_dev, int n, const void* psi, void* out, int first,
                  const double* alpha, double* epart, int64_t estride, int64_t batch, bool energy, bool apply,
                  hipStream_t st);
// np > 1 passes (independent tiles of the same states): energies only
template <typename T>
void launch_pauli_tile(const DPPass* P, int np, const PauliTileTables& D, const void* psi, const void* lam_in,
                       void* lam_out, int n, const double* alpha, double* epart, int64_t estride, int64_t batch,
                       bool energy, bool apply, hipStream_t st);
template <typename T>
void launch_inner(const void* a, const void* c, int n, int64_t batch, int nblk, double* part, int64_t pstride,
                  hipStream_t st);
void launch_sum_slots(const double* part, int64_t bstride, int64_t nslots, int ncomp, double* out, int64_t batch,
                      hipStream_t st);
// measurement
struct MeasureStep {
  int32_t nfree;     // free (not yet measured) index bits, enumerated
  int32_t nrun;      // runs of consecutive free bits
  int32_t bit;       // index bit of the qubit measured in this step
  int32_t first;     // 1 on the first step: no bits fixed yet
  int32_t run[34];   // counter bits src .. src+len-1 -> index bits dst ..
};
// a tile pass of dense 5-qubit blocks on FP32 matrix cores (complex64);
// false if the pass does not fit the kernel (tile bits 10..13, at most
// kMfmaTileMaxOps blocks)
bool launch_mfma_tile(const DPass& P, const DPass* passes_dev, int pi, const DOp* dop_dev, const int32_t* ukbits_dev,
                      const uint32_t* runoff_dev, const void* ctab, const void* src, void* state, int n, int64_t batch,
                      hipStream_t st);
template <typename T>
void launch_probability(const void* psi, void* out, int64_t total, hipStream_t st);
template <typename T>
void launch_pauli_coo(const DPGroup* groups, int ngroups, const DPTerm* terms, int n, int64_t nterms, int64_t* rows,
                      int64_t* cols, void* vals, hipStream_t st);
// per-term Pauli expectations and weighted applications (pauli_terms.hip);
// part: pauli_terms_blocks partial sums per (state, string); far: flip masks
// that leave the tile, complex64 and complex128
int pauli_terms_blocks(int n, bool c64);
int pauli_terms_far(uint32_t flip, int n, bool c64);  // 1 where the flip leaves the tile
template <typename T>
void launch_pauli_terms(const PauliTermTables& D, int nchunks, int nterms, const int* far, int n, const void* psi,
                        int64_t batch, double* part, double* out, hipStream_t st);
template <typename T>
void launch_pauli_terms_apply(const PauliTermTables& D, int nchunks, int nterms, int n, const void* psi, void* out,
                              const double* weights, int64_t batch, hipStream_t st);
// CSR matrices (csr.hip); drowptr null: A = A^dagger
constexpr int kCsrBlocks = 2048;  // most blocks, and partial sums, of a launch
template <typename T>
void launch_csr_matvec(const int64_t* rowptr, const int64_t* cols, const void* vals, const void* x, void* y,
                       int n, int64_t batch, hipStream_t st);
template <typename T>
void launch_csr_vjp(const int64_t* rowptr, const int64_t* cols, const void* vals, const int64_t* drowptr,
                    const int64_t* dcols, const void* dvals, const void* x, const void* g, void* y, int n,
                    int64_t batch, hipStream_t st);
template <typename T>
void launch_csr_expect(const int64_t* rowptr, const int64_t* cols, const void* vals, const void* psi, int n,
                       double* part, double* out, hipStream_t st);
// src: states [batch][2^n] (prob false) or probability vectors (prob true);
// cum: scratch of sample_ws (sample.hip)
constexpr int kSampleChunkLog = 10, kSampleSubLog = 6;
template <typename T>
void launch_sample(const void* src, bool prob, int n, int64_t batch, const double* u, int64_t shots, int64_t* out,
                   double* cum, hipStream_t st);
template <typename T>
void launch_measure_step(const void* psi, int n, int64_t batch, const MeasureStep& M, int k, int nmeas,
                         const double* status, uint64_t* fixval, double* prob, double* outcome, double* part,
                         int nblk, hipStream_t st);
void launch_reduce_gop(const double* part, int64_t pstride, int64_t nslots, const int32_t* gop_list, int gop_single,
                       int ngop_pass, double* gsum, int ngop, int64_t batch, hipStream_t st);
// energies (epart non-null: nslots (re, im) partials per state) and parameter
// gradients from the gop partials (gs) or, gs null, from gsum[b][gop] = part
void launch_finish(const double* epart, int64_t nslots, double* energy, const double* part, const DGopSum* gs, int ngop,
                   const int32_t* p_ptr, const int32_t* p_gops, const double* gfac, double mult, double* grad,
                   int nparams, int max_slots, int64_t batch, hipStream_t st);

}  // namespace tcm

// launch.hpp -- launch argument blocks and host launchers of the kernels.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "desc.hpp"

namespace lsp {

struct FactorLaunch {
    const void *mats;       // FactorDesc<T>[nmat]
    const FactorTask *task;
    const int *active;      // per-matrix mask (nullptr = all)
    int ntask;
    int *epoch;             // device epoch counter: read at start, bumped by the last wave
    int *ctr;               // kQueueInts: queue counters, waves finished
    int *abort_word;
    double *scratch;        // per-wave global fallback
    long scratch_stride;    // doubles per wave slice
    int cap;                // LDS doubles per wave
    int total_waves;
    double ptol;
    double stol;            // > 0: also classify each pivot against splu's choice at this tol
    int *dbg;               // 8 ints: first wait given up (dep, seen, epoch, rounds, column)
    int round_limit;        // a dependency wait gives up after this many polls
    long long *timeline;    // optional, 4 per task (100 MHz wall clock): start, flag
                            // published (end for a dense-block column), end of the
                            // last dependency wait, column
    long long *ticks;       // kTick*: start and end of the launch
    int poll_backoff;       // dependency polls back off to at most poll_backoff + 1 sleeps
    int nq;                 // queue counters (1, 2 or 4) in the ctr block
};

struct TriLaunch {
    const void *mats;       // TriDesc<T>[nmat]
    const int2 *task;       // (matrix, row) in level order
    const long *voff;       // per-matrix vector offsets
    const int *active;      // per-matrix mask (nullptr = all)
    const double *b;        // right-hand sides (original row order)
    double *x;              // solutions (original column order)
    double *y, *z;          // work vectors (position order), unset before the solve
    double *yp, *zp;        // partial sums of supernode rows (position order), unset before the solve
    const double *rs, *cs;  // optional row / column scales (Ruiz): b_s = R b, x = C z
    const int *n_active;    // optional: when *n_active == 0 no circuit is active, tasks are skipped
    long long *timeline;    // optional diagnostic, 2 per task: ticket granted, task finished
    long long *tick0, *tick1;   // optional: start and end of the launch (kTick*)
    int ntask;
    int *ctr;               // kQueueInts: queue counters, waves finished
    int *abort_word;
    int total_waves;
    int nq;                 // queue counters (1, 2 or 4) in the ctr block
};

// Active-circuit counts of a solve: one word per inner iteration in turn, two
// (by the cycle's parity) for the count at a cycle's start.
constexpr int kNact = 5;
#ifdef __HIPCC__
__host__ __device__
#endif
inline int nact_word(int cyc, int j) { return j == 0 ? 3 + (cyc & 1) : j % 3; }
// Basis vectors whose dot products the product's kernel takes along.
constexpr int kSpmvDots = 4;

struct KrylovArgs {
    int nmat;
    int mmax;               // restart length m
    long ntot;              // arena length
    const long *voff;       // per matrix
    const int4 *chunks;     // (matrix, r0, r1, 0)
    int nchunks;
    const int *cbeg;        // nmat+1 chunk ranges per matrix
    const int *sbeg;        // nmat+1 ranges of the product's workgroups per matrix
    double *V;              // basis, (mmax+1) * ntot
    double *w;              // the vector being orthogonalised
    double *spartial;       // sums of the product's workgroups (2 or kSpmvDots each)
    double *partial;        // nchunks * (mmax+1): V^T w after the first pass
    double *partial2;       // nchunks * (mmax+1): V^T w before it (more than kSpmvDots vectors)
    double *pnorm;          // nchunks: w^T w
    double *folded;         // nmat * max(mmax+1, 2): sums added up by a launch of their own (gmres.hip)
    const int *each;        // nmat+1: 0, 1, 2, .. (their parts: one per matrix)
    long sreads, creads;    // sums over the matrices of chunks times product parts / chunk parts
    double *H;              // nmat * (mmax+1) * mmax, H[i*mmax + j]
    double *cs, *sn;        // nmat * mmax
    double *g;              // nmat * (mmax+1)
    double *yv;             // nmat * mmax
    double *beta;           // nmat: ||r|| at cycle start
    double *nb;             // nmat: ||b||
    int *act;               // nmat: 1 while the inner cycle runs
    int *jfin;              // nmat: inner steps taken in the cycle
    int *conv;              // nmat: 1 once the outer test passed
    int *cycled;            // nmat: 1 if the cycle produced an update
    int *nact;              // kNact words
    double inner_tol, outer_tol;
};

// The solves' work values (position order).
struct UnsetArgs {
    double *y, *yp, *z, *zp;
};

// SELL products of the GMRES cycle (spmv.hip): one workgroup per four slices
// of one matrix, with the sums the next kernel needs.
enum SellMode {
    kSellResidual = 1,      // y = b - A x; sums of y^2 and (first) b^2
    kSellResidual0 = 2,     // the same for x = 0, which is written
    kSellDots = 3           // y = A x; sums of V_i y, i < nv (nv <= kSpmvDots; 0: none)
};
struct SellArgs {
    const int2 *blocks;     // (matrix, first slice)
    int nblocks;
    const int64_t *voff;
    double *x;              // written by kSellResidual0 only
    double *y;
    const double *b;
    const int *mask;        // per matrix: skipped unless mask[m] == run
    int run;
    const int *gate;        // see gated()
    int *zero_word;         // cleared by the launch
    double *partial;
    const double *V;
    long ntot;
    int nv;
    int first;
};
template <typename V>
hipError_t launch_sell_block(const SellDesc<V> *mats, const SellArgs &A, SellMode mode, hipStream_t st);

// One fused IR step over the circuits of a batch (irstep.hip).
struct IrStepArgs {
    const void *descs;      // IrDesc<T>[nmat]
    const double *b;        // right-hand sides (arena, original row order)
    double *x;              // solutions (arena, original column order), updated in place
    double *r;              // residual arena (original row order)
    double *yw;             // work arena (position order) for circuits larger than lds_n
    int *conv;              // per circuit: 1 = converged (the launch leaves it alone)
    double *rn2, *bn2;      // per circuit: ||b - A x||^2 and ||b||^2 at its last step
    double tol2;            // squared relative residual tolerance (< 0: every circuit steps)
    int lds_n;              // doubles of LDS per workgroup for the work vector
    int first;              // 1: x starts at 0 (r = b, x is overwritten rather than updated)
};
template <typename T> hipError_t launch_ir_step(const IrStepArgs &A, int nmat, hipStream_t st);
template <typename T> hipError_t ir_step_set_lds(int lds_n);

// factor.hip
template <typename T> hipError_t launch_refactor(const FactorLaunch &L, int blocks, hipStream_t st);
template <typename T> hipError_t refactor_set_lds(int cap);
constexpr int kFillSlots = 4096;         // factor slots per workgroup of the unset fill
template <typename T>
hipError_t launch_fill_unset(const void *mats, const int *active, const int2 *chunks, int nchunks, int *abort_word,
                             int *dbg, hipStream_t st);

// dense trailing blocks (dense.hip)
// Grids of the dense-block kernels as lists of the work items that exist, so
// that blocks of uneven order in one batch launch no empty workgroups.  Jobs
// are numbered by falling T.
struct DenseGridHost {
    std::vector<int4> lu;                // (job, tile row, tile column) in dependency order
    std::vector<int2> pivot;             // (job, group of 256 columns)
    std::vector<int2> gather, trsv;      // (matrix, group of 4 rows), (matrix, pair of 64-row blocks)
};
struct DenseGrid {
    const int4 *lu = nullptr;
    const int2 *pivot = nullptr, *gather = nullptr, *trsv = nullptr;
    int nlu = 0, npivot = 0, ngather = 0, ntrsv = 0;
};
void dense_grid_lists(const std::vector<int> &T, const std::vector<int> &mat, DenseGridHost &H);
template <typename T>
hipError_t launch_dense_lu(const DenseJob *jobs, const void *mats, const int *active, const DenseGrid &G, int *ctr,
                           int *epoch, int *abort_word, long long *tick1, int blocks, double ptol, double stol,
                           hipStream_t st);
template <typename T>
hipError_t launch_tail_solve(const void *mats, const DenseGrid &G, const long *voff, const int *active,
                             const double *b, double *y, double *yp, double *z, double *x, bool forward,
                             int *abort_word, const double *rs, const double *cs, const int *n_active,
                             long long *tick0, hipStream_t st);

// trisolve.hip
// Stores `bytes` (a multiple of 4) at dst in pinned host memory, then seq at
// *done (export.hip); ctr is zero before and after.
hipError_t launch_export(const void *src, void *dst, size_t bytes, unsigned *ctr, unsigned long long *done,
                         unsigned long long seq, hipStream_t st);

// Solves of the `count` circuits in `list`, one workgroup each, at most `rows`
// unknowns per circuit (localsolve.hip).
template <typename T>
hipError_t launch_local_solve(const TriLaunch &L, bool forward, const int *list, int count, int rows, hipStream_t st);
template <typename T>
hipError_t launch_trisolve_half(const TriLaunch &L, bool forward, int blocks, hipStream_t st);
hipError_t launch_solve_unset(const TriLaunch &L, long n, hipStream_t st);

// spmv.hip
template <typename V>
hipError_t launch_sell_spmv(const SellDesc<V> *mats, const int2 *tasks, int ntask,
                            const int64_t *voff, const double *x, double *y, hipStream_t st);
hipError_t launch_csr_spmv(int n, const int *rowptr, const int *colidx, const double *values,
                           const double *x, double *y, hipStream_t st);
hipError_t launch_csr_spmv_f32(int n, const int *rowptr, const int *colidx, const float *values,
                               const double *x, double *y, hipStream_t st);
template <typename Vout>
hipError_t launch_gather_cast(long count, const int *idx, const double *in, Vout *out,
                              hipStream_t st);

// gmres.hip
hipError_t k_solve_init(int *conv, int nmat, int *abort_word, int *nact, hipStream_t s);
hipError_t k_start(const KrylovArgs &K, const double *r, int cyc, double *hist, const int *gate,
                   const UnsetArgs &U, hipStream_t s);
hipError_t k_chunk_dots(const KrylovArgs &K, int nv, hipStream_t s);
hipError_t k_orth(const KrylovArgs &K, int j, bool first, hipStream_t s);
hipError_t k_basis(const KrylovArgs &K, int j, const UnsetArgs &U, hipStream_t s);
// steps: the most a matrix's cycle had
hipError_t k_update(const KrylovArgs &K, const double *Z, double *x, int steps, const int *gate, hipStream_t s);
hipError_t k_zero_int(int *p, long n, hipStream_t s);
hipError_t k_copy(const double *src, double *dst, long n, hipStream_t s);

// Ruiz equilibration of every circuit's values (one workgroup per circuit).
struct RuizArgs {
    const double *ain;      // values, caller order, all circuits
    double *aout;           // scaled values R A C, same layout
    const int *row, *col;   // per entry: circuit-local original row / column
    const long *aoff;       // ncirc+1 entry offsets
    const long *voff;       // ncirc+1 vector offsets
    double *rs, *cs;        // row / column scales (vector layout)
    unsigned long long *mx; // scratch, vector layout
    const int *active;      // per-circuit mask (nullptr = all)
    int sweeps;
    int pad_;
};
hipError_t launch_ruiz(const RuizArgs &R, int ncirc, hipStream_t st);
hipError_t launch_round_f32(const double *in, float *out, long count, hipStream_t st);
// Factor-only diagonal shift: dst[e] = src[e] + shift*|src[e]| for e in idx[0..nidx).
hipError_t launch_shift(const double *src, double *dst, const long *idx, long nidx, double shift,
                        hipStream_t st);

}  // namespace lsp

// desc.hpp -- per-matrix device descriptors shared by kernels and runtime.
//
// Every kernel works on a table of matrices so that one launch can serve one
// circuit or a whole batch of circuits of uneven size: a task is (matrix,
// index) and the matrix's arrays come from its descriptor.
#pragma once

#include <stdint.h>

namespace lsp {

// Abort codes raised by the persistent kernels.
enum : int {
    kErrNone = 0,
    kErrSpin = 1,        // a dependency wait exceeded its spin limit
    kErrCapacity = 2,    // a column/row exceeded its scratch capacity
};

// Polls after which a wait gives up (seconds), and what the report says was
// seen when the wait was for values and not for a flag.
constexpr int kRoundLimit = 1 << 21;
constexpr int kSeenUnset = -2;

// Ints in one persistent kernel's queue block: up to 4 queue counters, a
// cache line each, and the count of waves finished.
constexpr int kQueueInts = 128;

// Wall-clock ticks the kernels leave in the status block: the device times of
// the launches, without event records between them (each record drained the
// stream and left a gap of 5-7 us).
enum : int {
    kTickFactor0 = 0, kTickFactor1 = 1,  // refactor: first workgroup in, last wave out
    kTickDense1 = 2,                     // dense blocks done (the refactor's end when there are none)
    kTickFwd0 = 3, kTickBwd0 = 4, kTickBwd1 = 5,   // solves: forward start, backward start, end
    kTicks = 8
};

// Status words per matrix written by the refactor (FactorDesc::mstat).
constexpr int kMstat = 8;

// Trisolve task codes at or above kTriPacket name a packet of short rows
// (each lane of a packet row gathers up to kTriPacketLane of its entries);
// codes in [kTriWide, kTriPacket) name one 64-row block of a wide supernode.
constexpr int kTriPacket = 1 << 30;
constexpr int kTriWide = 1 << 29;
constexpr int kTriPacketLane = 4;

// Waves of a one-workgroup solve (localsolve.hip).
constexpr int kLocalSolveWaves = 16;

// One task of the refactor, as the kernel reads it: what it needs to start
// a column's loads, so that they depend on one record and not on a chain of
// pointers.
struct FactorTask {
    int mat, k;             // matrix, column
    int c0;                 // first slot
    int a0, na;             // A(:, k): first entry, count
    int d0;                 // first dependency record
    long long u;            // segment-map cursor
    uint16_t m, dl;         // slots, local slot of the diagonal
    uint16_t ndep;          // dependencies (U slots; left of the dense block)
    uint16_t tail;          // 1: a column of the dense trailing block
    int pad_;
};

// Numeric refactorization over the static column patterns.
template <typename T>
struct FactorDesc {
    const int64_t *cp;      // n+1 slot pointers
    const int *pos;         // slot -> row position
    const int *asrc;        // A entry -> input value index
    const int *aslot;       // A entry -> local slot (-1 skipped duplicate)
    const double *ain;      // input values (fp64, caller order)
    const uint16_t *rel;    // segment maps: local slots of each run's last L rows
    const uint64_t *dep;    // dependency records: first L slot; length of the run's
                            // last L column (16 bits), columns of the run after it
    const int *dst;         // slot -> index in lrow / urow / diag
    const int *dpos;        // n: position of the diagonal row q[k] (pinv[q[k]])
    T *val;                 // column storage of L and U
    T *lrow, *urow, *diag;  // row-wise copies for the trisolve
    int *done;              // per-column epoch flags
    int *mstat;             // kMstat ints: bad pivots, first bad column,
                            // first zero-pivot column, non-finite count,
                            // columns whose pivot splu would not pick, columns
                            // too close to call, first of either, pad
    // dense trailing block (tail_T = 0: none, tail_k0 = n)
    double *tail_S;         // tail_T^2 fp64 work block, column-major
    unsigned long long *tail_colmax;   // tail_T: max |L(i,c)| as bit patterns
    T *tail_F;              // tail_T^2 factor in storage precision (tail_S itself for fp64)
    int n;
    int tail_k0;
    int tail_T;
    int pad_;
};

// Row-gather triangular solves.  Vectors are passed per launch as arena
// bases (original order for b and x, position order for the work vectors),
// matrix m's slice starting at voff[m].
template <typename T>
struct TriDesc {
    const int *lrp, *lci;   // strict L by rows (positions)
    const int *urp, *uci;   // strict U by rows
    const T *lrow, *urow, *diag;
    const int *rowat;       // position -> original row (P)
    const int *q;           // position -> original column (Q)
    const int *twide;       // (supernode start, block) pairs of the wide-supernode block tasks
    // supernodes (rows below tail_k0)
    const T *val;           // column storage of L and U (FactorDesc::val)
    const int *dp;          // n diagonal slots (absolute)
    const int *snend;       // n: one past the last row of i's supernode
    const int *ru;          // n: U(j - ru[j] .. j-1, j) is column j's run in its supernode
    const int *fcut;        // n: end of row i's L entries left of its supernode
    const int *bcut;        // n: start of row i's U entries right of its supernode
    const int *fpk, *bpk;   // row packets forward / backward: [g, count, row codes]
    // dense trailing block: rows [tail_k0, n) are solved with tail_F
    const T *tail_F;        // tail_T^2, column-major, unit-L below / U on and above
    const int *tail_lcut;   // tail_T: end of the sparse part of L row tail_k0 + r
    int *tail_ctr;          // 4 ints: block ticket counter, exit counter, pad
    // one-workgroup solve, forward and backward: first task per wave, tasks
    // and records of four ints each, levels (of the circuits solved that way)
    const int *lwave[2], *ltask[2], *lrec[2];
    int lnlev[2];
    int n;
    int tail_k0;
    int tail_T;
    int pad_;
};

// One dense trailing block to factor (fp64 work in FactorDesc::tail_S, T x T,
// column-major; fixed pivot order), nt x nt tiles of 64 x 64.
struct DenseJob {
    double *P;              // nt * nt packed tiles: the final tiles of L and U as operands
    double *W;              // per panel 2 x 64 x 64: its diagonal block's factors as operands (dense.hip)
    unsigned long long *colmax;
    int *flag;              // nt * nt: epoch of the launch that made the tile final
    int T;
    int nt;
    int mat;                // matrix index (descriptor, mstat, active mask)
    int pad_;
};

// SELL-C-sigma SpMV with C = 64 (one wave per slice, one lane per row).
template <typename V>
struct SellDesc {
    const int64_t *off;     // nslices+1
    const int *rlen;        // per sorted row: stored length
    const int *col;         // slots
    const V *val;           // slots
    const int *perm;        // sorted row -> original row
    int nslices;
    int n;
};

// Fused IR step (irstep.hip): one circuit's arrays.
template <typename T>
struct IrDesc {
    SellDesc<double> A;     // A with fp64 values, for the residual
    const int *lrp, *lci;   // strict L by rows (positions)
    const int *urp, *uci;   // strict U by rows
    const T *lrow, *urow, *diag;
    const T *tail_F;        // dense trailing block, column-major (tail_T = 0: none)
    const int *rowat;       // position -> original row (P)
    const int *q;           // position -> original column (Q)
    const int *tail_lcut;   // tail_T: end of the sparse part of L row tail_k0 + r
    const int *frow, *flvp; // rows below tail_k0 by forward level; nlv_f + 1 level pointers
    const int *brow, *blvp; // the same for the backward solve
    long voff;              // first entry of the circuit in the vector arenas
    int n, tail_k0, tail_T, nlv_f, nlv_b, pad_;
};

}  // namespace lsp

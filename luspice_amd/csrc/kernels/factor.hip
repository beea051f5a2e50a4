// factor.hip -- persistent left-looking numeric refactorization (gfx950).
//
// Reference behaviour: the numeric phase of src/third_party/splu.h:151-206
// (per column: scatter A(:,k), apply every earlier L column j with U(j,k) != 0
// in ascending pivot order, U(:,k) = x on pivotal rows, pivot = x at the
// pivot row, L(:,k) = x / pivot elsewhere) with the pivot sequence and
// pattern fixed by the CPU symbolic analysis, the way a Newton refactor reuses
// them.  The reference launches one kernel per level
// (bench/test_lu_wave.cu:200-217, src/mp/multiblock_lu.cu:423-431); here one
// persistent launch walks every column of every matrix in the batch.
//
// Mapping to CDNA4
//   * one wave64 per column task; tasks come from a global queue in an order
//     that rises along every dependency, so a task only waits on tasks handed
//     out earlier, which are held by running waves: the schedule cannot
//     deadlock whatever the occupancy;
//   * the column's working vector x (fp64) lives in LDS when it fits
//     (cap doubles per wave), else in a per-wave global scratch slice;
//   * a task is one record and a dependency one more, so a column's loads are
//     a chain of four round trips (record; dependency records and A's entries;
//     flags and A's values; L), not ten through pointer arrays;
//   * dependencies are fetched 64 at a time (one lane per dependency) and
//     applied in order, by supernode segment, as soon as a leading group of
//     their flags has been seen; inside the last run, by their values; rows
//     below a segment are reached through 16-bit local slot indices precomputed
//     by the plan, so no search and no atomics touch x;
//   * the finished column's L part is stored with agent-coherent stores and
//     the column's flag is published once they are acknowledged, so no L2
//     write-back / invalidate is needed on either side;
//   * the pivot test (|pivot| >= ptol * max |L(:,k)|, in fp64, wave
//     max-reduction) and the stores read only after the launch (U, diagonal,
//     row-wise copies) follow the flag.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace lsp {


constexpr int kGemvBatch = 16;          // L values in flight per GEMV row pass

// Rows below a run's part in a chunk: row i gets sum_t' L(i, j_t') x[j_t']
// over the run's columns t' in [ta, tb), with L(i, j_t') at column offset
// (tb - t' - 1) + i.  Rows i < tri are the run's own later rows (slots
// s0 + tb + i); the rest are L(:, jl) through the map.  G row chunks of 64
// are processed per pass with B columns' values in flight, so a long run
// keeps G * B loads outstanding; every row is updated once.
template <int G, int B, typename T, typename XP>
__device__ __forceinline__ void run_gemv(const T *val, XP x, const LSP_GLOBAL uint16_t *map, int64_t u, double xc,
                                         int lb, int ta, int tb, int tri, int R, int s0, int lane)
{
    const int bw = tb - ta;
    for (int i0 = 0; i0 < R; i0 += G * kWave) {
        int i[G], slot[G];
        double acc[G];
#pragma unroll
        for (int g = 0; g < G; g++) {
            i[g] = min(i0 + g * kWave + lane, R - 1);
            acc[g] = 0.0;
        }
        // fp64 values: the target slots first, so their map loads overlap the
        // value loads (measured on c1: 3.92 -> 3.69 ms; with fp32 values the
        // same order measured slower, 3.55 -> 3.70 ms, so they load after)
        if constexpr (sizeof(T) == 8) {
#pragma unroll
            for (int g = 0; g < G; g++) slot[g] = i[g] < tri ? s0 + tb + i[g] : (int)*near_el(map + u, (uint32_t)(i[g] - tri));
        }
        for (int q0 = 0; q0 < bw; q0 += B) {
            T v[B][G];
#pragma unroll
            for (int h = 0; h < B; h++) {
                const int tp = ta + min(q0 + h, bw - 1);
                const int base = __builtin_amdgcn_readlane(lb, tp) + (tb - tp - 1);
#pragma unroll
                for (int g = 0; g < G; g++) v[h][g] = ld_coherent_near(gp(val) + (uint32_t)base, (uint32_t)i[g]);
            }
#pragma unroll
            for (int h = 0; h < B; h++) {
                if (q0 + h < bw) {
                    const double w = bcast_f64(xc, ta + q0 + h);
#pragma unroll
                    for (int g = 0; g < G; g++) acc[g] = fma(to_f64(v[h][g]), w, acc[g]);
                }
            }
        }
        if constexpr (sizeof(T) != 8) {
#pragma unroll
            for (int g = 0; g < G; g++) slot[g] = i[g] < tri ? s0 + tb + i[g] : (int)*near_el(map + u, (uint32_t)(i[g] - tri));
        }
        // (all reads of a pass before its writes: its rows are distinct slots,
        // which the compiler cannot know, and one LDS round trip serves them all)
        double xv[G];
#pragma unroll
        for (int g = 0; g < G; g++) xv[g] = x[slot[g]];
#pragma unroll
        for (int g = 0; g < G; g++)
            if (i0 + g * kWave + lane < R) x[slot[g]] = xv[g] - acc[g];
    }
}

// The rows below one dependency whose column has not been seen published: the
// values of L(:, j) are loaded until none is unset (the values array holds the
// unset marker before the launch, and every value is written once, as a
// whole), then applied as run_gemv would.  Used in a column's last run (the
// critical chain inside a supernode), which saves the producer's store
// acknowledgement and the flag round trip.  Row i is slot row0 + i for i < tri,
// map[u + i - tri] past that.  The lanes' unseen flags are looked at once, in
// the shadow of the values.  Returns false when abandoned.
template <int G, typename T, typename XP>
__device__ __forceinline__ bool dep_unset(const T *val, XP x, const LSP_GLOBAL uint16_t *map, int64_t u, double xj,
                                          int base, int row0, int tri, int R, const int *flag, int epoch, int &ok,
                                          int *abort_word, int lane, int *dbg, int j, int k, int limit)
{
    constexpr int H = G < 4 ? G : 4;            // chunks applied at a time
    for (int i0 = 0; i0 < R; i0 += G * kWave) {
        int slot[G];
        T v[G];
        // the rows' slots do not depend on the column's values: they are read
        // while those are polled, not after they arrive
#pragma unroll
        for (int g = 0; g < G; g++) {
            const int i = min(i0 + g * kWave + lane, R - 1);
            slot[g] = i < tri ? row0 + i : (int)*near_el(map + u, (uint32_t)(i - tri));
        }
        int seen = ok;
        if (i0 == 0 && !ok) seen = ld_relaxed(flag) == epoch;
        for (int round = 0;; round++) {
#pragma unroll
            for (int g = 0; g < G; g++)
                v[g] = ld_coherent_near(gp(val) + (uint32_t)base, (uint32_t)min(i0 + g * kWave + lane, R - 1));
            bool miss = false;
#pragma unroll
            for (int g = 0; g < G; g++) miss |= Unset<T>::is(v[g]);
            if (!__any(miss)) break;
            if ((round & 15) == 15 && aborted(abort_word)) return false;
            if (round > limit) {
                give_up(abort_word, dbg, j, kSeenUnset, epoch, round, k);
                return false;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        ok = seen;
#pragma unroll
        for (int g0 = 0; g0 < G; g0 += H) {
            double xv[H];
#pragma unroll
            for (int h = 0; h < H; h++) xv[h] = x[slot[g0 + h]];
#pragma unroll
            for (int h = 0; h < H; h++)
                if (i0 + (g0 + h) * kWave + lane < R) x[slot[g0 + h]] = xv[h] - to_f64(v[g0 + h]) * xj;
        }
    }
    return true;
}

// Before a refactor: marks the factor values of the active matrices' columns
// left of the dense block unset (the block's columns are never polled by
// value), and resets every matrix's status words.  One workgroup per chunk
// (matrix, kFillSlots slots); each matrix has at least one.  Kernels, not
// memsets, so the whole refactor sequence stays capturable in a HIP graph.
template <typename T>
__global__ void __launch_bounds__(256) fill_unset_kernel(const FactorDesc<T> *mats, const int *active,
                                                         const int2 *chunks, int *abort_word, int *dbg)
{
    const int2 ch = chunks[blockIdx.x];
    const FactorDesc<T> M = mats[ch.x];
    const int tid = threadIdx.x;
    if (ch.y == 0 && tid < kMstat)
        M.mstat[tid] = tid == 1 || tid == 2 || tid == 6 ? 0x7fffffff : 0;   // first-column words: none
    if (blockIdx.x == 0) {
        if (dbg && tid < 8) dbg[tid] = -1;
        if (abort_word && tid == 0) *abort_word = 0;
    }
    if (active && !active[ch.x]) return;
    const long n = (long)M.cp[M.tail_k0];
    const long s0 = (long)ch.y * kFillSlots + tid;
#pragma unroll
    for (int u = 0; u < kFillSlots / 256; u++)
        if (s0 + 256 * u < n) M.val[s0 + 256 * u] = Unset<T>::value();
}

// Runs of at most kSmallCols columns with at most 64 rows below, taken up to
// kPack at a time: the loads of all of them (triangle, values, map) are in
// flight together, one round trip instead of two per run, and they are then
// applied in order.  Most runs of a circuit's columns are of this kind (85 to
// 90 % on circuits of 100 to 5000 unknowns).  Together with the task records
// and a register budget of 4 waves per SIMD: refactor of 512 such circuits
// 3686 -> 2505 us (fp64), 3493 -> 2601 us (fp32); kPack = 1: 2630, 2645 us.
constexpr int kPack = 3;
constexpr int kSmallCols = 4;
template <int N> using Int = std::integral_constant<int, N>;
// Ready dependencies of a column's last run from which on they are applied
// together instead of one by one (2 to 12 measured the same).  Values instead
// of flags in the last run: refactor of one circuit of 200 / 1020 / 4999
// unknowns 149 / 161 / 336 -> 120 / 124 / 255 us (fp64), of a 316 x 316 grid
// 2993 -> 2580 us, where a link's 12 row chunks bound the chain.
constexpr int kBulk = 3;

// One column of the left-looking refactorization.  XP is the work vector's
// pointer type: an LSP_LDS pointer when the column fits the wave's LDS slice,
// an LSP_GLOBAL scratch pointer otherwise.
//
// Dependencies are applied by supernode segment.  The U slots of column k
// whose rows j_s .. e-1 are consecutive columns of one supernode D (e =
// min(end of D, k)) form a run; inside the run L(j_t, j_t') is entry
// (t - t' - 1) of column j_t', and below the run every column of D holds
// the same rows (the run's later rows, then L(:, e-1)).  So a run is
//   * a unit-lower triangular solve on the run's x entries, done in registers
//     (lane t holds x[j_t]; step t' broadcasts x[j_t'] with readlane), and
//   * a dense update of the rows below: row i gets sum_t' L(i, j_t') x[j_t'],
//     with the L values read as coalesced runs and one x update per row.
// Columns outside any supernode are runs of length 1.  Slots are taken 64 at
// a time; each lane fetches the metadata and waits on the flag of one slot.
template <typename T, typename XP>
__device__ void factor_column(const LSP_CONST FactorDesc<T> *M, const LSP_CONST FactorTask *tk, XP x,
                              int epoch, int *abort_word, double ptol, double stol, int *dbg, long long *tw,
                              int backoff, int limit, int *tctr, TicketReq &treq)
{
    // chunks of 64 rows per pass of dep_unset (316 x 316 grid with 4 / 8 / 12 / 16:
    // 2781 / 2410 / 2584 / 2819 us fp32; a global x costs registers)
    constexpr bool kLds = std::is_same<XP, LSP_LDS double *>::value;
    constexpr int kWide = kLds ? 8 : 4;
    const int lane = lane_id();
    const int k = tk->k;
    const int c0 = tk->c0;
    const int m = tk->m;
    const int dl = tk->dl;                     // local slot of the diagonal
    const int ndep = tk->ndep;
    const bool tail = tk->tail;
    const LSP_GLOBAL int *pos = gp(M->pos) + c0;
    const LSP_GLOBAL uint64_t *dep = gp(M->dep) + tk->d0;
    const LSP_GLOBAL uint16_t *map = gp(M->rel);
    T *const val = M->val;
    int *const done = M->done;

    // everything the column's record points at, in flight together: the first
    // dependencies' records and the entries of A(:, k)
    int j = -2, ok = 1;
    uint64_t dr = 0;
    {
        int as = -1;
        double av = 0.0;
        const int na = tk->na;
        const LSP_GLOBAL int *aslot = gp(M->aslot) + tk->a0;
        const LSP_GLOBAL int *asrc = gp(M->asrc) + tk->a0;
        const LSP_GLOBAL double *ain = gp(M->ain);
        int src = 0;
        if (lane < na) {
            as = aslot[lane];
            src = asrc[lane];
        }
        if (lane < ndep) {
            j = pos[lane];
            dr = dep[lane];
        }
        for (int i = lane; i < m; i += kWave) x[i] = 0.0;
        wave_fence();
        if (as >= 0) av = ain[src];
        if (lane < ndep) ok = ld_relaxed(done + j) == epoch;
        for (int p = lane + kWave; p < na; p += kWave) {
            const int s = aslot[p];
            if (s >= 0) x[s] = ain[asrc[p]];
        }
        if (as >= 0) x[as] = av;
        wave_fence();
    }

    // A column of the dense trailing block applies only its dependencies
    // outside the block (a prefix of its U slots); the block itself is
    // factored densely afterwards.
    long long u = tk->u;                       // map cursor
    for (int s0 = 0; s0 < ndep; s0 += kWave) {
        const int nd = min(kWave, ndep - s0);
        if (s0 > 0) {
            j = -2;
            dr = 0;
            ok = 1;
            if (lane < nd) {
                j = pos[s0 + lane];
                dr = dep[s0 + lane];
                ok = 0;
            }
        }
        const int *flag = lane < nd ? done + j : nullptr;
        const int lb = (int)(uint32_t)dr;                // first L slot of column j
        const int nl = (int)((uint32_t)(dr >> 32) & 0xffffu);   // length of its run's last L column
        const int after = (int)(dr >> 48);               // columns of its run after it
        const int jp = __shfl_up(j, 1, kWave);
        const int ap = __shfl_up(after, 1, kWave);
        const bool head = lane < nd && (lane == 0 || j != jp + 1 || after != ap - 1);
        const unsigned long long heads = __ballot(head);
        double xc = lane < nd ? (double)x[s0 + lane] : 0.0;
        // Dependencies are applied as soon as a leading group of the chunk's
        // flags has been seen: a column whose last dependency is its
        // predecessor in the same supernode (the critical chain) applies all
        // the others while that one is still being factored, and then only
        // the predecessor's column.  A run that continues past the ready
        // prefix is cut there; its later rows stay in the rows below.
        // Inside the column's last run the dependencies come one by one, a
        // chain step apart: while fewer than kBulk of them are ready, each is
        // applied by its values as they appear (dep_unset), without the flag.
        for (int have = 0; have < nd;) {
            const int aft = __builtin_amdgcn_readlane(after, have);
            const unsigned long long wait = ~(__ballot(ok) >> have);    // (lanes past nd count as ready)
            if (s0 + have + aft + 1 == ndep && wait && __builtin_ctzll(wait) < kBulk) {
                int lane = lane_id();                // opaque, as below
                asm volatile("" : "+v"(lane));
                const int base = __builtin_amdgcn_readlane(lb, have);
                const int R = aft + __builtin_amdgcn_readlane(nl, have);
                const double xj = bcast_f64(xc, have);
                const auto direct = [&](auto g) {
                    return dep_unset<decltype(g)::value>(val, x, map, u, xj, base, s0 + have + 1, aft, R, flag, epoch,
                                                         ok, abort_word, lane, dbg,
                                                         __builtin_amdgcn_readlane(j, have), k, limit);
                };
                if (!(R <= kWave ? direct(Int<1>()) : R <= 4 * kWave ? direct(Int<4>()) : direct(Int<kWide>()))) return;
                if (aft == 0) u += R;
                wave_fence();
                have++;
                if (lane >= have && lane < nd) xc = x[s0 + lane];
                continue;
            }
            const int p = wave_wait_prefix(flag, epoch, abort_word, ok, have, nd, dbg, k, backoff, j, limit);
            if (p < 0) return;                                      // aborted; kernel drains
            if (tw) tw[0] = (long long)wall_clock64();
            unsigned long long hs = (heads & ~((1ull << have) - 1)) | (1ull << have);
            if (p < kWave) hs &= (1ull << p) - 1;
            while (hs) {
                // opaque per step: nothing lane-dependent is hoisted out of the
                // loops (and held in registers through them)
                int lane = lane_id();
                asm volatile("" : "+v"(lane));
                const int ta = __builtin_ctzll(hs);
                const unsigned long long hn = hs & (hs - 1);
                const int tb = hn ? __builtin_ctzll(hn) : p;
                const int bw = tb - ta;
                const int tri = __builtin_amdgcn_readlane(after, tb - 1);   // run rows after this part
                const int nlast = __builtin_amdgcn_readlane(nl, ta);
                const int R = tri + nlast;                // rows below the part
                if (bw <= kSmallCols && R <= kWave) {
                    // this run and the next ones while they are small
                    int pa[kPack], pb[kPack], pR[kPack], slot[kPack];
                    T tv[kPack][kSmallCols - 1], v[kPack][kSmallCols];
                    int np = 0;
                    bool small = true;
#pragma unroll
                    for (int r = 0; r < kPack; r++) {
                        pa[r] = pb[r] = pR[r] = 0;
                        slot[r] = 0;            // (set on every path, or the compiler carries
#pragma unroll                                  //  last round's values through the loop)
                        for (int q = 0; q < kSmallCols; q++) v[r][q] = T(0);
#pragma unroll
                        for (int q = 0; q < kSmallCols - 1; q++) tv[r][q] = T(0);
                        if (small && hs) {
                            const int a = __builtin_ctzll(hs);
                            const unsigned long long h = hs & (hs - 1);
                            const int b = h ? __builtin_ctzll(h) : p;
                            const int w = b - a;
                            const int tr = __builtin_amdgcn_readlane(after, b - 1);
                            const int nr = __builtin_amdgcn_readlane(nl, a);
                            small = w <= kSmallCols && tr + nr <= kWave;
                            if (small) {
                                pa[r] = a;
                                pb[r] = b;
                                pR[r] = tr + nr;
                                if (pR[r] > 0) {
                                    const int i = min(lane, pR[r] - 1);
                                    slot[r] = i < tr ? s0 + b + i : (int)*near_el(map + u, (uint32_t)(i - tr));
#pragma unroll
                                    for (int q = 0; q < kSmallCols; q++)
                                        if (q < w) {
                                            const int base = __builtin_amdgcn_readlane(lb, a + q) + (w - q - 1);
                                            v[r][q] = ld_coherent_near(gp(val) + (uint32_t)base, (uint32_t)i);
                                        }
                                }
#pragma unroll
                                for (int q = 0; q < kSmallCols - 1; q++)
                                    if (q < w - 1) {
                                        const int base = __builtin_amdgcn_readlane(lb, a + q);
                                        const int off = min(max(lane - a - q - 1, 0), w - q - 2);
                                        tv[r][q] = ld_coherent_near(gp(val) + (uint32_t)base, (uint32_t)off);
                                    }
                                if (tr == 0) u += nr;
                                hs = h;
                                np = r + 1;
                            }
                        }
                    }
#pragma unroll
                    for (int r = 0; r < kPack; r++) {
                        if (r < np) {
                            const int w = pb[r] - pa[r];
#pragma unroll
                            for (int q = 0; q < kSmallCols - 1; q++)
                                if (q < w - 1) {
                                    const int tp = pa[r] + q;
                                    const double nx = fma(-to_f64(tv[r][q]), bcast_f64(xc, tp), xc);
                                    xc = (lane > tp && lane < pb[r]) ? nx : xc;
                                }
                            if (w > 1 && lane >= pa[r] && lane < pb[r]) x[s0 + lane] = xc;
                            if (pR[r] > 0) {
                                double acc = 0.0;
#pragma unroll
                                for (int q = 0; q < kSmallCols; q++)
                                    if (q < w) acc = fma(to_f64(v[r][q]), bcast_f64(xc, pa[r] + q), acc);
                                if (lane < pR[r]) x[slot[r]] -= acc;
                                wave_fence();
                                if (lane >= pb[r] && lane < nd) xc = x[s0 + lane];   // later lanes of this chunk
                            }
                        }
                    }
                    wave_fence();
                    continue;
                }
                hs = hn;
                if (bw > 1) {
                    if (bw <= 9) {
                        xc = run_triangle<8>(val, xc, lb, ta, tb, lane);
                    } else {
                        // 16 (fp64 values) or 24 triangle columns in registers
                        // at a time (the same steps in the same order), for the
                        // register budget of 4 waves per SIMD
                        constexpr int kPart = sizeof(T) == 8 ? 16 : 24;
                        for (int t0 = ta; t0 < tb - 1; t0 += kPart)
                            xc = run_triangle<kPart>(val, xc, lb, t0, tb, lane);
                    }
                }
                if (lane >= ta && lane < tb) x[s0 + lane] = xc;
                // rows below this part of the run: the run's later rows, then
                // the rows of L(:, jl) through the map
                // (a narrow part, such as a single column, covers more rows per
                // round trip)
                // (fp64 values: half the columns in flight per pass, for the
                // register budget of 4 waves per SIMD)
                constexpr int kB8 = sizeof(T) == 8 ? 4 : 8;
                if constexpr (!kLds) {
                    run_gemv<4, 4>(val, x, map, u, xc, lb, ta, tb, tri, R, s0, lane);
                } else if (bw >= 8) {
                    if (R > 2 * kWave) run_gemv<4, kB8>(val, x, map, u, xc, lb, ta, tb, tri, R, s0, lane);
                    else run_gemv<1, kGemvBatch>(val, x, map, u, xc, lb, ta, tb, tri, R, s0, lane);
                } else if (R <= kWave) {
                    run_gemv<1, 8>(val, x, map, u, xc, lb, ta, tb, tri, R, s0, lane);
                } else if (bw == 1) {
                    run_gemv<8, 1>(val, x, map, u, xc, lb, ta, tb, tri, R, s0, lane);
                } else if (bw <= 4) {
                    run_gemv<4, 4>(val, x, map, u, xc, lb, ta, tb, tri, R, s0, lane);
                } else {
                    run_gemv<4, kB8>(val, x, map, u, xc, lb, ta, tb, tri, R, s0, lane);
                }
                if (tri == 0) u += nlast;
                wave_fence();
                if (lane >= tb && lane < nd) xc = x[s0 + lane];   // later lanes of this chunk
            }
            have = p;
        }
        wave_fence();
    }
    T *const cv = val + c0;
    if (tail) {
        // U entries above the block are final; the rest of the column is the
        // Schur-complement column S(:, c) = A22(:, c) - L21 U12(:, c).
        const LSP_GLOBAL int *dst = gp(M->dst) + c0;
        const int k0 = M->tail_k0, c = k - k0, T_ = M->tail_T;
        T *const urow = M->urow;
        for (int i = lane; i < ndep; i += kWave) {
            const T v = from_f64<T>(x[i]);
            st_g(&cv[i], v);
            st_g(&urow[dst[i]], v);
        }
        LSP_GLOBAL double *Sc = gp(M->tail_S) + (size_t)c * (size_t)T_;
        for (int r = lane; r < T_; r += kWave) Sc[r] = 0.0;
        wave_fence();                           // same-address stores of one wave stay ordered
        for (int s = ndep + lane; s < m; s += kWave) Sc[pos[s] - k0] = x[s];
        if (lane == 0) gp(M->tail_colmax)[c] = 0ull;
        return;
    }

    // L(:, k) is read by later columns of this launch: coherent stores, then
    // the flag once they are acknowledged.  The pivot test, U, the diagonal
    // and the row-wise copies are needed only after the launch, so they come
    // after the flag, off the dependency chain.
    const double piv = x[dl];
    const double rpiv = 1.0 / piv;             // one division; L = x * (1 / pivot)
    for (int i0 = dl + 1 + lane; i0 < m; i0 += 4 * kWave) {
        double xi[4];
#pragma unroll
        for (int h = 0; h < 4; h++) xi[h] = x[min(i0 + h * kWave, m - 1)];
#pragma unroll
        for (int h = 0; h < 4; h++)
            if (i0 + h * kWave < m) st_coherent(&cv[i0 + h * kWave], from_f64<T>(xi[h] * rpiv));
    }
    store_complete();
    if (tw) tw[1] = (long long)wall_clock64();  // timeline: flag published
    if (lane == 0) st_relaxed(&done[k], epoch);
    // The wave's next ticket is requested now: what follows waits on no
    // other wave, so the ticket is not held behind a dependency, and the
    // atomic's round trip overlaps the bookkeeping.
    treq = ticket_issue(tctr);

    // U, the diagonal and the row-wise copies, four slots per lane at a time
    // (their targets' loads in flight together), and the pivot test's maximum
    // a stored value must be finite in the storage type (65504 for FP16)
    const double vmax = sizeof(T) == 2 ? 65504.0 : sizeof(T) == 4 ? 3.4028234663852886e38 : 1.0e308;
    double amax = 0.0;
    int nonfinite = 0;
    {
        const LSP_GLOBAL int *dst = gp(M->dst) + c0;
        T *const lrow = M->lrow, *const urow = M->urow, *const diag = M->diag;
        const double lmax = vmax * fabs(piv);
        for (int i0 = lane; i0 < m; i0 += 4 * kWave) {
            int d[4];
#pragma unroll
            for (int h = 0; h < 4; h++) d[h] = dst[min(i0 + h * kWave, m - 1)];
#pragma unroll
            for (int h = 0; h < 4; h++) {
                const int i = i0 + h * kWave;
                if (i < m) {
                    const double xi = x[i];
                    const double a = fabs(xi);
                    if (i > dl) {
                        amax = fmax(amax, a);
                        nonfinite |= !(a <= 1.0e308) || !(a <= lmax);
                        st_g(&lrow[d[h]], from_f64<T>(xi * rpiv));
                    } else {
                        nonfinite |= !(a <= vmax);
                        const T v = from_f64<T>(xi);
                        st_g(&cv[i], v);
                        st_g(i < dl ? &urow[d[h]] : &diag[k], v);
                    }
                }
            }
        }
    }
    amax = wave_max(amax);
    nonfinite = __any(nonfinite);
    int *const mstat = M->mstat;
    if (lane == 0) {
        if (piv == 0.0) {
            atomicMin(&mstat[2], k);
        } else if (!(fabs(piv) >= ptol * amax)) {
            atomicAdd(&mstat[0], 1);
            atomicMin(&mstat[1], k);
        }
        if (nonfinite) atomicAdd(&mstat[3], 1);
    }
    if (stol > 0.0) {
        // would splu (tol = stol) pick this pivot on these values?
        const int dpos = gp(M->dpos)[k];
        double dv = -1.0;
        if (dpos > k) {
            for (int i = dl + 1 + lane; i < m; i += kWave)
                if (pos[i] == dpos) dv = fabs(x[i]);
            dv = wave_max(dv);
        }
        if (lane == 0) {
            const int v = splu_pivot_verdict(dpos == k, fabs(piv), amax, dv, stol);
            if (v) {
                atomicAdd(&mstat[v == 1 ? 4 : 5], 1);
                atomicMin(&mstat[6], k);
            }
        }
    }
}

// 4 waves per SIMD: 128 VGPRs (with 141 VGPRs, 3 waves, the fp32 refactor of 512
// circuits took 3062 us instead of 2613).
template <typename T>
__global__ void __launch_bounds__(256, 4) refactor_kernel(FactorLaunch L)
{
    extern __shared__ double lds[];
    const int wv = threadIdx.x >> 6;
    const int waves_per_block = blockDim.x >> 6;
    LSP_LDS double *xl = (LSP_LDS double *)lds + (long)wv * L.cap;
    LSP_GLOBAL double *xg = gp(L.scratch) + ((long)blockIdx.x * waves_per_block + wv) * L.scratch_stride;
    const FactorDesc<T> *mats = (const FactorDesc<T> *)L.mats;
    const int epoch = read_epoch(L.epoch);
    if (blockIdx.x == 0 && threadIdx.x == 0) L.ticks[kTickFactor0] = (long long)wall_clock64();

    const int nq = queue_count(L.nq);
    const int q = queue_index(nq);
    int *const qc = L.ctr + 32 * q;                           // this wave's counter
    TicketReq req{0, -1};
    for (;;) {
        // ticket k of counter q is task k * nq + q; the request comes from
        // the previous column when it reached its bookkeeping
        const int t = (req.leader >= 0 ? ticket_take(req) : wave_ticket(qc)) * nq + q;
        req.leader = -1;
        if (t >= L.ntask) break;
        const int gone = ld_relaxed(L.abort_word);            // in flight with the record
        const LSP_CONST FactorTask *tk = kp(L.task) + t;
        const int mat = tk->mat, m = tk->m;
        if (L.active && !kp(L.active)[mat]) continue;
        if (uniform(gone)) continue;                          // drain
        const LSP_CONST FactorDesc<T> *M = kp(mats) + mat;
        long long tw[2] = {0, 0};               // end of the last wait, flag published
        long long *wp = L.timeline ? tw : nullptr;
        const long long t0 = L.timeline ? (long long)wall_clock64() : 0;
        if (m <= L.cap) {
            factor_column<T>(M, tk, xl, epoch, L.abort_word, L.ptol, L.stol, L.dbg, wp, L.poll_backoff, L.round_limit, qc,
                             req);
        } else if (m <= L.scratch_stride) {
            factor_column<T>(M, tk, xg, epoch, L.abort_word, L.ptol, L.stol, L.dbg, wp, L.poll_backoff, L.round_limit, qc,
                             req);
        } else {
            if (lane_id() == 0) st_relaxed(L.abort_word, kErrCapacity);
        }
        if (L.timeline && lane_id() == 0) {
            long long *r = L.timeline + 4L * t;
            r[0] = t0;
            r[1] = tw[1] ? tw[1] : (long long)wall_clock64();
            r[2] = tw[0];
            r[3] = tk->k;
        }
    }
    // the last wave out re-arms the queue and advances the epoch
    if (leave_queue(L.ctr, nq, L.total_waves)) {
        advance_epoch(L.epoch, epoch);
        L.ticks[kTickFactor1] = L.ticks[kTickDense1] = (long long)wall_clock64();
    }
}

}  // namespace lsp

// ---------------------------------------------------------------------------
// host launchers (C++ linkage, used by the runtime)
// ---------------------------------------------------------------------------
namespace lsp {

template <typename T>
hipError_t launch_refactor(const FactorLaunch &L, int blocks, hipStream_t st)
{
    const size_t lds = (size_t)L.cap * sizeof(double) * 4;
    hipLaunchKernelGGL(refactor_kernel<T>, dim3(blocks), dim3(256), lds, st, L);
    return hipGetLastError();
}

template hipError_t launch_refactor<float>(const FactorLaunch &, int, hipStream_t);
template hipError_t launch_refactor<double>(const FactorLaunch &, int, hipStream_t);
template hipError_t launch_refactor<__half>(const FactorLaunch &, int, hipStream_t);

template <typename T>
hipError_t launch_fill_unset(const void *mats, const int *active, const int2 *chunks, int nchunks, int *abort_word,
                             int *dbg, hipStream_t st)
{
    hipLaunchKernelGGL(fill_unset_kernel<T>, dim3(nchunks), dim3(256), 0, st, (const FactorDesc<T> *)mats, active,
                       chunks, abort_word, dbg);
    return hipGetLastError();
}
template hipError_t launch_fill_unset<float>(const void *, const int *, const int2 *, int, int *, int *, hipStream_t);
template hipError_t launch_fill_unset<double>(const void *, const int *, const int2 *, int, int *, int *, hipStream_t);
template hipError_t launch_fill_unset<__half>(const void *, const int *, const int2 *, int, int *, int *, hipStream_t);

template <typename T>
hipError_t refactor_set_lds(int cap)
{
    const int bytes = cap * (int)sizeof(double) * 4;
    return hipFuncSetAttribute((const void *)refactor_kernel<T>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}
template hipError_t refactor_set_lds<float>(int);
template hipError_t refactor_set_lds<double>(int);
template hipError_t refactor_set_lds<__half>(int);

}  // namespace lsp

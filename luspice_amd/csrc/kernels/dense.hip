// dense.hip -- the dense trailing block of the factorization and of the
// triangular solves (gfx950).
//
// After a fill-reducing column order, the last columns of a circuit matrix
// (the top separators) are nearly dense: on the 316x316 power grid the last
// ~3000 of 99906 positions hold half of all left-looking updates, and every
// one of their levels has width 1.  A left-looking column there is a chain of
// ~3000 dependent vector steps; factoring the block as a dense matrix turns
// the chain into 64-column panels.
//
// Refactorization (fixed pivot order; no pivot search, as in the sparse part):
//   the persistent refactor kernel applies every column outside the block and
//   leaves S = A22 - L21 U12 (fp64, column-major T x T).  Then
//     dense_lu_kernel     factors every block of the batch in one launch, as a
//                         dataflow of 64 x 64 tiles (see there)
//     dense_pivot_kernel  applies the pivot test (|pivot| >= ptol max_i |x_i|,
//                         i.e. ptol * max |L(:,c)| <= 1) and copies the diagonal
//   The factor of the block stays dense: in S itself for fp64 storage (tail_F
//   is S then), else in tail_F, which the tiles fill as they become final.
// Structural zeros stay exactly zero (every product that reaches them has a
// structurally zero factor), so the sparse pattern is reproduced.
//
// Triangular solves: rows of the block are solved after the rows above it
// (forward) and before them (backward):
//   tail_fwd_gather_kernel  yp_T = b_T - L21 y  (one wave per row)
//   tail_trsv_kernel<lower> y_T = L22^-1 yp_T
//   tail_trsv_kernel<upper> z_T = U22^-1 y_T, x[q] = z
// A trsv launch has one workgroup per two 64-row blocks; workgroups take
// tickets in solve order and wait (bounded) only on blocks ticketed earlier,
// accumulating each finished block's contribution as it arrives.  Blocks
// hand over their values as the sparse solves do: y and z are unset before
// the solve and a waiting block polls the values themselves.
#include <algorithm>

#include "common.hpp"
#include "launch.hpp"

namespace lsp {

constexpr int kNb = 64;            // panel width
constexpr int kTile = kNb * kNb;   // doubles per packed tile

__device__ __forceinline__ unsigned long long dbits(double v)
{
    return (unsigned long long)__double_as_longlong(v);
}

// Broadcast of lane `src`'s value to the wave (src wave-uniform).
__device__ __forceinline__ double bcast(double v, int src)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(unsigned)(b & 0xffffffffLL), src);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), src);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// Maxima of 16 non-negative values over the lanes that differ in the four
// lane bits from `top` (8 or 32) down: each step keeps half of the values and
// exchanges the other half.  Returns value i's maximum in the lanes whose
// four bits spell i.
template <int H>
__device__ __forceinline__ void max_halve(double (&a)[16], int lane, int off)
{
    const bool up = lane & off;
#pragma unroll
    for (int i = 0; i < H; i++) {
        const double other = __shfl_xor(up ? a[i] : a[H + i], off, kWave);
        a[i] = fmax(up ? a[H + i] : a[i], other);
    }
}
__device__ __forceinline__ double max_scatter16(double (&a)[16], int lane, int top)
{
    max_halve<8>(a, lane, top);
    max_halve<4>(a, lane, top >> 1);
    max_halve<2>(a, lane, top >> 2);
    max_halve<1>(a, lane, top >> 3);
    return a[0];
}

typedef double v4d __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Diagonal block: LU of a 64 x 64 block held by the four waves of a workgroup,
// wave w its columns 16w .. 16w + 15 as the matrix cores leave them
// (acc[x][e]: row 16x + 4e + lane / 16, column 16w + lane % 16).
// v_mfma_f64_16x16x4f64 takes four columns of L and four rows of U, and a
// register e of acc[x] is those four rows as its right operand, so the block is
// factored in groups of four columns:
//   * wave k factors its own 16 columns: per group it turns the four columns to
//     one row per lane through LDS, eliminates them (the pivot row broadcast by
//     readlane, l = A(i, q) / p through the pivot's reciprocal), and updates its
//     other columns on the matrix cores: the group's rows become U = (4 x 4
//     unit-lower inverse) acc, the rows below lose L U;
//   * one barrier, then the waves w > k apply the four groups the same way and
//     wave k + 1 goes on at once;
//   * wave k meanwhile stores what the panel's other tiles need.
// The panel's other tiles solve with L (or U^T) from the left by the same
// groups, from two operand tiles W: at 64 c + r the entry L (r, c), negated
// below the 4 x 4 diagonal blocks and the blocks' inverses on them; at
// 4096 + 64 c + r the same of U^T.
//
// Bound by the chain of 64 pivots and by one wave's instruction issue: a group
// (four reciprocals, two trips through LDS, two dependent products) takes
// 0.85 us.  Per block, in the launch below on one MI355X, T = 720: 17 us, against
// 21 us with 16-column eliminations on one wave (15 broadcasts and updates a
// step) and 19 us with both 64 x 64 inverses carried along on the vector units.
constexpr int kDgLd = 66;                  // column stride of a panel in LDS (two lanes per bank)
constexpr int kDgPanel = 16 * kDgLd;       // panel: A(i, k0 + q) at q * kDgLd + i
constexpr int kDgInv = 128;                // per group: L4^-1(i, k) at 4k + i, U4^-1(k, j) at 16 + 4k + j
constexpr int kDgBuf = kDgPanel + kDgInv;  // two buffers: panel k + 1 is written while k is read
constexpr size_t kDiagLds = sizeof(double) * 2 * kDgBuf;

// Rows 4e .. 4e + 3 of block t become U = (inverse operand) t, the rows below
// them lose L u; a is the group's operand of this block (rows 4e .. 4e + 3 the
// 4 x 4 inverse, below them -L, above them anything).  Returns U as operand.
__device__ __forceinline__ double group_solve(double a, v4d &t, int e, int li)
{
    const v4d zero = (v4d){0.0, 0.0, 0.0, 0.0};
    const double u = __builtin_amdgcn_mfma_f64_16x16x4f64((li >> 2) == e ? a : 0.0, t[e], zero, 0, 0, 0)[e];
    t[e] = u;
    if (e < 3) t = __builtin_amdgcn_mfma_f64_16x16x4f64((li >> 2) > e ? a : 0.0, u, t, 0, 0, 0);
    return u;
}

// Leaves L\U of the wave's own panel in v (row lane >= 16w, column 16w + q) and
// its U blocks above the panel in acc[x], x < w.
__device__ __forceinline__ void diag_block(double *Wg, double *sm_, int wv, int lane_, v4d (&acc)[4], double (&v)[16])
{
    LSP_LDS double *sm = (LSP_LDS double *)sm_;
    LSP_GLOBAL double *W = gp(Wg);
#pragma unroll 1
    for (int kb = 0; kb < 4; kb++) {
        int lane = lane_;                       // opaque per panel: nothing lane-dependent is hoisted (and spilled)
        asm volatile("" : "+v"(lane));
        const int li = lane & 15, lk = lane >> 4;
        LSP_LDS double *pn = sm + (kb & 1) * kDgBuf, *iv = pn + kDgPanel;
        const int k0 = 16 * kb;
        // acc[y] is row block (kb + y) % 4: the panel's own block is acc[0]
        // throughout (the blocks rotate below), the rows below it acc[1 .. 3 - kb]
        // (all operands are read before the first product; those past the
        // block's end are not used)
        auto apply = [&](int e, double inv) {
            double a[4];
#pragma unroll
            for (int y = 0; y < 4; y++) a[y] = -pn[(4 * e + lk) * kDgLd + k0 + 16 * y + li];
            const double u = group_solve((li >> 2) == e ? inv : a[0], acc[0], e, li);
#pragma unroll
            for (int y = 1; y < 4; y++)
                if (kb + y < 4) acc[y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[y], u, acc[y], 0, 0, 0);
            return u;
        };
        if (wv == kb) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int c = k0 + 4 * e;
                if ((li >> 2) == e) {
#pragma unroll
                    for (int y = 0; y < 4; y++)
                        if (kb + y < 4) {
#pragma unroll
                            for (int r = 0; r < 4; r++) pn[li * kDgLd + k0 + 16 * y + 4 * r + lk] = acc[y][r];
                        }
                }
                wave_fence();
                double *g = v + 4 * e;                  // the group's columns, row lane
#pragma unroll
                for (int q = 0; q < 4; q++) g[q] = pn[(4 * e + q) * kDgLd + lane];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const double lq = lane > c + q ? g[q] * (1.0 / bcast(g[q], c + q)) : 0.0;
                    if (lane > c + q) g[q] = lq;
#pragma unroll
                    for (int j = q + 1; j < 4; j++) g[j] = fma(-lq, bcast(g[j], c + q), g[j]);
                }
#pragma unroll
                for (int q = 0; q < 4; q++) pn[(4 * e + q) * kDgLd + lane] = g[q];
                // L4^-1 (li % 4, lk): column lk by substitution in every lane
                double y[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    y[i] = lk == i ? 1.0 : 0.0;
#pragma unroll
                    for (int m = 0; m < i; m++) y[i] = fma(-bcast(g[m], c + i), y[m], y[i]);
                }
                const double inv = (li & 2) ? ((li & 1) ? y[3] : y[2]) : ((li & 1) ? y[1] : y[0]);
                if (li < 4) iv[32 * e + 4 * lk + li] = inv;
                wave_fence();
                if (e < 3) apply(e, inv);
            }
        }
        __syncthreads();
        if (wv == kb) {
            // operand tiles, while the others update
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const int e = q >> 2, i = lane - k0;
                if (lane >= k0 + 4 * e)
                    st_coherent((double *)&W[(k0 + q) * kNb + lane],
                                i < 4 * e + 4 ? (double)iv[32 * e + 4 * (q & 3) + (i & 3)] : -v[q]);
            }
            // U4^-1 of group lane % 4, row by row
            {
                const int e = lane & 3;
                const LSP_LDS double *d = pn + 4 * e * kDgLd + k0 + 4 * e;
                double rp[4];
#pragma unroll
                for (int k = 0; k < 4; k++) rp[k] = 1.0 / d[k * kDgLd + k];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    double z[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        z[j] = j < k ? 0.0 : rp[k];
                        if (j > k) {
                            double t = 0.0;
#pragma unroll
                            for (int m = k; m < j; m++) t = fma(z[m], d[j * kDgLd + m], t);
                            z[j] = -t * rp[j];
                        }
                        if (lane < 4) iv[32 * e + 16 + 4 * k + j] = z[j];
                    }
                }
                wave_fence();
            }
#pragma unroll
            for (int e = 0; e < 4; e++)
                if ((li >> 2) >= e)
                    st_coherent((double *)&W[kTile + (k0 + 4 * e + lk) * kNb + k0 + li],
                                (li >> 2) == e ? (double)iv[32 * e + 16 + 4 * lk + (li & 3)]
                                               : -(double)pn[li * kDgLd + k0 + 4 * e + lk]);
        } else if (wv > kb) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const double u = apply(e, iv[32 * e + 4 * lk + (li & 3)]);
                st_coherent((double *)&W[kTile + (k0 + 4 * e + lk) * kNb + 16 * wv + li], -u);
            }
        }
        const v4d first = acc[0];
        acc[0] = acc[1];
        acc[1] = acc[2];
        acc[2] = acc[3];
        acc[3] = first;
    }
}

// ---------------------------------------------------------------------------
// The block's LU in one persistent launch over every job of the batch.
//
// Tile (i, j) is one task, done once: it subtracts its products
// L(i, p) U(p, j), p < q = min(i, j), from S in registers as the operand tiles
// become final, then
//   i == j  factors the 64 x 64 block and publishes its inverses (diag_block),
//   i > j   solves with U(q, q): a tile of L,
//   i < j   solves with L(q, q): a tile of U,
// and publishes its flag.  Workgroups of four waves take tasks from a queue
// ordered by the panels that remain (longest block first, then by q), so a
// task only waits on tasks handed out before it, which running workgroups
// hold: the schedule cannot deadlock at any occupancy.  Waits are bounded.
//
// What bounds it: on one large block the chain from diagonal block to diagonal
// block (27 us a panel: the block 17, its edge tiles' solve 3, two hand-offs
// through memory 2, the next block's last product 4); on many blocks the
// workgroups that wait in such chains.  One launch per panel, each updating the
// whole trailing matrix, took 41 us a panel and read and wrote every trailing
// tile once a panel.  T = 1853: 1.25 -> 0.83 ms; T = 720: 0.45 -> 0.31 ms; 420
// blocks of T 64..705, with the former pass that scattered the block into the
// sparse factors: 1.53 -> 0.72 ms.
//
// fp64 matrix cores, v_mfma_f64_16x16x4f64; operands and result sit in the
// lanes as
//   A(i, k): lane i + 16k      B(k, j): lane j + 16k
//   D(i, j): lane j + 16 (i % 4), register i / 4,
// so a D block fed back as B is the same value in the same lane: register r
// of D holds the rows 4r .. 4r + 3 that step r of the next product needs.  A
// wave therefore keeps all 64 rows of 16 columns, and the final solve with
// the diagonal block needs no LDS and no barrier.  A tile of L is computed
// transposed, which makes both kinds the same code: with r, c the result's
// row and column, U has (r, c) = (i, j) and takes L from the left, L has
// (r, c) = (j, i) and takes U from the left.  Final tiles go to a packed copy,
// element (r, c) at 64 r + c, which is the layout both operands of a later
// product are read in (coalesced, no line shared between tiles); L is stored
// negated there, so that the matrix cores subtract.
constexpr int kStage = 4;                  // k-steps of operands per register stage

// One register stage of a product: kStage steps of both operands.
struct TileStage {
    double a[kStage][4], b[kStage];
    __device__ __forceinline__ void load(const double *X, const double *Y, int s0, int wv, int li, int lk)
    {
        const LSP_GLOBAL double *xp = gp(X) + (4 * s0 + lk) * kNb + li;
        const LSP_GLOBAL double *yp = gp(Y) + (4 * s0 + lk) * kNb + 16 * wv + li;
#pragma unroll
        for (int s = 0; s < kStage; s++) {
#pragma unroll
            for (int x = 0; x < 4; x++) a[s][x] = ld_coherent_val(xp, (uint32_t)(4 * s * kNb + 16 * x));
            b[s] = ld_coherent_val(yp, (uint32_t)(4 * s * kNb));
        }
    }
    __device__ __forceinline__ void apply(v4d (&acc)[4]) const
    {
#pragma unroll
        for (int s = 0; s < kStage; s++)
#pragma unroll
            for (int x = 0; x < 4; x++) acc[x] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s][x], b[s], acc[x], 0, 0, 0);
    }
};

template <typename T>
__global__ void __launch_bounds__(256, 2) dense_lu_kernel(const DenseJob *jobs, const void *mats, const int *active,
                                                          const int4 *tasks, int ntask, int *ctr, int *epoch_word,
                                                          int *abort_word, long long *tick1)
{
    extern __shared__ double lds[];
    __shared__ int s_t;
    const int epoch = read_epoch(epoch_word);
    for (;;) {
        // opaque per task: the compiler would otherwise hoist every lane
        // address of the body out of the loop and spill them
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & (kWave - 1), wv = uniform(tid >> 6);
        const int li = lane & 15, lk = lane >> 4;
        // one ticket per workgroup; an abort is seen by all its waves or none
        if (tid == 0) s_t = aborted(abort_word) ? ntask : wave_ticket(ctr);
        __syncthreads();
        const int t = uniform(s_t);
        __syncthreads();
        if (t >= ntask) break;
        const int4 tk = tasks[t];
        const DenseJob J = jobs[tk.x];
        if (active && !active[J.mat]) continue;
        T *F = ((const FactorDesc<T> *)mats)[J.mat].tail_F;
        double *S = ((const FactorDesc<T> *)mats)[J.mat].tail_S;
        const int ti = tk.y, tj = tk.z;
        const int q = min(ti, tj);
        const bool low = ti > tj;                       // a tile of L: (r, c) = (j, i)
        const int nt = J.nt;
        const size_t ld = (size_t)J.T;
        const int *ready = J.flag;
        // the result's rows r come from tile row / column q, its columns c from the other index
        const int r0 = q * kNb, c0 = (low ? ti : tj) * kNb;
        const int c = c0 + 16 * wv + li;
        // S(i, j) at rs * r + cs * c; rows and columns past T are zero (a
        // diagonal block's are the identity's)
        const size_t rs = low ? ld : 1, cs = low ? 1 : ld;
        v4d acc[4];
#pragma unroll
        for (int x = 0; x < 4; x++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = r0 + 16 * x + 4 * e + lk;
                const double v = gp(S)[rs * min(r, J.T - 1) + cs * min(c, J.T - 1)];
                acc[x][e] = r < J.T && c < J.T ? v : (ti == tj && r == c ? 1.0 : 0.0);
            }
        // operand tiles of product p: X left (rows r), Y right (columns c)
        const int xs = low ? nt : 1, xo = low ? q : q * nt;           // L(q, p) or U(p, q)
        const int ys = low ? 1 : nt, yo = low ? ti * nt : tj;         // U(p, j) or L(i, p)
        int ok = 1;
        for (int p0 = 0; p0 < q && ok; p0 += kWave / 2) {
            // lanes 2p, 2p + 1: the flags of product p's two tiles
            const int np = min(kWave / 2, q - p0);
            const int p = p0 + (lane >> 1);
            const int *flag = p < q ? &ready[(lane & 1) ? ys * p + yo : xs * p + xo] : nullptr;
            int seen = flag == nullptr;
            for (int done = 0, have = 0; done < np;) {
                const int pre = wave_wait_prefix(flag, epoch, abort_word, seen, have, 2 * np, nullptr, -1, kSolveBackoff);
                if (pre < 0) {
                    ok = 0;
                    break;
                }
                have = pre;
                const int np1 = (pre >> 1) - done;      // products ready now
                if (np1 <= 0) continue;
                const int pb = p0 + done;
                auto xt = [&](int n) { return J.P + (size_t)(xs * (pb + n) + xo) * kTile; };
                auto yt = [&](int n) { return J.P + (size_t)(ys * (pb + n) + yo) * kTile; };
                static_assert(4 * kStage == 16, "a product is four stages");
                TileStage s0, s1;
                s0.load(xt(0), yt(0), 0, wv, li, lk);
                for (int n = 0; n < np1; n++) {
                    // each product is summed by itself and added once: one
                    // rounding at the magnitude of S per 64 terms, not 64
                    v4d t[4];
#pragma unroll
                    for (int x = 0; x < 4; x++) t[x] = (v4d){0.0, 0.0, 0.0, 0.0};
                    s1.load(xt(n), yt(n), kStage, wv, li, lk);
                    s0.apply(t);
                    s0.load(xt(n), yt(n), 2 * kStage, wv, li, lk);
                    s1.apply(t);
                    s1.load(xt(n), yt(n), 3 * kStage, wv, li, lk);
                    s0.apply(t);
                    if (n + 1 < np1) s0.load(xt(n + 1), yt(n + 1), 0, wv, li, lk);
                    s1.apply(t);
#pragma unroll
                    for (int x = 0; x < 4; x++) acc[x] += t[x];
                }
                done = pre >> 1;
            }
        }
        if (ti == tj) {
            if (!__syncthreads_and(ok)) continue;
            double v[16];
            diag_block(J.W + (size_t)q * 2 * kTile, lds, wv, lane, acc, v);
            store_complete();
            __syncthreads();
            if (tid == 0) st_relaxed(&J.flag[(size_t)q * (nt + 1)], epoch);
            // what only later launches read: the factor in place and in
            // storage precision, and the column maxima of |L|
            auto put = [&](int r, int cc, double f) {
                if (r < J.T && cc < J.T) {
                    gp(S)[ld * cc + r] = f;
                    if constexpr (sizeof(T) != 8) st_g(&F[ld * cc + r], from_f64<T>(f));
                }
            };
            double am[16];
#pragma unroll
            for (int e = 0; e < 16; e++) am[e] = lane > 16 * wv + e && r0 + lane < J.T ? fabs(v[e]) : 0.0;
            double mx = max_scatter16(am, lane, 32);    // lanes 4e .. 4e + 3: column e
            mx = fmax(mx, __shfl_xor(mx, 2, kWave));
            mx = fmax(mx, __shfl_xor(mx, 1, kWave));
            const int mc = r0 + 16 * wv + (lane >> 2);
            if ((lane & 3) == 0 && mc < J.T) atomicMax(&J.colmax[mc], dbits(mx));
            if (lane >= 16 * wv) {
#pragma unroll
                for (int e = 0; e < 16; e++) put(r0 + lane, r0 + 16 * wv + e, v[e]);
            }
#pragma unroll
            for (int x = 0; x < 3; x++)
                if (x < wv) {
#pragma unroll
                    for (int e = 0; e < 4; e++) put(r0 + 16 * x + 4 * e + lk, c, acc[x][e]);
                }
            continue;
        }
        // the panel's triangle from the left, by groups of four rows
        ok = ok && wave_wait(lane == 0 ? &ready[(size_t)q * (nt + 1)] : nullptr, epoch, abort_word, kSolveBackoff);
        if (ok) {
            const LSP_GLOBAL double *wp = gp(J.W) + (size_t)q * 2 * kTile + (low ? kTile : 0) + lk * kNb + li;
            double w[16][4];
#pragma unroll
            for (int s = 0; s < 16; s++)
#pragma unroll
                for (int x = s / 4; x < 4; x++) w[s][x] = ld_coherent_val(wp, (uint32_t)(4 * s * kNb + 16 * x));
#pragma unroll
            for (int s = 0; s < 16; s++) {
                const double u = group_solve(w[s][s / 4], acc[s / 4], s % 4, li);
#pragma unroll
                for (int x = s / 4 + 1; x < 4; x++)
                    acc[x] = __builtin_amdgcn_mfma_f64_16x16x4f64(w[s][x], u, acc[x], 0, 0, 0);
            }
            double *Pt = J.P + (size_t)(ti * nt + tj) * kTile;
#pragma unroll
            for (int x = 0; x < 4; x++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    st_coherent(&Pt[(16 * x + 4 * e + lk) * kNb + 16 * wv + li], low ? -acc[x][e] : acc[x][e]);
            store_complete();
        }
        if (!__syncthreads_and(ok)) continue;
        if (tid == 0) st_relaxed(&J.flag[(size_t)ti * nt + tj], epoch);
        // what only later launches read: the factor in place and in storage
        // precision, and the column maxima of |L| for the pivot test
        // (rows opaque again, or the first loads' addresses stay live)
        int rl = r0 + lk;
        asm volatile("" : "+v"(rl));
        double am[16];
#pragma unroll
        for (int x = 0; x < 4; x++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = rl + 16 * x + 4 * e;
                const bool in = r < J.T && c < J.T;
                am[4 * x + e] = in ? fabs(acc[x][e]) : 0.0;
                if (in) {
                    const size_t at = rs * r + cs * c;
                    gp(S)[at] = acc[x][e];
                    if constexpr (sizeof(T) != 8) st_g(&F[at], from_f64<T>(acc[x][e]));
                }
            }
        if (low) {
            const double mx = max_scatter16(am, lane, 8);   // lane li: register li's row of the result
            const int r = rl + 4 * li;
            if (r < J.T) atomicMax(&J.colmax[r], dbits(mx));
        }
    }
    if (threadIdx.x < kWave && leave_queue(ctr, 1, (int)gridDim.x)) {
        advance_epoch(epoch_word, epoch);
        *tick1 = (long long)wall_clock64();
    }
}

// ---------------------------------------------------------------------------
// One thread per block column: pivot test and the diagonal of the factors.
template <typename T>
__global__ void __launch_bounds__(256) dense_pivot_kernel(const DenseJob *jobs, const void *mats, const int *active,
                                                          double ptol, double stol, const int2 *items)
{
    const int2 tk = items[blockIdx.x];
    const DenseJob J = jobs[tk.x];
    const int c = tk.y * 256 + (int)threadIdx.x;
    if (c >= J.T || (active && !active[J.mat])) return;
    const FactorDesc<T> M = ((const FactorDesc<T> *)mats)[J.mat];
    const double *Sc = M.tail_S + (size_t)c * (size_t)J.T;
    const int k = M.tail_k0 + c;
    const double piv = Sc[c];
    const double lmax = __longlong_as_double((long long)J.colmax[c]);
    M.diag[k] = from_f64<T>(piv);
    if (piv == 0.0) {
        atomicMin(&M.mstat[2], k);
    } else if (!(ptol * lmax <= 1.0)) {
        atomicAdd(&M.mstat[0], 1);
        atomicMin(&M.mstat[1], k);
    }
    const double vmax = sizeof(T) == 2 ? 65504.0 : sizeof(T) == 4 ? 3.4028234663852886e38 : 1.0e308;
    if (!(fabs(piv) <= vmax) || !(lmax <= vmax)) atomicAdd(&M.mstat[3], 1);
    if (stol > 0.0) {
        // splu's choice on these values, in units of |pivot|: the other
        // candidates are the multipliers L(r, c), r > c, of the block
        const int dpos = M.dpos[k];
        const double md = dpos > k ? fabs(Sc[dpos - M.tail_k0]) : -1.0;
        const int v = piv == 0.0 ? (lmax > 0.0 ? 1 : 0) : splu_pivot_verdict(dpos == k, 1.0, lmax, md, stol);
        if (v) {
            atomicAdd(&M.mstat[v == 1 ? 4 : 5], 1);
            atomicMin(&M.mstat[6], k);
        }
    }
}

// ---------------------------------------------------------------------------
// Forward solve, rows of the block: yp[k0 + r] = b[rowat] - L(k0 + r, :k0) y.
template <typename T>
__global__ void __launch_bounds__(256) tail_fwd_gather_kernel(const void *mats, const int2 *groups,
                                                              const long *voff, const int *active,
                                                              const double *b, const double *y, double *yp,
                                                              const double *rs, const int *n_active)
{
    if (n_active && uniform(ld_relaxed(n_active)) == 0) return;
    const int2 tk = groups[blockIdx.x];                // (matrix, group of four rows)
    const int mi = tk.x;
    if (active && !active[mi]) return;
    const TriDesc<T> M = ((const TriDesc<T> *)mats)[mi];
    const int r = tk.y * 4 + (threadIdx.x >> 6);
    if (r >= M.tail_T) return;
    const int lane = lane_id();
    const int i = M.tail_k0 + r;
    const long vo = voff[mi];
    const int e1 = M.tail_lcut[r];
    double acc = 0.0;
    for (int e = M.lrp[i] + lane; e < e1; e += kWave) acc += to_f64(M.lrow[e]) * y[vo + M.lci[e]];
    acc = wave_sum(acc);
    if (lane == 0) {
        const int ro = M.rowat[i];
        yp[vo + i] = (rs ? b[vo + ro] * rs[vo + ro] : b[vo + ro]) - acc;
    }
}

// Dense triangular solve of the block rows (see the file comment), two
// 64-row blocks (128 rows, in solve order) per workgroup:
//   lower: y_T <- L22^-1 yp_T (unit diagonal)
//   upper: z_T <- U22^-1 y_T, x[q] = z (the sparse backward solve, a later
//          launch, reads these z values)
// Waves 2..7 accumulate the contributions of the blocks solved before this
// pair (waves 2, 4, 6 for the first block's rows, 3, 5, 7 for the second's,
// three earlier blocks each in turn): per block the 64 x 64 factor slab (one
// row per lane, in registers) is loaded before the block's values are
// awaited, so the wait overlaps the loads; the polls return the solved
// values, broadcast by readlane.  Waves 0 and 1 hold the two diagonal blocks,
// right-hand sides and diagonal reciprocals.  After the first block is
// solved, the six accumulator waves apply it to the second block's rows (a
// slice of its columns each, from LDS), and wave 1 solves the second block:
// one hand-off through memory per 128 rows instead of per 64.
constexpr int kTailAcc = 6;                 // accumulator waves per workgroup
constexpr int kTailSlice = (kNb + kTailAcc - 1) / kTailAcc;   // coupling columns per accumulator wave

template <typename T, bool kLower>
__global__ void __launch_bounds__(512) tail_trsv_kernel(const void *mats, const int2 *pairs,
                                                        const long *voff, const int *active,
                                                        double *y, const double *yp, double *z, double *x,
                                                        int *abort_word, const double *cs, const int *n_active,
                                                        long long *tick0)
{
    // nothing active: every workgroup returns before it takes a ticket
    if (n_active && uniform(ld_relaxed(n_active)) == 0) return;
    if (tick0 && blockIdx.x == 0 && threadIdx.x == 0) *tick0 = (long long)wall_clock64();
    const int mi = pairs[blockIdx.x].x;                // as many workgroups per matrix as it has pairs
    const TriDesc<T> M = ((const TriDesc<T> *)mats)[mi];
    const int lane = lane_id();
    const int wv = threadIdx.x >> 6;
    __shared__ int s_ticket;
    __shared__ double red[kTailAcc][kWave];            // accumulators' sums over the earlier blocks
    __shared__ double red2[kTailAcc][kWave];           // the first block's contribution to the second's rows
    __shared__ double ys[kWave];                       // the first block's solution
    const bool live = !(active && !active[mi]);
    const int nblk = (M.tail_T + kNb - 1) / kNb;
    const int npair = (nblk + 1) / 2;
    if (live) {
        if (threadIdx.x == 0) s_ticket = atomicAdd(&M.tail_ctr[0], 1);
        __syncthreads();
        const int t = uniform(s_ticket);
        if (t < npair) {
            const size_t ld = (size_t)M.tail_T;
            const long vo = voff[mi];
            const int k0 = M.tail_k0;
            const double *src = kLower ? y : z;
            const int nsub = min(2, nblk - 2 * t);      // blocks in this pair
            // block in solve order so -> its first row
            auto row0 = [&](int so) { return (kLower ? so : nblk - 1 - so) * kNb; };
            // the rows of the pair's block u, clamped per lane
            const int u = wv < 2 ? wv : (wv - 2) & 1;  // the block whose rows this wave handles
            const bool has = u < nsub;
            const int r0 = has ? row0(2 * t + u) : 0;
            const int bi = has ? min(kNb, M.tail_T - r0) : 1;
            const int rr = r0 + min(lane, bi - 1);
            double acc = 0.0;
            bool ok = true;
            T dg[kNb];                                  // waves 0, 1: row lane of the diagonal block
            T fc[kTailSlice];                           // waves 2..7: row of block 1 against a slice of block 0
            double rd = 1.0;                            // waves 0, 1, upper: 1 / U(rr, rr)
            double yb = 0.0;                            // waves 0, 1: right-hand side of row rr
            int qo = 0;                                 // waves 0, 1, upper: output index of row rr
            if (wv < 2) {
                if (has) {
#pragma unroll
                    for (int c = 0; c < kNb; c++) dg[c] = M.tail_F[(size_t)(r0 + min(c, bi - 1)) * ld + rr];
                    if (!kLower) {
                        // zero past the block's end: those lanes then pass zeros
                        rd = lane < bi ? 1.0 / to_f64(M.tail_F[(size_t)rr * ld + rr]) : 0.0;
                        qo = M.q[k0 + rr];
                    }
                    yb = kLower ? yp[vo + k0 + rr] : y[vo + k0 + rr];
                }
            } else {
                if (nsub == 2) {
                    // slice of the coupling block: rows of block 1, columns of block 0
                    // (block 0 is partial only for the upper solve's first pair;
                    // its missing columns meet zeros in ys)
                    const int ra = row0(2 * t), rb = row0(2 * t + 1);
                    const int ba = min(kNb, M.tail_T - ra);
                    const int bb = min(kNb, M.tail_T - rb);
                    const int rr1 = rb + min(lane, bb - 1);
                    const int c0 = (wv - 2) * kTailSlice;
#pragma unroll
                    for (int c = 0; c < kTailSlice; c++)
                        fc[c] = M.tail_F[(size_t)(ra + min(c0 + c, ba - 1)) * ld + rr1];
                }
                if (has) {
                    for (int s = (wv - 2) >> 1; s < 2 * t && ok; s += 3) {
                        const int c0 = row0(s);
                        const int bj = min(kNb, M.tail_T - c0);
                        T fv[kNb];
#pragma unroll
                        for (int c = 0; c < kNb; c++) fv[c] = M.tail_F[(size_t)(c0 + min(c, bj - 1)) * ld + rr];
                        double sv;                                   // zero beyond bj
                        ok = wave_wait_value(lane < bj ? &src[vo + k0 + c0 + lane] : nullptr, sv, abort_word);
                        if (!ok) break;
#pragma unroll
                        for (int c = 0; c < kNb; c++) {
                            const double yc = bcast(sv, c);          // zero beyond bj
                            acc += to_f64(fv[c]) * yc;
                        }
                    }
                }
                red[wv - 2][lane] = has && lane < bi ? acc : 0.0;
            }
            const bool all_ok = __syncthreads_and(ok);
            // triangle of one block on its solver wave: tr = right-hand side
            // minus the contributions gathered, solved in place
            auto solve = [&](double tr) {
                if (kLower) {
#pragma unroll
                    for (int c = 0; c < kNb; c++) {
                        const double yc = bcast(tr, c);
                        if (lane > c && c < bi) tr -= to_f64(dg[c]) * yc;
                    }
                } else {
                    // z_c = tr_c / U(c, c), one broadcast per step; rows past
                    // bi hold tr = 0 and rd = 0 and broadcast zeros.  Row c's
                    // tr is final from step c on, so every row's z is the
                    // same product tr * rd, formed once at the end.
#pragma unroll
                    for (int c = kNb - 1; c >= 0; c--) {
                        const double zc = bcast(tr * rd, c);
                        if (lane < c) tr -= to_f64(dg[c]) * zc;
                    }
                    tr = tr * rd;
                }
                if (lane < bi) {
                    if (kLower) {
                        st_coherent(&y[vo + k0 + rr], tr);
                    } else {
                        st_coherent(&z[vo + k0 + rr], tr);
                        x[vo + qo] = cs ? tr * cs[vo + qo] : tr;
                    }
                }
                return tr;
            };
            if (all_ok && wv == 0) {
                double tr = 0.0;
                if (lane < bi) tr = yb - (red[0][lane] + red[2][lane] + red[4][lane]);
                tr = solve(tr);
                ys[lane] = lane < bi ? tr : 0.0;
            }
            if (nsub == 2) {
                __syncthreads();                        // ys written
                if (all_ok && wv >= 2) {
                    const int c0 = (wv - 2) * kTailSlice;
                    double a2 = 0.0;
#pragma unroll
                    for (int c = 0; c < kTailSlice; c++)
                        if (c0 + c < kNb) a2 += to_f64(fc[c]) * ys[c0 + c];
                    red2[wv - 2][lane] = a2;
                }
                __syncthreads();                        // red2 written
                if (all_ok && wv == 1) {
                    double tr = 0.0;
                    if (lane < bi) {
                        tr = yb - (red[1][lane] + red[3][lane] + red[5][lane]);
#pragma unroll
                        for (int w = 0; w < kTailAcc; w++) tr -= red2[w][lane];
                    }
                    solve(tr);
                }
            }
        }
        // the last workgroup of this matrix re-arms its ticket counter
        if (threadIdx.x == 0) {
            const int fin = atomicAdd(&M.tail_ctr[1], 1);
            if (fin == npair - 1) {
                st_relaxed(&M.tail_ctr[0], 0);
                st_relaxed(&M.tail_ctr[1], 0);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
template <typename T>
hipError_t launch_dense_lu(const DenseJob *jobs, const void *mats, const int *active, const DenseGrid &G, int *ctr,
                           int *epoch, int *abort_word, long long *tick1, int blocks, double ptol, double stol,
                           hipStream_t st)
{
    hipLaunchKernelGGL(dense_lu_kernel<T>, dim3(std::min(blocks, G.nlu)), dim3(256), kDiagLds, st, jobs, mats, active,
                       G.lu, G.nlu, ctr, epoch, abort_word, tick1);
    hipLaunchKernelGGL(dense_pivot_kernel<T>, dim3(G.npivot), dim3(256), 0, st, jobs, mats, active, ptol, stol,
                       G.pivot);
    return hipGetLastError();
}
template hipError_t launch_dense_lu<float>(const DenseJob *, const void *, const int *, const DenseGrid &, int *, int *,
                                           int *, long long *, int, double, double, hipStream_t);
template hipError_t launch_dense_lu<double>(const DenseJob *, const void *, const int *, const DenseGrid &, int *, int *,
                                           int *, long long *, int, double, double, hipStream_t);
template hipError_t launch_dense_lu<__half>(const DenseJob *, const void *, const int *, const DenseGrid &, int *, int *,
                                           int *, long long *, int, double, double, hipStream_t);

// The lists behind the grids (see DenseGrid): jobs by falling T, so that the
// longest ones start first.
void dense_grid_lists(const std::vector<int> &T, const std::vector<int> &mat, DenseGridHost &H)
{
    const int nj = (int)T.size();
    H = DenseGridHost();
    // Tiles by the panels that remain from theirs on.  Of one panel: the
    // diagonal blocks, then the previous panel's other tiles (ready by now;
    // put right after their own diagonal block they would hold a workgroup
    // each while it is factored), then the two tiles the next diagonal block
    // waits for.
    const int most = nj ? (T[0] + kNb - 1) / kNb : 0;
    auto panels = [&](int left, auto put) {
        for (int j = 0; j < nj; j++) {
            const int nt = (T[j] + kNb - 1) / kNb;
            if (nt < left) break;                        // smaller blocks start later
            put(j, nt, nt - left);
        }
    };
    for (int left = most; left >= 0; left--) {
        panels(left, [&](int j, int nt, int q) { if (q < nt) H.lu.push_back(make_int4(j, q, q, 0)); });
        panels(left + 1, [&](int j, int nt, int q) {
            for (int i = q + 2; i < nt; i++) {
                H.lu.push_back(make_int4(j, i, q, 0));
                H.lu.push_back(make_int4(j, q, i, 0));
            }
        });
        panels(left, [&](int j, int nt, int q) {
            if (q + 1 < nt) {
                H.lu.push_back(make_int4(j, q + 1, q, 0));
                H.lu.push_back(make_int4(j, q, q + 1, 0));
            }
        });
    }
    for (int j = 0; j < nj; j++) {
        for (int c = 0; c * 256 < T[j]; c++) H.pivot.push_back(make_int2(j, c));
        for (int g = 0; g * 4 < T[j]; g++) H.gather.push_back(make_int2(mat[j], g));
        for (int t = 0; t * 2 * kNb < T[j]; t++) H.trsv.push_back(make_int2(mat[j], t));
    }
}

template <typename T>
hipError_t launch_tail_solve(const void *mats, const DenseGrid &G, const long *voff, const int *active,
                             const double *b, double *y, double *yp, double *z, double *x, bool forward,
                             int *abort_word, const double *rs, const double *cs, const int *n_active,
                             long long *tick0, hipStream_t st)
{
    if (forward) {
        hipLaunchKernelGGL(tail_fwd_gather_kernel<T>, dim3(G.ngather), dim3(256), 0, st, mats, G.gather, voff,
                           active, b, y, yp, rs, n_active);
        hipLaunchKernelGGL((tail_trsv_kernel<T, true>), dim3(G.ntrsv), dim3(512), 0, st, mats, G.trsv, voff,
                           active, y, yp, z, x, abort_word, cs, n_active, (long long *)nullptr);
    } else {
        hipLaunchKernelGGL((tail_trsv_kernel<T, false>), dim3(G.ntrsv), dim3(512), 0, st, mats, G.trsv, voff,
                           active, y, yp, z, x, abort_word, cs, n_active, tick0);
    }
    return hipGetLastError();
}
template hipError_t launch_tail_solve<float>(const void *, const DenseGrid &, const long *, const int *, const double *,
                                              double *, double *, double *, double *, bool, int *,
                                              const double *, const double *, const int *, long long *,
                                              hipStream_t);
template hipError_t launch_tail_solve<double>(const void *, const DenseGrid &, const long *, const int *, const double *,
                                              double *, double *, double *, double *, bool, int *,
                                              const double *, const double *, const int *, long long *,
                                              hipStream_t);
template hipError_t launch_tail_solve<__half>(const void *, const DenseGrid &, const long *, const int *, const double *,
                                              double *, double *, double *, double *, bool, int *,
                                              const double *, const double *, const int *, long long *,
                                              hipStream_t);

}  // namespace lsp

// localsolve.hip -- triangular solves of circuits whose vector fits one
// workgroup's LDS: one workgroup per circuit, a barrier per level (gfx950).
//
// Same solves as trisolve.hip, x = Q U^-1 L^-1 P b over the rows below the dense
// block.  There every level of dependencies costs a hand-off through memory
// (0.95 us: store, poll, sum, store; 2 to 4 us for the tasks of a large grid's
// critical chain) and every task a chain of loads (4 us on one of 1024 waves); a circuit of 1000 to 5000 unknowns has 40 to 90 levels
// and 150 to 800 tasks per solve.  Here the vector is in LDS, a level costs a
// barrier and an LDS gather (0.64 us), and what a task reads from memory (its
// header, its rows' records, their entries) is static, so it is loaded one task
// (entries) and two tasks (records) ahead of the barriers.  A level's tasks go
// to the waves in turn, so in a chain of one-task levels each wave has the time
// of 16 levels for its loads.  What bounds it: instruction issue of the one CU
// (0.16 us a task), so lone circuits with many tasks per level stay on the
// queue (lsp_choose_local).
//
// Measured, pair of solves with the dense block's, queue -> here: 512 circuits
// of 100 to 5000 unknowns 954 -> 463 us (fp32), 1032 -> 521 us (fp64); 17 circuits
// of a cohort 197 -> 157 us; n = 200 81 -> 56 us; 8 waves instead of 16: 553 us
// on the 512 circuits.
#include <algorithm>

#include "common.hpp"
#include "launch.hpp"

namespace lsp {

typedef int v4i __attribute__((ext_vector_type(4)));
constexpr int kPer = kTriPacketLane;    // entries of a row per lane and pass
constexpr int kLocalThreads = kWave * kLocalSolveWaves;
constexpr int kPart = 16;               // triangle columns in registers at a time

// This wave's LDS accesses done, then the workgroup's: nothing else is waited
// for, so the next tasks' loads stay in flight across it.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// A task with its lanes' records (see the plan), and a row task's entries.
// They are loaded the same way whatever the task's kind (addresses clamped, what
// does not apply masked), so that the compiler can count the loads in flight
// and wait for a task's own and not for the next one's.
struct TaskRec {
    int kind, g, cnt, first, lev, passes;
    v4i r;
};
template <typename T> struct Entries {
    T val[kPer];
    int idx[kPer];
    unsigned on;                        // bit h: entry h exists (kept apart: a mask on idx would wait for its load)
    T dia;
};

__device__ __forceinline__ TaskRec task_of(v4i h)
{
    TaskRec A;
    const int head = uniform(h.x);
    A.kind = head & 255;
    A.g = (head >> 8) & 255;
    A.cnt = head >> 16;
    A.first = uniform(h.y);
    A.lev = uniform(h.z);
    A.passes = uniform(h.w);
    A.r = (v4i){0, 0, 0, 0};
    return A;
}
__device__ __forceinline__ void load_records(const LSP_GLOBAL v4i *rec, TaskRec &A, int lane)
{
    const int grp = A.kind == 0 ? min(lane >> __builtin_ctz(A.g), A.cnt - 1) : lane;
    A.r = *near_el(rec, (uint32_t)(A.first + grp));
}

template <typename T, bool kForward>
__device__ __forceinline__ void load_pass(const LSP_GLOBAL T *rv, const LSP_GLOBAL int *ci, const TaskRec &A, int lane,
                                          int pass, Entries<T> &B)
{
    const int l = lane & (A.g - 1);
    const int e1 = A.kind == 0 && lane >> __builtin_ctz(A.g) < A.cnt ? A.r.z : 0;
    const int e0 = A.r.y + l + pass * kPer * A.g;
    B.on = 0;
#pragma unroll
    for (int h = 0; h < kPer; h++) {
        const int e = e0 + h * A.g;
        const uint32_t at = e < e1 ? (uint32_t)e : 0u;
        B.val[h] = ld_plain(near_el(rv, at), 0u);
        B.idx[h] = *near_el(ci, at);
        B.on |= e < e1 ? 1u << h : 0u;
    }
}

// The sum over the g lanes of each group (g a power of two), in all of them.
template <int kCtrl> __device__ __forceinline__ double dpp_f64(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, kCtrl, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), kCtrl, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double group_sum(double v, int g)
{
    v += dpp_f64<0xB1>(v);                      // quad_perm [1, 0, 3, 2]
    if (g > 2) v += dpp_f64<0x4E>(v);           // quad_perm [2, 3, 0, 1]
    if (g > 4) v += dpp_f64<0x141>(v);          // row_half_mirror: the other quad's sum
    if (g > 8) v += dpp_f64<0x140>(v);          // row_mirror: the other half row's
    if (g > 16) v += __shfl_xor(v, 16, kWave);
    if (g > 32) v += __shfl_xor(v, 32, kWave);
    return v;
}
// Lane Q's value of each group of g lanes (4, 8 or 16).
template <int Q> __device__ __forceinline__ double group_bcast(double v, int g, int lane)
{
    if (g == 4) return dpp_f64<(Q & 3) * 0x55>(v);                // quad_perm [Q, Q, Q, Q]
    const double a = dpp_f64<0x150 + (Q & 15)>(v);                // row_newbcast
    if (g == 16) return a;
    const double b = dpp_f64<0x150 + ((Q + 8) & 15)>(v);
    return lane & 8 ? b : a;
}
template <int Q> __device__ __forceinline__ int group_bcast(int v, int g, int lane)
{
    if (g == 4) return __builtin_amdgcn_update_dpp(0, v, (Q & 3) * 0x55, 0xf, 0xf, true);
    const int a = __builtin_amdgcn_update_dpp(0, v, 0x150 + (Q & 15), 0xf, 0xf, true);
    if (g == 16) return a;
    const int b = __builtin_amdgcn_update_dpp(0, v, 0x150 + ((Q + 8) & 15), 0xf, 0xf, true);
    return lane & 8 ? b : a;
}
// The packets' triangles, column by column: the loads, then the steps.  Column
// q is at this group's dp (s + q); `inside` collects the columns that touch
// this lane's row.
template <int Q, bool kForward, typename T>
__device__ __forceinline__ void tri_loads(const LSP_GLOBAL T *val, const v4i &r, T (&tv)[kPart], unsigned &inside, int g,
                                          int l, int lane)
{
    if (Q < g) {
        const int dq = group_bcast<Q>(r.y, g, lane);
        const int rq = kForward ? 0 : group_bcast<Q>(r.w, g, lane);
        const bool in = max(l, Q) < r.z && (kForward ? Q < l : l < Q && Q - l <= rq);
        tv[Q] = ld_plain(near_el(val, (uint32_t)(dq + (in ? l - Q : 0))), 0u);
        if (in) inside |= 1u << Q;
        if constexpr (Q + 1 < kPart) tri_loads<Q + 1, kForward>(val, r, tv, inside, g, l, lane);
    }
}
template <int Q, bool kForward, typename T>
__device__ __forceinline__ void tri_steps(const T (&tv)[kPart], double &p, double rd, unsigned inside, int g, int lane)
{
    constexpr int q = kForward ? Q : kPart - 1 - Q;
    if (q < (kForward ? g - 1 : g)) {
        const double yq = group_bcast<q>(kForward ? p : p * rd, g, lane);
        const double np = fma(-to_f64(tv[q]), yq, p);
        p = inside >> q & 1 ? np : p;
    }
    if constexpr (Q + 1 < kPart) tri_steps<Q + 1, kForward>(tv, p, rd, inside, g, lane);
}

template <typename T>
__device__ __forceinline__ double gather(const Entries<T> &B, const LSP_LDS double *v, double acc)
{
    double s[kPer];
#pragma unroll
    for (int h = 0; h < kPer; h++) s[h] = v[B.idx[h]];
#pragma unroll
    for (int h = 0; h < kPer; h++) {
        const double t = acc + to_f64(B.val[h]) * s[h];
        acc = B.on >> h & 1 ? t : acc;
    }
    return acc;
}

// Columns q0 .. q0 + kPart - 1 of a block's triangle: L(t, q) = val[dp_q + t - q]
// below the diagonal, U(t, q) = val[dp_q - (q - t)] within column q's run above.
template <typename T, bool kForward>
__device__ __forceinline__ void load_part(const LSP_GLOBAL T *val, int dpc, int ru, int bw, int q0, int lane,
                                          T (&tv)[kPart])
{
#pragma unroll
    for (int h = 0; h < kPart; h++) {
        const int q = min(q0 + h, bw - 1);
        const int base = __builtin_amdgcn_readlane(dpc, q);
        const int off = kForward ? min(max(lane - q, 0), bw - 1 - q)
                                 : -min(max(q - lane, 0), __builtin_amdgcn_readlane(ru, q));
        tv[h] = ld_plain(near_el(val, (uint32_t)(base + off)), 0u);
    }
}

template <typename T, bool kForward>
__global__ void __launch_bounds__(kLocalThreads, 4) local_solve_kernel(TriLaunch L, const int *list)
{
    extern __shared__ double lds_v[];
    LSP_LDS double *v = (LSP_LDS double *)lds_v;
    constexpr int D = kForward ? 0 : 1;
    if (L.n_active && uniform(ld_relaxed(L.n_active)) == 0) return;
    if (L.tick0 && blockIdx.x == 0 && threadIdx.x == 0) *L.tick0 = (long long)wall_clock64();
    const int mi = kp(list)[blockIdx.x];
    if (L.active && !kp(L.active)[mi]) return;
    const LSP_CONST TriDesc<T> *M = kp((const TriDesc<T> *)L.mats) + mi;
    const long vo = kp(L.voff)[mi];
    const int k0 = M->tail_k0;
    const int tid = threadIdx.x;

    const int lane_ = lane_id(), wv = uniform(tid >> 6);
    const LSP_CONST int *wp = kp(M->lwave[D]);
    const int t0 = wp[wv], t1 = wp[wv + 1], nlev = M->lnlev[D];
    const LSP_GLOBAL v4i *task = (const LSP_GLOBAL v4i *)M->ltask[D], *rec = (const LSP_GLOBAL v4i *)M->lrec[D];
    const LSP_GLOBAL T *rv = gp(kForward ? M->lrow : M->urow);
    const LSP_GLOBAL int *ci = gp(kForward ? M->lci : M->uci);
    const LSP_GLOBAL T *val = gp(M->val), *diag = gp(M->diag);
    const int tl = max(t1 - 1, 0);              // (a wave without tasks loads the circuit's first)
    // Rings of two, by the task's parity: a task's records are loaded when the
    // task two before it is done, its entries while the one before it waits.
    // (No copies between them: a copy would wait for the load.)
    TaskRec Ae = task_of(task[min(t0, tl)]), Ao = task_of(task[min(t0 + 1, tl)]);
    load_records(rec, Ae, lane_);
    load_records(rec, Ao, lane_);
    v4i He = task[min(t0 + 2, tl)], Ho = task[min(t0 + 3, tl)];

    // the vector: b (forward), or y with the block's z behind it (backward)
    if (kForward) {
        const LSP_GLOBAL int *rowat = gp(M->rowat);
        for (int i = tid; i < k0; i += kLocalThreads) {
            const int ro = rowat[i];
            v[i] = L.rs ? gp(L.b)[vo + ro] * gp(L.rs)[vo + ro] : gp(L.b)[vo + ro];
        }
    } else {
        for (int i = tid; i < M->n; i += kLocalThreads) v[i] = i < k0 ? gp(L.y)[vo + i] : gp(L.z)[vo + i];
    }
    Entries<T> Be, Bo;
    load_pass<T, kForward>(rv, ci, Ae, lane_, 0, Be);
    Be.dia = kForward ? T(0) : ld_plain(near_el(diag, (uint32_t)Ae.r.x), 0u);
    Bo = Be;
    lds_barrier();

    int lev = 0;
    T tv[kPart];                            // triangle columns (not set per task: a set waits for earlier loads)
#pragma unroll
    for (int q = 0; q < kPart; q++) tv[q] = T(0);
    auto run = [&](int t, TaskRec &A0, const Entries<T> &B0, const TaskRec &A1, Entries<T> &B1, v4i &H) {
        int lane = lane_;                       // opaque per task: nothing lane-dependent is kept through the loop
        asm volatile("" : "+v"(lane));
        // The barriers up to the task's level come between the parts of its
        // preparation, so that a wave that has just finished a task keeps the
        // others waiting for one part at most.
        auto step = [&]() {
            if (lev < A0.lev) {
                lds_barrier();
                lev++;
            }
        };
        step();
        const int g = A0.g, l = lane & (g - 1);
        double rd = 1.0;
        unsigned inside = 0;                    // kind 1: columns that touch this lane's row
        if (A0.kind == 1) {
            tri_loads<0, kForward>(val, A0.r, tv, inside, g, l, lane);
        } else if (A0.kind == 2) {
            const int bw = __builtin_amdgcn_readlane(A0.r.z, 0);
            load_part<T, kForward>(val, A0.r.y, A0.r.w, bw, kForward ? 0 : (bw - 1) / kPart * kPart, lane, tv);
        }
        step();
        load_pass<T, kForward>(rv, ci, A1, lane, 0, B1);       // the next task's entries
        B1.dia = kForward ? T(0) : ld_plain(near_el(diag, (uint32_t)A1.r.x), 0u);
        if (!kForward && A0.kind > 0) rd = 1.0 / to_f64(B0.dia);
        for (; lev < A0.lev; lev++) lds_barrier();
        if (A0.kind == 0) {
            double acc = gather(B0, v, 0.0);
            for (int p = 1; p < A0.passes; p++) {
                Entries<T> B;
                load_pass<T, kForward>(rv, ci, A0, lane, p, B);
                acc = gather(B, v, acc);
            }
            acc = group_sum(acc, g);
            if (l == 0 && lane >> __builtin_ctz(g) < A0.cnt) {
                const int i = A0.r.x;
                const double r = v[i] - acc;
                v[i] = kForward || A0.r.w ? r : r / to_f64(B0.dia);
            }
        } else if (A0.kind == 1) {
            const bool on = l < A0.r.z;
            double p = v[A0.r.x];
            tri_steps<0, kForward>(tv, p, rd, inside, g, lane);
            if (!kForward) p *= rd;
            if (on) v[A0.r.x] = p;
        } else {
            // one 64-row block: the blocks solved before it, then its triangle
            const int bw = __builtin_amdgcn_readlane(A0.r.z, 0), b = A0.passes & 4095;
            const int row = A0.r.x, base = __builtin_amdgcn_readlane(row, 0);
            const int c0 = kForward ? base - kWave * b : base + bw;             // first column of the solved blocks
            const LSP_CONST int *dp = kp(M->dp), *ru = kp(M->ru);
            double acc = 0.0;
            for (int q0 = 0; q0 < kWave * b; q0 += kPart) {
                T f[kPart];
                int top[kPart];
#pragma unroll
                for (int h = 0; h < kPart; h++) {
                    const int j = c0 + q0 + h;
                    top[h] = kForward ? 0 : j - ru[j];
                    f[h] = ld_plain(near_el(val, (uint32_t)(dp[j] + (kForward ? row - j : -min(j - row, ru[j])))), 0u);
                }
#pragma unroll
                for (int h = 0; h < kPart; h++)
                    if (row >= top[h]) acc = fma(to_f64(f[h]), v[c0 + q0 + h], acc);
            }
            double p = v[row] - acc;
            const int last = (bw - 1) / kPart * kPart;
            for (int x = 0; x <= last; x += kPart) {
                const int q0 = kForward ? x : last - x;
                if (x > 0) load_part<T, kForward>(val, A0.r.y, A0.r.w, bw, q0, lane, tv);
#pragma unroll
                for (int hh = 0; hh < kPart; hh++) {
                    const int h = kForward ? hh : kPart - 1 - hh, q = q0 + h;
                    if (q < bw) {
                        if (kForward) {
                            const double yq = bcast_f64(p, q);
                            const double np = fma(-to_f64(tv[h]), yq, p);
                            p = lane > q ? np : p;
                        } else {
                            const double zq = bcast_f64(p * rd, q);
                            const double np = fma(-to_f64(tv[h]), zq, p);
                            p = lane < q && q - lane <= __builtin_amdgcn_readlane(A0.r.w, q) ? np : p;
                        }
                    }
                }
            }
            if (!kForward) p *= rd;
            if (lane < bw) v[row] = p;
        }
        A0 = task_of(H);                        // the task after the next: its records, and the header after that
        load_records(rec, A0, lane);
        H = task[min(t + 4, tl)];
    };
    for (int t = t0; t < t1; t += 2) {
        run(t, Ae, Be, Ao, Bo, He);
        if (t + 1 < t1) run(t + 1, Ao, Bo, Ae, Be, Ho);
    }
    for (; lev < nlev; lev++) lds_barrier();
    lds_barrier();
    if (kForward) {
        for (int i = tid; i < k0; i += kLocalThreads) gp(L.y)[vo + i] = v[i];
    } else {
        const LSP_GLOBAL int *q = gp(M->q);
        for (int i = tid; i < k0; i += kLocalThreads) {
            const int qo = q[i];
            gp(L.x)[vo + qo] = L.cs ? v[i] * gp(L.cs)[vo + qo] : v[i];
        }
    }
    if (L.tick1 && tid == 0) atomicMax((unsigned long long *)L.tick1, (unsigned long long)wall_clock64());
}

template <typename T>
hipError_t launch_local_solve(const TriLaunch &L, bool forward, const int *list, int count, int rows, hipStream_t st)
{
    const size_t lds = (size_t)rows * sizeof(double);
    if (forward)
        hipLaunchKernelGGL((local_solve_kernel<T, true>), dim3(count), dim3(kLocalThreads), lds, st, L, list);
    else
        hipLaunchKernelGGL((local_solve_kernel<T, false>), dim3(count), dim3(kLocalThreads), lds, st, L, list);
    return hipGetLastError();
}
template hipError_t launch_local_solve<float>(const TriLaunch &, bool, const int *, int, int, hipStream_t);
template hipError_t launch_local_solve<double>(const TriLaunch &, bool, const int *, int, int, hipStream_t);
template hipError_t launch_local_solve<__half>(const TriLaunch &, bool, const int *, int, int, hipStream_t);

}  // namespace lsp

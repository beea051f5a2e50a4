// CPU emulation of the one-workgroup solves' schedule (run by
// tests/test_local_solve.py): every level's tasks are run wave by wave, in
// both wave orders; each value read must have become final at an earlier
// level, each triangle entry must be the one its slot holds, every row must
// be solved, and the result must match plain substitution.
// usage: local_solve <kind: 0 = c0, else n of a sized circuit> <tail max T (0 = none)> [plant: 1 = one task a level early]
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "host_internal.h"
#include "mna.h"
#include "csc.h"

static int fail(const char *what, long a = 0, long b = 0)
{
    std::printf("FAIL %s (%ld, %ld)\n", what, a, b);
    return 2;
}
static double entry(int i, int j) { return i == j ? 2.0 + 0.01 * (i % 7) : 0.3 * std::sin(1.0 + 3.0 * i + 7.0 * j); }

int main(int argc, char **argv)
{
    const int kind = argc > 1 ? std::atoi(argv[1]) : 0, tail_max = argc > 2 ? std::atoi(argv[2]) : 0;
    const int plant = argc > 3 ? std::atoi(argv[3]) : 0;
    LspMnaSpec sp;
    if (kind == 0) lsp_spec_c0(&sp, 0);
    else lsp_spec_sized(&sp, kind, 0.02, 3);
    LspCoo A;
    if (lsp_mna_build(&sp, A) != 0) return 1;
    const int n = A.n;
    std::vector<int> q(n), Ap, Ai, src;
    lsp_colamd_coo(n, (long)A.val.size(), A.row.data(), A.col.data(), q.data());
    lsp_coo_to_csc(n, (long)A.val.size(), A.row.data(), A.col.data(), q.data(), Ap, Ai, src);
    std::vector<double> Ax(A.val.size());
    for (size_t p = 0; p < Ax.size(); p++) Ax[p] = A.val[src[p]];
    LspGpLu F;
    if (lsp_gp_factor(n, Ap.data(), Ai.data(), Ax.data(), q.data(), 1.0, F) != -1) return 1;
    LspPlan P;
    if (lsp_build_plan(n, Ap.data(), Ai.data(), src.data(), F, q.data(), P) != 0) return 1;
    if (tail_max > 0 && lsp_plan_set_tail(P, 64, tail_max, 0.5) < 0) return 1;
    const int k0 = P.tail_k0;
    std::vector<int> col(P.cp[n]);
    for (int k = 0; k < n; k++)
        for (int64_t s = P.cp[k]; s < P.cp[k + 1]; s++) col[s] = k;

    for (int dir = 0; dir < 2; dir++) {
        const bool fwd = dir == 0;
        LspLocalSolve S;
        lsp_plan_local_solve(P, fwd, S);
        if ((int)S.wave.size() != kLocalWaves + 1 || S.wave[kLocalWaves] * 4 != (int)S.task.size()) return fail("waves");
        if (plant == 1)
            for (size_t t = 0; t < S.task.size(); t += 4)
                if (S.task[t + 2] == S.nlev / 2) { S.task[t + 2]--; break; }
        for (int order = 0; order < 2; order++) {
            std::vector<double> v(n), ref(n);
            std::vector<int> fin(n, fwd ? S.nlev + 1 : S.nlev + 1);      // level at which a row became final
            for (int i = 0; i < n; i++) v[i] = ref[i] = std::cos(0.7 * i);
            for (int i = k0; i < n; i++) fin[i] = -1;
            if (fwd) {
                for (int i = 0; i < k0; i++)
                    for (int e = P.lrp[i]; e < P.lrp[i + 1]; e++) ref[i] -= entry(i, P.lci[e]) * ref[P.lci[e]];
            } else {
                for (int i = k0 - 1; i >= 0; i--) {
                    for (int e = P.urp[i]; e < P.urp[i + 1]; e++) ref[i] -= entry(i, P.uci[e]) * ref[P.uci[e]];
                    ref[i] /= entry(i, i);
                }
            }
            std::vector<int> at(S.wave.begin(), S.wave.end() - 1);
            std::vector<char> partial(n, 0);
            for (int lev = 0; lev < S.nlev; lev++) {
                std::vector<std::pair<int, double>> out;                 // writes of this level
                std::vector<std::pair<int, int>> done;
                for (int ww = 0; ww < kLocalWaves; ww++) {
                    const int w = order ? kLocalWaves - 1 - ww : ww;
                    for (; at[w] < S.wave[w + 1] && S.task[4 * at[w] + 2] <= lev; at[w]++) {
                        const int *T = &S.task[4 * at[w]];
                        if (T[2] != lev) return fail("level order", at[w], lev);
                        const int kd = T[0] & 255, g = (T[0] >> 8) & 255, cnt = T[0] >> 16;
                        if (kd == 0) {
                            for (int r = 0; r < cnt; r++) {
                                const int *R = &S.rec[4 * (T[1] + r)];
                                const int i = R[0];
                                if (R[2] - R[1] > T[3] * g * kTriPacketPerLane) return fail("passes", i, T[3]);
                                double acc = 0.0;
                                for (int e = R[1]; e < R[2]; e++) {
                                    const int j = fwd ? P.lci[e] : P.uci[e];
                                    if (fin[j] >= lev) return fail("read", i, j);
                                    acc += entry(i, j) * v[j];
                                }
                                const double x = v[i] - acc;
                                out.push_back({i, fwd || R[3] ? x : x / entry(i, i)});
                                if (R[3]) partial[i] = 1;
                                else done.push_back({i, lev});
                            }
                            continue;
                        }
                        struct Blk { int s, b, w; };
                        std::vector<Blk> blk;
                        if (kd == 1) {
                            for (int r = 0; r < cnt; r++) {
                                const int *R = &S.rec[4 * (T[1] + r * g)];
                                if (R[2] > g) return fail("triangle width", R[0], R[2]);
                                for (int l = 0; l < g; l++) {
                                    const int *Q = R + 4 * l;
                                    const int row = R[0] + std::min(l, R[2] - 1);
                                    if (Q[0] != row || Q[1] != P.dp[row] || Q[3] != P.ru[row] || Q[2] != (l < R[2] ? R[2] : 0))
                                        return fail("triangle record", row, l);
                                }
                                blk.push_back({R[0], 0, R[2]});
                            }
                        } else {
                            const int b = T[3] & 4095, bwid = T[3] >> 12, bw = std::min(64, bwid - 64 * b);
                            const int row0 = S.rec[4 * T[1]];
                            for (int l = 0; l < 64; l++) {
                                const int *Q = &S.rec[4 * (T[1] + l)], row = row0 + std::min(l, bw - 1);
                                if (Q[0] != row || Q[1] != P.dp[row] || Q[2] != bw || Q[3] != P.ru[row])
                                    return fail("block record", row, l);
                            }
                            blk.push_back({fwd ? row0 - 64 * b : row0 - (bwid - 64 * b - bw), b, bwid});
                        }
                        for (const Blk &B : blk) {
                            const int bw = std::min(64, B.w - 64 * B.b);
                            const int r0 = fwd ? B.s + 64 * B.b : B.s + B.w - 64 * B.b - bw;
                            std::vector<double> p(bw);
                            for (int t = 0; t < bw; t++) p[t] = v[r0 + t];
                            for (int t = 0; t < bw; t++)
                                if (P.fcut[r0 + t] > P.lrp[r0 + t] && fwd && !partial[r0 + t]) return fail("partial", r0 + t);
                            for (int jj = 0; jj < 64 * B.b; jj++) {       // blocks solved before
                                const int j = fwd ? B.s + jj : r0 + bw + jj;
                                if (fin[j] >= lev) return fail("block read", r0, j);
                                for (int t = 0; t < bw; t++) {
                                    const int row = r0 + t;
                                    if (!fwd && j - row > P.ru[j]) continue;
                                    const int64_t slot = fwd ? P.dp[j] + row - j : P.dp[j] - (j - row);
                                    if (P.pos[slot] != row || col[slot] != j) return fail("block slot", row, j);
                                    p[t] -= entry(row, j) * v[j];
                                }
                            }
                            for (int x = 0; x < bw; x++) {
                                const int c = fwd ? x : bw - 1 - x, j = r0 + c;
                                if (!fwd) p[c] /= entry(j, j);
                                for (int t = fwd ? c + 1 : 0; t < (fwd ? bw : c); t++) {
                                    const int row = r0 + t;
                                    if (!fwd && j - row > P.ru[j]) continue;
                                    const int64_t slot = fwd ? P.dp[j] + row - j : P.dp[j] - (j - row);
                                    if (P.pos[slot] != row || col[slot] != j) return fail("slot", row, j);
                                    p[t] -= entry(row, j) * p[c];
                                }
                            }
                            for (int t = 0; t < bw; t++) { out.push_back({r0 + t, p[t]}); done.push_back({r0 + t, lev}); }
                        }
                    }
                }
                for (auto &o : out) v[o.first] = o.second;
                for (auto &d : done) {
                    if (fin[d.first] <= S.nlev) return fail("solved twice", d.first);
                    fin[d.first] = d.second;
                }
            }
            double diff = 0.0, mx = 0.0;
            for (int i = 0; i < k0; i++) {
                if (fin[i] > S.nlev) return fail("not solved", i);
                diff = std::max(diff, std::fabs(v[i] - ref[i]));
                mx = std::max(mx, std::fabs(ref[i]));
            }
            if (!(diff <= 1e-9 * mx)) return fail("values", fwd, (long)(diff / mx * 1e15));
        }
    }
    std::printf("ok %d %d\n", n, P.tail_T);
    return 0;
}

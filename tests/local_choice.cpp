// Prints which circuits of a batch are solved by one workgroup each (run by
// tests/test_local_choice.py).
// usage: local_choice <tail_max (0 = default, < 0 = none)> <n seed count>...   (sized circuits, lr 0.02)
#include <cstdio>
#include <cstdlib>
#include <map>
#include <utility>
#include <vector>

#include "csc.h"
#include "host_internal.h"
#include "mna.h"

static int load_of(int n_req, int seed, int tail_max, LspSolveLoad &out)
{
    LspMnaSpec sp;
    lsp_spec_sized(&sp, n_req, 0.02, seed);
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
    if (lsp_build_plan(n, Ap.data(), Ai.data(), src.data(), F, q.data(), P, tail_max < 0) != 0) return 1;
    if (tail_max >= 0 && lsp_plan_set_tail(P, 64, tail_max ? tail_max : 8192, 0.5) < 0) return 1;
    LspLocalSolve S[2];
    if (lsp_local_solve_fits(P))
        for (int d = 0; d < 2; d++) lsp_plan_local_solve(P, d == 0, S[d]);
    out = lsp_solve_load(P, S);
    return 0;
}

int main(int argc, char **argv)
{
    const int tail_max = std::atoi(argv[1]);
    std::map<std::pair<int, int>, LspSolveLoad> known;
    std::vector<LspSolveLoad> batch;
    for (int a = 2; a + 2 < argc; a += 3) {
        const std::pair<int, int> key{std::atoi(argv[a]), std::atoi(argv[a + 1])};
        if (!known.count(key) && load_of(key.first, key.second, tail_max, known[key])) return 1;
        for (int c = 0; c < std::atoi(argv[a + 2]); c++) batch.push_back(known[key]);
    }
    for (char on : lsp_choose_local(batch)) std::putchar(on ? '1' : '0');
    std::putchar('\n');
    return 0;
}

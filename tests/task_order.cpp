// Checks the refactor's task order of one generated circuit (run by
// tests/test_task_order.py): the list holds every column once, its keys never
// fall, and every dependency has a smaller key than the column waiting for it
// (so it also comes first when circuits are merged by key).
// usage: task_order <kind: 0 = c0, 1 = c1, else n of a sized circuit> <tail max T (0 = none)>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "host_internal.h"
#include "mna.h"
#include "csc.h"

int main(int argc, char **argv)
{
    const int kind = argc > 1 ? std::atoi(argv[1]) : 0, tail_max = argc > 2 ? std::atoi(argv[2]) : 0;
    LspMnaSpec sp;
    if (kind == 0) lsp_spec_c0(&sp, 0);
    else if (kind == 1) lsp_spec_c1(&sp, 1);
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
    lsp_plan_set_tail(P, tail_max > 0 ? 64 : 1, tail_max, 0.5);
    std::vector<char> seen(n, 0);
    if ((int)P.ftask.size() != n || (int)P.fkey.size() != n) { std::puts("FAIL sizes"); return 2; }
    for (int t = 0; t < n; t++) {
        const int k = P.ftask[t];
        if (k < 0 || k >= n || seen[k]) { std::puts("FAIL columns"); return 2; }
        if (t && P.fkey[P.ftask[t - 1]] > P.fkey[k]) { std::puts("FAIL falling key"); return 2; }
        const int64_t e = k < P.tail_k0 ? P.dp[k] : P.cp[k] + P.tail_ds[k - P.tail_k0];
        for (int64_t s = P.cp[k]; s < e; s++)
            if (!seen[P.pos[s]] || P.fkey[P.pos[s]] >= P.fkey[k]) { std::puts("FAIL dependency"); return 2; }
        seen[k] = 1;
    }
    std::printf("ok %d %d\n", n, P.tail_T);
    return 0;
}

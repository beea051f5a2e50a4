"""The device memory estimate that admission relies on is an upper one: with
both factor sets a batch holds no more.  Byte counts are whole numbers."""
import pytest

import luspice_amd as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,opts", [
    ([64] * 200, {}), ([64] * 200, {"ir_inner": 120}), ([200], {}), ([1020], {}), ([3000], {"chunk_rows": 1}),
    ([3000], {"tail_max": -1}), ([3000], {"ir_inner": 3}), ([300, 8192, 5000] + [700] * 20, {}),
    ([1020] * 8, {"krylov_spmv": 1, "factor_shift": 1e-3}), ([12000], {"lds_cap": -256}),
])
def test_estimate_is_an_upper_one(sizes, opts):
    print("case: memory", len(sizes), "circuits of", sizes[:3], opts, flush=True)
    known = {}
    for n in sizes:
        if n not in known:
            known[n] = L.mna("sized", n=n, lr=0.02, seed=5)
            known[n].q = L.colamd(known[n])
    B = L.Batch([known[n] for n in sizes], **opts)
    estimate = B.estimate_bytes()
    for prec in ("fp32", "fp64"):
        assert B.refactor(prec)["rc"] == 0
    held = B.device_bytes()
    assert held <= estimate <= 4 * held + (2 << 20), (held, estimate)
    B.close()

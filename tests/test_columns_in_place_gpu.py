"""GeKMM chains of small square factors in groups whose digits stay in place (kernels/small_inplace.hip, columns) against
the oracle: few columns and many, tiles that cross batch entries, a last tile that is not full, one, two and three passes,
chains of several groups and with other factors between them.  TOL of gpu_util: the sums have at most 8 terms per factor
and ten factors, so u * 80 = 4.8e-6 / 8.9e-15 bounds the error."""
import numpy as np
import pytest

from oracle import kron_oracle as ko
from tests.gpu_util import TOL, make_case, normwise, oracle_answer, run_gpu

pytestmark = pytest.mark.gpu

CASES = [
    # columns, factors, groups expected
    (2, [7] * 3, 1), (33, [7] * 3, 1), (64, [7] * 2, 1), (65, [8] * 3, None), (130, [8] * 3, 1), (3, [8] * 5, 2), (31, [6] * 3, 1), (500, [5] * 4, 1),
    (17, [5] * 4, 1), (9, [3] * 5, 1), (70, [3] * 3, 1), (5, [4] * 4, None), (13, [4] * 3, None), (6, [2] * 6, None), (11, [2] * 5, None),
    (10, [7] * 6, 2), (88, [7] * 4, 2), (4, [5] * 7, 2), (150, [6] * 5, 2), (7, [3] * 8, 2), (23, [8] * 4, 2), (3, [7, 7, 24], 2),
    (12, [24, 5, 5, 5], 2), (5, [6, 6, 16, 3, 3, 3], 3), (2200, [7] * 3, 1), (4100, [5] * 4, 1), (2, [3] * 10, 2), (40, [7] * 7, 3),
]


@pytest.fixture(scope="module")
def fk():
    import os
    import fastkron_amd
    old = os.environ.get("FASTKRON_SHIPPED_PLANS")
    os.environ["FASTKRON_SHIPPED_PLANS"] = "0"
    h = fastkron_amd.FastKron()
    if old is None:
        del os.environ["FASTKRON_SHIPPED_PLANS"]
    else:
        os.environ["FASTKRON_SHIPPED_PLANS"] = old
    yield h
    h.close()


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
@pytest.mark.parametrize("M,Ps,groups", CASES, ids=lambda v: str(v) if not isinstance(v, list) else "x".join(map(str, v)))
def test_columns_in_place(fk, M, Ps, groups, dt):
    for seed, kw in enumerate([dict(alpha=1.5, beta=0.5), dict(alpha=1.0, beta=0.0, opFs=ko.OP_T), dict(alpha=-2.0, beta=1.0, batch=3, share_f=True),
                               dict(alpha=1.5, beta=0.5, batch=2), dict(alpha=0.5, beta=2.0, y_is_z=True), dict(alpha=1.0, beta=0.0, opX=ko.OP_T)]):
        alpha, beta, y_is_z = kw.pop("alpha"), kw.pop("beta"), kw.pop("y_is_z", False)
        batch, share = kw.get("batch", 1), dict(share_f=True) if kw.get("share_f") else {}
        X, Fs, Y = make_case(ko.KMM, M, Ps, Ps, dt, seed=3 + 50 * seed, with_y=beta != 0.0, batch=batch, **share)
        want = oracle_answer(ko.KMM, M, Ps, Ps, X, Fs, Y, alpha, beta, **kw)
        got, e = run_gpu(fk, ko.KMM, M, Ps, Ps, X, Fs, Y, alpha, beta, y_is_z=y_is_z, **kw)
        assert e == 0 and normwise(got, want) <= TOL[dt], (fk.last_plan(), kw)
        if groups and batch == 1 and "opX" not in kw:
            assert len(fk.last_plan()) == groups and any("columns" in s[2] for s in fk.last_plan()), fk.last_plan()


@pytest.mark.parametrize("tune", [False, True])
def test_records_of_groups_in_place(tmp_path, tune):
    """A record says that the digits stay in place (M2), in other groups than the rule's: that is what runs.  A handle that tunes
    stores what it runs, and one that does not runs it from the file."""
    import fastkron_amd
    db = tmp_path / "plans.txt"
    M, Ps, k = 5, [7] * 5, "kmm_hip_gfx950_512_d_small_fused_columns_8"
    X, Fs, Y = make_case(ko.KMM, M, Ps, Ps, np.float64, seed=5)
    want = oracle_answer(ko.KMM, M, Ps, Ps, X, Fs, Y, 1.5, 0.5)
    if not tune:
        db.write_text(f"(7x7^5)*16807x5_NN_d 0.01 M2 S0 2 3 4 {k} 0 2 {k}\n")
    plans = []
    for t in ([True, False] if tune else [False]):
        h = fastkron_amd.FastKron(tune=t)
        h.set_tuned_db(str(db))
        got, e = run_gpu(h, ko.KMM, M, Ps, Ps, X, Fs, Y, 1.5, 0.5)
        assert e == 0 and normwise(got, want) <= TOL[np.float64], h.last_plan()
        plans.append(h.last_plan())
        h.close()
    if tune:
        assert plans[0] == plans[1] and (" M2 " in db.read_text()) == any("columns" in s[2] for s in plans[0])
    else:
        assert plans == [[(3, 4, k), (0, 2, k)]]

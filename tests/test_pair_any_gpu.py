"""Two factors of any sizes up to 64 in one launch (kernels/pair_any_mfma.hip) against the oracle: one row and more than the
device holds at once, every alignment of a tile, sizes at the edges of the 16-wide blocks and of the four-wide steps, several
rows per workgroup, sizes that differ between the factors.  TOL of gpu_util: normwise 1e-5 / 1e-12; two sums of at most 64
terms, so u * 2 * 64 = 7.6e-6 / 1.4e-14 bounds the error."""
import numpy as np
import pytest

from oracle import kron_oracle as ko
from tests.gpu_util import TOL, make_case, normwise, oracle_answer, run_gpu

pytestmark = pytest.mark.gpu

CASES = [
    # rows, (P, Q) of the two factors
    (1, (31, 63), (31, 63)), (7, (63, 31), (63, 31)), (600, (31, 63), (31, 63)), (2500, (33, 17), (9, 12)), (5, (64, 64), (63, 64)),
    (3, (50, 50), (50, 50)), (1100, (50, 40), (12, 20)), (1030, (9, 9), (9, 9)), (9001, (10, 3), (3, 10)), (13, (17, 1), (1, 17)),
    (6, (2, 33), (5, 48)), (4, (16, 16), (16, 8)), (5000, (12, 16), (12, 16)), (2, (47, 49), (64, 33)), (2060, (24, 24), (24, 24)),
    (2055, (31, 31), (31, 31)), (11, (4, 60), (60, 4)), (3, (1, 64), (64, 1)), (2049, (20, 20), (20, 20)), (700, (32, 16), (32, 16)),
    (515, (48, 64), (48, 64)), (129, (8, 32), (8, 32)),
]


@pytest.fixture(scope="module")
def fk():
    import fastkron_amd
    h = fastkron_amd.FastKron()
    yield h
    h.close()


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
@pytest.mark.parametrize("M,a,b", CASES, ids=lambda v: str(v) if isinstance(v, int) else "%dx%d" % v)
def test_two_factors_of_any_size(fk, M, a, b, dt):
    Ps, Qs = [a[0], b[0]], [a[1], b[1]]
    for seed, kw in enumerate([dict(alpha=1.5, beta=0.5), dict(alpha=1.0, beta=0.0, opFs=ko.OP_T), dict(alpha=2.0, beta=1.0, batch=3),
                               dict(alpha=1.0, beta=0.0, batch=2, share_f=True)]):
        alpha, beta = kw.pop("alpha"), kw.pop("beta")
        if M > 600 and kw.get("batch", 1) > 1:
            continue
        batch, share = kw.get("batch", 1), dict(share_f=True) if kw.get("share_f") else {}
        X, Fs, Y = make_case(ko.MKM, M, Ps, Qs, dt, seed=9 + 50 * seed, with_y=beta != 0.0, batch=batch, **share)
        want = oracle_answer(ko.MKM, M, Ps, Qs, X, Fs, Y, alpha, beta, **kw)
        got, e = run_gpu(fk, ko.MKM, M, Ps, Qs, X, Fs, Y, alpha, beta, **kw)
        assert e == 0 and normwise(got, want) <= TOL[dt], (fk.last_plan(), kw)
        assert len(fk.last_plan()) == 1, fk.last_plan()


@pytest.mark.parametrize("M,Ps,Qs", [(1, [31] * 3, [63] * 3), (3, [50] * 3, [50] * 3), (2, [6, 6, 50, 50], [6, 6, 50, 50]), (9, [12, 20, 30], [12, 20, 30])],
                         ids=lambda v: str(v) if isinstance(v, int) else "x".join(map(str, v)))
@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
def test_trailing_factors_of_longer_chains(fk, M, Ps, Qs, dt):
    for seed, kw in enumerate([dict(alpha=1.5, beta=0.5), dict(alpha=1.0, beta=0.0, opFs=ko.OP_T, batch=2, share_f=True)]):
        alpha, beta = kw.pop("alpha"), kw.pop("beta")
        batch, share = kw.get("batch", 1), dict(share_f=True) if kw.get("share_f") else {}
        X, Fs, Y = make_case(ko.MKM, M, Ps, Qs, dt, seed=5 + 50 * seed, with_y=beta != 0.0, batch=batch, **share)
        want = oracle_answer(ko.MKM, M, Ps, Qs, X, Fs, Y, alpha, beta, **kw)
        got, e = run_gpu(fk, ko.MKM, M, Ps, Qs, X, Fs, Y, alpha, beta, **kw)
        assert e == 0 and normwise(got, want) <= TOL[dt], (fk.last_plan(), kw)
        assert fk.last_plan()[0][0] == len(Ps) - 2 and "_anyxany_64x64_2_" in fk.last_plan()[0][2], fk.last_plan()


def test_infinities_stay_in_their_rows_and_operands_off_a_16_byte_boundary(fk):
    """A row of infinities between others: the elements beyond P that a lane reads belong to its neighbours."""
    import torch
    M, P, Q = 41, 31, 18
    K, L = P * P, Q * Q
    X, Fs, Y = make_case(ko.MKM, M, [P] * 2, [Q] * 2, np.float32, seed=3)
    want = oracle_answer(ko.MKM, M, [P] * 2, [Q] * 2, X, Fs, Y, 1.5, 0.5).reshape(M, L)
    fs = [torch.from_numpy(f).cuda() for f in Fs]
    for off in (0, 1, 2, 3):
        x = torch.full((M * K + 8,), float("inf"), device="cuda")
        z = torch.full((M * L + 8,), 77.0, device="cuda")
        x[off:off + M * K] = torch.from_numpy(X).cuda().reshape(-1)
        x[off + 20 * K:off + 21 * K] = float("inf")
        z[off:off + M * L] = torch.from_numpy(Y).cuda().reshape(-1)
        t1, t2 = torch.empty(M * max(K, L, P * Q), device="cuda"), torch.empty(M * max(K, L, P * Q), device="cuda")
        zv = z[off:off + M * L]
        assert fk.xgemkm(M, [P] * 2, [Q] * 2, x[off:off + M * K], fs, zv, 1.5, 0.5, zv, t1, t2) == 0
        torch.cuda.synchronize()
        assert "_anyxany_64x64_2_" in fk.last_plan()[0][2], fk.last_plan()
        got = zv.cpu().numpy().reshape(M, L)
        rows = [i for i in range(M) if i != 20]
        assert normwise(got[rows], want[rows]) <= TOL[np.float32]
        assert bool((z[:off] == 77.0).all()) and bool((z[off + M * L:] == 77.0).all())


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
@pytest.mark.parametrize("M,a,b", [(3, (31, 63), (31, 63)), (7, (50, 50), (50, 50)), (2100, (24, 48), (24, 48)), (2, (12, 20), (12, 20)), (5, (33, 17), (9, 12)),
                                   (2, (63, 31), (47, 49)), (40, (2, 33), (5, 48)), (2, (17, 64), (64, 17))],
                         ids=lambda v: str(v) if isinstance(v, int) else "%dx%d" % v)
def test_infinities_of_the_factors_reach_their_columns_only(fk, M, a, b, dt):
    """One infinity in either factor, everything else positive: infinite results in its columns, no NaN, the others as they were."""
    import torch
    Ps, Qs = [a[0], b[0]], [a[1], b[1]]
    X, Fs, _ = make_case(ko.MKM, M, Ps, Qs, dt, seed=7, with_y=False, integer=True)
    want = oracle_answer(ko.MKM, M, Ps, Qs, X, Fs, None, 1.0, 0.0).reshape(M, Qs[0], Qs[1])
    for which, (p, q) in [(0, (0, 1)), (0, (a[0] - 1, a[1] - 1)), (1, (0, 0)), (1, (b[0] - 1, b[1] - 1))]:
        fs = [f.copy() for f in Fs]
        fs[which].reshape(Ps[which], Qs[which])[p, q] = np.inf
        got, e = run_gpu(fk, ko.MKM, M, Ps, Qs, X, fs, None, 1.0, 0.0)
        got = got.reshape(M, Qs[0], Qs[1])
        hit = np.zeros((Qs[0], Qs[1]), bool)
        (hit if which == 0 else hit.T)[q] = True
        assert e == 0 and "_anyxany_64x64_2_" in fk.last_plan()[0][2], fk.last_plan()
        assert np.all(np.isposinf(got[:, hit])) and normwise(got[:, ~hit], want[:, ~hit]) <= TOL[dt], (which, p, q)

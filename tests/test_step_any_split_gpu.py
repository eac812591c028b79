"""One factor of any shape per launch (kernels/step_any_mfma.hip): lines of a few elements side by side, slabs of output columns
by the number of tiles, and sizes at the edges of the 16 contraction indices that a wave reads at once, against the oracle.  TOL
of gpu_util: normwise 1e-5 / 1e-12.  The rounding errors of a sum of P <= 256 terms add up like a random walk of P / 4 fused
steps, and there are at most three sums one behind the other: 3 * 8 * u = 1.4e-6 / 2.7e-15."""
import numpy as np
import pytest

from oracle import kron_oracle as ko
from tests.gpu_util import TOL, make_case, normwise, oracle_answer, run_gpu

pytestmark = pytest.mark.gpu

CASES = [
    # lines of fewer than 16 elements, or a little more, enough of them to be put side by side
    (ko.KMM, 2, [50, 50, 24], [50, 50, 40]), (ko.KMM, 3, [40, 40, 40], [40, 33, 40]), (ko.KMM, 15, [33, 33, 33], [33, 33, 33]),
    (ko.KMM, 33, [31, 31, 31], [31, 31, 31]), (ko.KMM, 5, [66, 7, 66], [64, 9, 50]), (ko.KMM, 12, [130, 100], [140, 100]),
    (ko.MKM, 1100, [100], [100]), (ko.MKM, 1300, [3, 66], [3, 65]), (ko.MKM, 500, [17, 70], [20, 70]), (ko.MKM, 1025, [2, 129], [1, 100]),
    # few tiles: every 16 columns of the factor a workgroup of their own
    (ko.MKM, 1, [100, 100], [100, 100]), (ko.MKM, 3, [96, 128], [200, 100]), (ko.KMM, 17, [96, 96], [96, 96]), (ko.KMM, 2, [256, 65], [17, 512]),
    (ko.KMM, 1, [255, 66], [66, 255]), (ko.MKM, 9, [67, 68], [69, 70]), (ko.MKM, 20, [80, 113], [113, 80]), (ko.KMM, 16, [112, 128], [128, 112]),
    # factors for whose registers a CU has room once (fp64 KMM above 128: multiples of 16, the plain kernel has the others)
    (ko.MKM, 100, [200, 200], [200, 200]), (ko.MKM, 130, [90, 90], [90, 91]), (ko.KMM, 130, [208, 144], [200, 160]), (ko.MKM, 300, [150], [256]),
    (ko.KMM, 200, [128, 128], [128, 128]), (ko.MKM, 200, [65, 80], [129, 80]),
]


@pytest.fixture(scope="module")
def fk():
    import fastkron_amd
    h = fastkron_amd.FastKron()
    yield h
    h.close()


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
@pytest.mark.parametrize("mm,M,Ps,Qs", CASES, ids=lambda v: str(v) if isinstance(v, int) else "x".join(map(str, v)))
def test_steps_of_any_size(fk, mm, M, Ps, Qs, dt):
    seen = ""
    for seed, kw in enumerate([dict(alpha=1.5, beta=0.5), dict(alpha=1.0, beta=0.0, opX=ko.OP_T), dict(alpha=1.0, beta=0.0, opFs=ko.OP_T),
                               dict(alpha=2.0, beta=1.0, batch=3)]):
        alpha, beta = kw.pop("alpha"), kw.pop("beta")
        if M * np.prod([max(p, q) for p, q in zip(Ps, Qs)]) > 1e6 and kw.get("batch", 1) > 1:
            continue
        X, Fs, Y = make_case(mm, M, Ps, Qs, dt, seed=3 + 50 * seed, with_y=beta != 0.0, batch=kw.get("batch", 1))
        want = oracle_answer(mm, M, Ps, Qs, X, Fs, Y, alpha, beta, **kw)
        got, e = run_gpu(fk, mm, M, Ps, Qs, X, Fs, Y, alpha, beta, **kw)
        assert e == 0 and normwise(got, want) <= TOL[dt], (fk.last_plan(), kw)
        seen += str(fk.last_plan())
    assert "_anyxany_256x512_" in seen, seen


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
def test_padding_leaves_infinities_where_they_belong(fk, dt):
    """Indices beyond P must not bring a neighbour's infinity in: row 1 of X is infinite, the others' results are finite."""
    import torch
    for P in (50, 66, 100, 131):
        x = torch.ones((3, P * 3), device="cuda", dtype=torch.float32 if dt == np.float32 else torch.float64)
        x[1] = float("inf")
        fs = [torch.ones((3, 3), device="cuda", dtype=x.dtype), torch.ones((P, P), device="cuda", dtype=x.dtype)]
        import fastkron_amd
        z = fastkron_amd.gemkm(x, fs)
        assert torch.all(z[0] == 3 * P) and torch.all(z[2] == 3 * P) and torch.all(torch.isinf(z[1])), P

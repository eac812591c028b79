"""Rows of small square factors applied in place in LDS (kernels/small_inplace.hip) against the oracle, at the edges of
its tiles: one row and several per workgroup, a last workgroup that is not full, rows that start off a 16-byte
boundary, single digits and groups of them, stores from registers and from LDS.  TOL of gpu_util: normwise 1e-5 / 1e-12;
the sums have at most 8 terms per factor and nine factors, so u * 72 = 4.3e-6 / 8e-15 bounds the error."""
import numpy as np
import pytest

from oracle import kron_oracle as ko
from tests.gpu_util import TOL, make_case, normwise, oracle_answer, run_gpu

pytestmark = pytest.mark.gpu

CASES = [
    # rows, factors
    (1, [5] * 6),            # one row
    (7, [5] * 6),            # odd row length: every alignment of a row
    (2, [5] * 5), (3, [3] * 8), (3, [7] * 5), (2, [6] * 5), (5, [6, 6, 6]),
    (1100, [3, 3]),          # several rows per workgroup, last one not full
    (2051, [5, 5, 5]), (1031, [7, 7]), (1029, [2, 2, 2, 2, 2]), (4111, [6, 2]), (1057, [4, 4, 4]),
    (13, [8, 8, 8]), (9, [8] * 4), (4, [2, 3, 5, 7, 8]), (3, [8, 7, 5, 3, 2]), (2, [4, 4, 8, 3, 3, 3, 3]),
    (2, [2, 3, 4, 5, 6, 7, 8]),      # few long rows in passes of one digit: not in place
    (96, [2, 3, 4, 5, 6, 7, 8]), (96, [3, 4, 5, 6, 7, 8]),      # 161280 bytes, a whole CU's LDS, in fp32 and in fp64
    (96, [7] * 5), (33, [4, 4, 8, 3, 3, 3, 3]),
]


def runs_in_place(M, Ps, dt, batch, own_factors):
    """Which calls the kernel is meant for: rows that fit, not few long ones in passes of one digit, and no neighbours that
    are merged into a larger factor instead (which factors of one batch entry only are not)."""
    bytes_ = int(np.prod(Ps)) * np.dtype(dt).itemsize
    one_digit = len(set(Ps)) > 1 or (dt is np.float64 and Ps[-1] >= 6)
    merged = (2, 4) if dt is np.float32 else (2, 4, 8)
    return (bytes_ + 16 <= 160 * 1024 and not (one_digit and bytes_ > 65536 and M * batch < 96) and
            (own_factors or not any(a in merged and b in merged for a, b in zip(Ps, Ps[1:]))))


@pytest.fixture(scope="module")
def fk():
    import fastkron_amd
    h = fastkron_amd.FastKron()
    yield h
    h.close()


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
@pytest.mark.parametrize("M,Ps", CASES, ids=lambda v: str(v) if isinstance(v, int) else "x".join(map(str, v)))
def test_small_factors_in_place(fk, M, Ps, dt):
    for seed, kw in enumerate([dict(alpha=1.5, beta=0.5), dict(alpha=1.0, beta=0.0, opFs=ko.OP_T),
                               dict(alpha=1.0, beta=0.0, batch=3), dict(alpha=-2.0, beta=1.0, batch=2, share_f=True),
                               dict(alpha=1.5, beta=0.5, batch=3)]):
        alpha, beta = kw.pop("alpha"), kw.pop("beta")
        batch, share = kw.get("batch", 1), dict(share_f=True) if kw.get("share_f") else {}
        X, Fs, Y = make_case(ko.MKM, M, Ps, Ps, dt, seed=7 + 50 * seed, with_y=beta != 0.0, batch=batch, **share)
        want = oracle_answer(ko.MKM, M, Ps, Ps, X, Fs, Y, alpha, beta, **kw)
        got, e = run_gpu(fk, ko.MKM, M, Ps, Ps, X, Fs, Y, alpha, beta, **kw)
        assert e == 0 and normwise(got, want) <= TOL[dt], (fk.last_plan(), kw)
        in_place = len(fk.last_plan()) == 1 and "inplace" in fk.last_plan()[0][2]
        assert in_place == runs_in_place(M, Ps, dt, batch, batch > 1 and not share), (fk.last_plan(), kw)


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
@pytest.mark.parametrize("M,Ps", [(3, [5] * 7), (1, [3] * 9), (2, [6] * 6), (2, [7] * 6), (5, [4, 2] + [5] * 6), (100, [2] + [7] * 5)],
                         ids=lambda v: str(v) if isinstance(v, int) else "x".join(map(str, v)))
def test_rows_beyond_the_lds_run_their_trailing_factors_in_place(fk, M, Ps, dt):
    """A two-part plan: blocks of 3^8, 5^6, 6^5 or 7^5 columns in place, the leading factors across the blocks."""
    few_long_rows = dt is np.float64 and Ps[-1] >= 6 and M < 20       # (few blocks in passes of one digit)
    for seed, kw in enumerate([dict(alpha=1.5, beta=0.5), dict(alpha=1.0, beta=0.0, opFs=ko.OP_T, batch=2, share_f=True)]):
        alpha, beta = kw.pop("alpha"), kw.pop("beta")
        batch, share = kw.get("batch", 1), dict(share_f=True) if kw.get("share_f") else {}
        X, Fs, Y = make_case(ko.MKM, M, Ps, Ps, dt, seed=5 + 50 * seed, with_y=beta != 0.0, batch=batch, **share)
        want = oracle_answer(ko.MKM, M, Ps, Ps, X, Fs, Y, alpha, beta, **kw)
        got, e = run_gpu(fk, ko.MKM, M, Ps, Ps, X, Fs, Y, alpha, beta, **kw)
        assert e == 0 and normwise(got, want) <= TOL[dt], (fk.last_plan(), kw)
        assert few_long_rows or "inplace" in fk.last_plan()[0][2], fk.last_plan()


# rows, factors, type: more rows than the device holds at once (workgroups that go from row to row, the next one loaded
# ahead): a few more, a few less than twice as many, and sizes at which operands are streamed
MANY = [(515, 5, 6, "f"), (1030, 5, 6, "f"), (258, 5, 6, "d"), (517, 7, 5, "f"), (259, 7, 5, "d"), (1027, 6, 5, "f"), (513, 6, 5, "d"),
        (1283, 3, 8, "f"), (771, 3, 8, "d"), (2563, 5, 5, "f"), (1539, 5, 5, "d"), (3077, 7, 4, "f"), (2200, 3, 8, "d"), (16000, 5, 5, "f")]


@pytest.mark.parametrize("M,P,n,t", MANY, ids=lambda v: str(v))
def test_more_rows_than_the_device_holds(fk, M, P, n, t):
    dt = np.float32 if t == "f" else np.float64
    Ps = [P] * n
    for seed, (m, kw) in enumerate([(M, dict(alpha=1.5, beta=0.5)), (M, dict(alpha=1.0, beta=0.0, opFs=ko.OP_T)),
                                    (M // 3 + 1, dict(alpha=-1.0, beta=0.0, batch=3))]):
        alpha, beta, batch = kw.pop("alpha"), kw.pop("beta"), kw.get("batch", 1)
        X, Fs, Y = make_case(ko.MKM, m, Ps, Ps, dt, seed=11 + seed, with_y=beta != 0.0, batch=batch)
        want = oracle_answer(ko.MKM, m, Ps, Ps, X, Fs, Y, alpha, beta, **kw)
        got, e = run_gpu(fk, ko.MKM, m, Ps, Ps, X, Fs, Y, alpha, beta, **kw)
        assert e == 0 and normwise(got, want) <= TOL[dt], (fk.last_plan(), kw)
        assert len(fk.last_plan()) == 1 and "inplace" in fk.last_plan()[0][2], fk.last_plan()


def test_rows_off_a_16_byte_boundary(fk):
    """Base addresses that are only 4-byte aligned, of X and of Z, and the in-place epilogue (Y is Z)."""
    import torch
    M, Ps = 6, [5, 5, 5, 5]
    K = 625
    X, Fs, Y = make_case(ko.MKM, M, Ps, Ps, np.float32, seed=3)
    want = oracle_answer(ko.MKM, M, Ps, Ps, X, Fs, Y, 1.5, 0.5).reshape(-1)
    fs = [torch.from_numpy(f).cuda() for f in Fs]
    for off in (1, 2, 3):
        x = torch.full((M * K + 8,), float("nan"), device="cuda")
        z = torch.full((M * K + 8,), 77.0, device="cuda")
        x[off:off + M * K] = torch.from_numpy(X).cuda().reshape(-1)
        z[off:off + M * K] = torch.from_numpy(Y).cuda().reshape(-1)
        t1, t2 = torch.empty(M * K, device="cuda"), torch.empty(M * K, device="cuda")
        zv = z[off:off + M * K]
        assert fk.xgemkm(M, Ps, Ps, x[off:off + M * K], fs, zv, 1.5, 0.5, zv, t1, t2) == 0
        torch.cuda.synchronize()
        assert "inplace" in fk.last_plan()[0][2]
        assert normwise(zv.cpu().numpy(), want) <= TOL[np.float32]
        assert bool((z[:off] == 77.0).all()) and bool((z[off + M * K:] == 77.0).all())

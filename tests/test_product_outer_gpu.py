"""fastKronProductOuter (include/fastkron_ext.h) against one oracle call per entry: X along one dimension, the factors along the
other, X and Y shared along one, both or none of them, one entry in either, op N and T, Y and Z one buffer.  Result and
temporaries are NaN before the call, so what a launch reads must have been written.  TOL of gpu_util."""
import ctypes

import numpy as np
import pytest

from fastkron_amd import capi
from oracle import kron_oracle as ko
from tests.gpu_util import TOL, normwise, seeded

pytestmark = pytest.mark.gpu

PROBLEMS = [  # layout, rows or columns, factors (P, Q)
    (ko.MKM, 8, [(8, 8)] * 5), (ko.MKM, 5, [(5, 5)] * 3), (ko.MKM, 7, [(31, 18), (9, 20)]), (ko.MKM, 3, [(3, 4), (4, 2)]), (ko.MKM, 2, [(10, 10)] * 3),
    (ko.KMM, 9, [(7, 7)] * 4), (ko.KMM, 3, [(4, 3), (5, 6)]), (ko.KMM, 2, [(50, 40)]), (ko.KMM, 1, [(6, 6)] * 3), (ko.MKM, 4, [(4, 4)] * 6),
    (ko.MKM, 5, [(7, 7)] * 4), (ko.MKM, 2, [(5, 5)] * 6), (ko.MKM, 1, [(9, 9)] * 3)]
# entries of the two dimensions, which of them X and Y have
CALLS = [((1, 1), (1, 1), (1, 1)), ((3, 1), (1, 0), (1, 0)), ((1, 3), (0, 1), (0, 0)), ((2, 3), (1, 0), (1, 1)), ((2, 3), (0, 0), (1, 1)),
         ((3, 2), (1, 1), (0, 1)), ((4, 2), (0, 1), (1, 0)), ((3, 1), (0, 0), (1, 1))]


@pytest.fixture(scope="module")
def fk():
    import fastkron_amd
    h = fastkron_amd.FastKron()
    yield h
    h.close()


def outer_call(fk, mm, dt, M, Ps, Qs, count, X, sx, Fs, Z, sz, alpha, beta, Y, sy, t1, t2, opX, opF):
    p = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None
    return fk.lib.fastKronProductOuter(fk.h, mm == ko.MKM, dt == np.float64, M, len(Ps), capi.arr_u32(Ps), capi.arr_u32(Qs), p(X), opX, capi.arr_u64(sx),
                                       capi.arr_ptr([f.data_ptr() for f in Fs]), opF, p(Z), capi.arr_u64(sz), alpha, beta, capi.arr_u32(count), p(Y),
                                       capi.arr_u64(sy), p(t1), p(t2))


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
@pytest.mark.parametrize("mm,M,fs", PROBLEMS, ids=lambda v: str(v) if isinstance(v, int) else "x".join("%d:%d" % f for f in v))
def test_every_entry_is_its_own_product(fk, mm, M, fs, dt):
    import torch
    Ps, Qs = [p for p, _ in fs], [q for _, q in fs]
    K, L = int(np.prod(Ps)), int(np.prod(Qs))
    _, te = fk.sizes(M, Ps, Qs)
    for n, (count, xd, yd) in enumerate(CALLS):
        opX, opF, inplace = (ko.OP_T if n % 2 else ko.OP_N), (ko.OP_T if n % 3 == 1 else ko.OP_N), yd == (1, 1) and n % 2 == 1
        nb = count[0] * count[1]
        strides = lambda d, block: [(count[1] if d[1] else 1) * block * d[0], block * d[1]]
        sx, sy, sz = strides(xd, M * K), strides(yd, M * L), [count[1] * M * L, M * L]
        X = seeded(3 + n, (nb, M * K), dt)[:1 + (sx[0] * (count[0] - 1) + sx[1] * (count[1] - 1)) // (M * K)]
        Y = seeded(90 + n, (nb, M * L), dt)[:1 + (sy[0] * (count[0] - 1) + sy[1] * (count[1] - 1)) // (M * L)]
        Fs = [seeded(30 + n + i, (count[1], p * q), dt) for i, (p, q) in enumerate(fs)]
        dev = lambda a: torch.from_numpy(a).cuda()
        nan = lambda k: torch.full((k,), float("nan"), dtype=dev(X[:0]).dtype, device="cuda")
        Z = dev(Y).reshape(-1) if inplace else nan(nb * M * L)
        x, y, f = dev(X), Z if inplace else dev(Y), [dev(a) for a in Fs]
        e = outer_call(fk, mm, dt, M, Ps, Qs, count, x, sx, f, Z, sz, 1.5, 0.5, y, sy, nan(nb * te), nan(nb * te), opX, opF)
        torch.cuda.synchronize()
        assert e == capi.SUCCESS
        got = Z.cpu().numpy().reshape(nb, M * L)
        for o in range(count[0]):
            for i in range(count[1]):
                want = ko.sliced_multiply(mm, M, Ps, Qs, X[(o * sx[0] + i * sx[1]) // (M * K)].reshape(1, -1), [a[i].reshape(1, -1) for a in Fs], alpha=1.5,
                                          beta=0.5, Y=Y[(o * sy[0] + i * sy[1]) // (M * L)].reshape(1, -1), opX=opX, opFs=opF, batch=1, strideX=M * K,
                                          strideF=[0] * len(fs), strideZ=M * L, strideY=M * L)
                assert normwise(got[o * count[1] + i], want) <= TOL[dt], (fk.last_plan(), count, xd, yd, o, i)

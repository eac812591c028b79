"""Batches of several dimensions through the PyTorch front end: X and the factors broadcast against each other along different
ones (one series of launches with both, or a loop), alike in several (one dimension of the call), Y broadcast as well; against
dense Kronecker products in 64 bits.  Sums of at most 512 terms in two or three factors: u * 3 * 8 bounds the error per factor
chain at 1.5e-6 / 2.7e-15 of the largest value."""
import numpy as np
import pytest

from tests.kron_ref import kmm_dense, mkm_dense, normwise

pytestmark = pytest.mark.gpu

CASES = [
    # X's and the factors' batch dimensions, Y's
    ((2, 1), (3,), (2, 3)), ((3, 1), (4,), ()), ((5,), (2, 1), (2, 1)), ((2, 4), (2, 4), (4,)), ((2, 4), (4,), (2, 1)), ((2, 1, 3), (2, 4, 1), ()),
    ((1, 3), (2, 1), (1, 1)), ((4, 1), (1,), (4, 1)), ((), (2, 3), (3,)), ((1, 1), (1, 1), (1, 1)), ((9, 1), (2,), (9, 2)), ((2, 3), (2, 1), (2, 3)),
]


@pytest.mark.parametrize("dt", ["float32", "float64"])
@pytest.mark.parametrize("mm", ["mkm", "kmm"])
@pytest.mark.parametrize("ps,m", [([8, 8, 8], 8), ([5, 5, 5], 3), ([9, 14], 5), ([3, 4], 2), ([31, 2], 4)], ids=lambda v: str(v))
def test_batches_of_several_dimensions(mm, dt, ps, m):
    import torch
    import fastkron_amd as fk
    dtype = getattr(torch, dt)
    gen = torch.Generator().manual_seed(5)
    k = int(np.prod(ps))
    for n, (xb, fb, yb) in enumerate(CASES):
        trx, trf = n % 3 == 0, n % 2 == 0
        zb = tuple(torch.broadcast_shapes(xb, fb))
        mat = lambda b, r, c, t: (torch.rand(b + ((c, r) if t else (r, c)), generator=gen, dtype=dtype) * 2 - 1).cuda().requires_grad_(False)
        x = mat(xb, *((m, k) if mm == "mkm" else (k, m)), trx)
        fs = [mat(fb, p, p, trf) for p in ps]
        x, fs = x.mT if trx else x, [f.mT if trf else f for f in fs]
        y = mat(yb, *((m, k) if mm == "mkm" else (k, m)), False)
        z = fk.gemkm(x, fs, 1.5, 0.5, y) if mm == "mkm" else fk.gekmm(fs, x, 1.5, 0.5, y)
        assert tuple(z.shape[:-2]) == zb
        flat = lambda t: t.expand(zb + t.shape[-2:]).reshape((-1,) + t.shape[-2:]).double().cpu().numpy()
        X, Y, Z, F = flat(x), flat(y), flat(z), [flat(f) for f in fs]
        for b in range(X.shape[0]):
            want = (mkm_dense if mm == "mkm" else kmm_dense)(X[b], [f[b] for f in F], 1.5, 0.5, Y[b])
            assert normwise(Z[b], want) <= (1e-5 if dt == "float32" else 1e-12), (xb, fb, yb, b)


def test_both_dimensions_are_one_series_of_launches():
    import torch
    import fastkron_amd as fk
    h = fk.default_handle()
    x = torch.randn(2, 1, 32768, 32, device="cuda").mT
    fs = [torch.randn(3, 8, 8, device="cuda").mT for _ in range(5)]
    z = fk.gemkm(x, fs)
    plan = h.last_plan()
    assert len(plan) == 2 and plan[0][2].startswith("transpose_") and "_8x8_8x8_5_1x32768" in plan[1][2], plan
    for i in range(2):
        for j in range(3):
            assert torch.equal(z[i, j], fk.gemkm(x[i, 0].contiguous(), [f[j].contiguous() for f in fs]))


@pytest.mark.parametrize("xb,fb", [((5, 1), (2,)), ((2,), (5, 1)), ((3, 1), (4,)), ((4,), (3, 1))])
@pytest.mark.parametrize("dt,m,ps", [("float64", 3, [5] * 6), ("float64", 30, [6, 4, 2, 8, 7]), ("float32", 5, [7, 3, 9, 5, 4])], ids=lambda v: str(v))
def test_gekmm_of_a_transposed_x_keeps_to_its_entries_of_the_result(dt, m, ps, xb, fb):
    """The calls' entries lie between those of other calls, in chains whose GeMKM takes several launches."""
    import torch
    import fastkron_amd as fk
    dtype, k = getattr(torch, dt), int(np.prod(ps))
    x = torch.randn(xb + (m, k), device="cuda", dtype=dtype).mT
    fs = [torch.randn(fb + (p, p), device="cuda", dtype=dtype) / p ** 0.5 for p in ps]
    z = fk.gekmm(fs, x)
    zb = tuple(torch.broadcast_shapes(xb, fb))
    X, F = x.expand(zb + (k, m)), [f.expand(zb + f.shape[-2:]) for f in fs]
    for at in np.ndindex(*zb):
        want = X[at].double()
        for i, f in enumerate(F):
            v = want.reshape(int(np.prod(ps[:i])), ps[i], -1)
            want = torch.matmul(f[at].double(), v).reshape(k, m)
        assert normwise(z[at].cpu().numpy(), want.cpu().numpy()) <= (1e-5 if dt == "float32" else 1e-12), at


@pytest.mark.parametrize("ps,m,kernel", [([8] * 3, 8, "_small_fused_inplace_"), ([5] * 3, 3, "_small_fused_inplace_"), ([9, 14], 5, "_anyxany_64x64_2_"),
                                         ([3, 4], 2, "_small_fused_inplace_"), ([13] * 3, 4, "_generic_")], ids=lambda v: str(v))
def test_the_kernels_of_two_dimensions_run_them_as_one_call(ps, m, kernel):
    import ctypes
    import torch
    import fastkron_amd as fk
    h = fk.default_handle()
    fk.gemkm(torch.randn(2, 1, m, int(np.prod(ps)), device="cuda"), [torch.randn(3, p, p, device="cuda") for p in ps])
    buf = ctypes.create_string_buffer(4096)
    h.lib.fastKronGetLastPlan(h.h, buf, 4096)
    assert "_stridedBatched_6" in buf.value.decode() and kernel in buf.value.decode(), buf.value


def test_empty_dimensions_as_before():
    import torch
    import fastkron_amd as fk
    fs = [torch.randn(3, 4, 4, device="cuda") for _ in range(2)]
    assert fk.gemkm(torch.randn(0, 1, 5, 16, device="cuda"), fs).shape == (0, 3, 5, 16)
    with pytest.raises(fk.FastKronError):
        fk.gemkm(torch.randn(3, 0, 5, 16, device="cuda"), [torch.randn(0, 4, 4, device="cuda") for _ in range(2)])


@pytest.mark.parametrize("xb,fb,entries", [((6, 1), (2,), 2), ((3, 2), (3, 2), 2), ((6, 1), (6, 1), 1)])
def test_temporaries_of_large_entries_stay_those_of_the_innermost_dimension(xb, fb, entries):
    """Entries of 64 MB: two temporaries of as many as the innermost dimension has, not of all that could be one call."""
    import torch
    import fastkron_amd as fk
    x = torch.randn(xb + (4096, 4096), device="cuda")
    fs = [torch.randn(fb + (64, 64), device="cuda") / 8 for _ in range(2)]
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    z = fk.gemkm(x, fs)
    torch.cuda.synchronize()
    entry = 4096 * 4096 * 4
    assert torch.cuda.max_memory_allocated() - before <= z.numel() * 4 + max(2 * entries * entry, 512 << 20) + (8 << 20)
    last = tuple(n - 1 for n in z.shape[:-2])
    at = lambda t: t[tuple(min(i, n - 1) for i, n in zip(last[len(last) - t.dim() + 2:], t.shape[:-2]))]
    want = fk.gemkm(at(x).contiguous(), [at(f).contiguous() for f in fs])
    assert (z[last] - want).abs().max() <= 1e-5 * want.abs().max()

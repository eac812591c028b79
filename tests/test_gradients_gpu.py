"""Gradients of gemkm / gekmm (kernels/gradient_mfma.hip) against PyTorch's autograd of the dense Kronecker product in
float64 on the CPU.  Bounds: a factor gradient is a sum of n = rows products of random sign; with u the unit roundoff a
sum of n terms in blocks of 16 and then pairs of waves has an error of about sqrt(n) * u in the norm of the result, here
n <= 2^14: 128 u (fp32 7.6e-6, fp64 1.4e-14), doubled for the steps in front of it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BOUND = {"float32": 2 * 128 * 2.0 ** -24, "float64": 2 * 128 * 2.0 ** -53}

CASES = [
    # mm, m, (P, Q) of every factor, batch of x, of the factors, x transposed, factors transposed
    ("mkm", 64, [(16, 16), (16, 16)], (), (), False, False),          # whole tiles, one block
    ("mkm", 5, [(3, 3), (5, 2), (4, 7)], (), (), False, False),       # small, ragged
    ("kmm", 7, [(3, 3), (5, 2), (4, 7)], (), (), False, True),        # rows of 7: no 16-byte accesses
    ("kmm", 64, [(8, 8), (8, 8), (8, 8)], (), (), True, False),       # X copied transposed
    ("mkm", 33, [(32, 32), (32, 32)], (), (), False, False),          # two blocks, last tile incomplete
    ("mkm", 9, [(31, 17), (18, 33)], (), (), True, True),             # padded blocks
    ("mkm", 3, [(64, 64), (50, 64)], (), (), False, False),           # 64x64 block
    ("mkm", 4, [(100, 70)], (), (), False, False),                    # several blocks of the factor, one step
    ("kmm", 20, [(128, 128), (2, 2)], (), (), False, False),
    ("mkm", 3, [(2, 3), (260, 300)], (), (), False, False),           # F beyond LDS in fp64
    ("kmm", 1, [(16, 16), (4, 4)], (), (), False, False),             # a single column
    ("mkm", 1, [(4, 4)] * 6, (), (), False, False),                   # one row
    ("mkm", 6, [(8, 8), (8, 8)], (3,), (), False, False),             # batch of X, shared factors
    ("kmm", 6, [(12, 12), (9, 9)], (3,), (), False, False),
    ("mkm", 6, [(16, 8), (8, 16)], (), (4,), False, False),           # shared X, factors per entry
    ("kmm", 5, [(6, 6), (4, 4), (5, 5)], (2, 1), (3,), False, True),  # broadcast both ways
    ("mkm", 8, [(16, 16), (16, 16)], (2, 3), (2, 3), True, False),
    ("mkm", 6, [(8, 3), (5, 5)], (3,), (), True, False),              # a transposed X larger than Z: read as it is stored
    ("kmm", 6, [(8, 3), (5, 5)], (2,), (2,), True, True),
    ("mkm", 9, [(20, 30)], (2,), (), True, False),                    # ... and in a single step
    ("kmm", 9, [(20, 30)], (), (), True, False),
    ("mkm", 6, [(3, 8), (5, 5)], (3,), (), True, False),              # ... copied to Z, batch folded into rows
    ("kmm", 6, [(3, 8), (5, 5)], (2, 1), (3,), True, False),
    ("mkm", 5, [(2, 3), (258, 260)], (2,), (), True, False),          # a first factor of the plain kernel: as it is stored
    ("kmm", 5, [(2, 3), (3, 515)], (), (), True, True),
    # steps whose input's gradient is a product of PyTorch's, alone, in front of, behind and between steps that are not
    ("mkm", 5, [(130, 400)], (), (), False, True),
    ("kmm", 5, [(40, 400)], (), (), False, False),
    ("mkm", 3, [(4, 390), (3, 5)], (), (), False, False),
    ("kmm", 3, [(3, 5), (4, 390)], (), (), False, True),
    ("mkm", 2, [(2, 3), (5, 387), (3, 2)], (2,), (), True, False),
    ("kmm", 2, [(2, 3), (5, 387), (3, 2)], (2,), (), False, False),
    ("kmm", 2, [(3, 385), (2, 385)], (), (2,), False, True),
    ("mkm", 3, [(7, 385), (2, 2)], (2, 1), (3,), False, False),
    ("kmm", 1, [(7, 385), (2, 2)], (3,), (), False, False),
]


def reference(mm, x, fs, gz):
    """Gradients from dense products in float64 on the CPU."""
    import torch
    x = x.detach().cpu().double().requires_grad_(True)
    fs = [f.detach().cpu().double().requires_grad_(True) for f in fs]
    k = fs[0]
    for f in fs[1:]:
        k = (k[..., :, None, :, None] * f[..., None, :, None, :]).reshape(k.shape[:-2] + (k.shape[-2] * f.shape[-2], k.shape[-1] * f.shape[-1]))
    z = x @ k if mm == "mkm" else k @ x
    return z.detach(), torch.autograd.grad(z, [x, *fs], gz.cpu().double())


def operands(mm, m, shapes, xb, fb, trx, trf, dtype, seed=1):
    import torch
    g = torch.Generator().manual_seed(seed)
    k, l = int(np.prod([p for p, _ in shapes])), int(np.prod([q for _, q in shapes]))

    def rand(shape, tr):
        t = torch.randn(shape[:-2] + (shape[-1], shape[-2]) if tr else shape, generator=g, dtype=dtype).cuda()
        return t.mT if tr else t
    x = rand(xb + ((m, k) if mm == "mkm" else (k, m)), trx)
    fs = [rand(fb + ((p, q) if mm == "mkm" else (q, p)), trf) for p, q in shapes]
    zb = tuple(torch.broadcast_shapes(xb, fb))
    return x, fs, rand(zb + ((m, l) if mm == "mkm" else (l, m)), False)


def rel(a, b):
    return float((a.cpu().double() - b).norm() / b.norm())


@pytest.mark.parametrize("dt", ["float32", "float64"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}_{c[1]}_{'_'.join('%dx%d' % s for s in c[2])}_{c[3]}_{c[4]}_{int(c[5])}{int(c[6])}")
def test_gradients(case, dt):
    import torch
    import fastkron_amd as fk
    mm, m, shapes, xb, fb, trx, trf = case
    x, fs, gz = operands(mm, m, shapes, xb, fb, trx, trf, getattr(torch, dt))
    zr, want = reference(mm, x, fs, gz)
    x.requires_grad_(True)
    for f in fs:
        f.requires_grad_(True)
    z = fk.gemkm(x, fs) if mm == "mkm" else fk.gekmm(fs, x)
    assert rel(z.detach(), zr) <= BOUND[dt]
    got = torch.autograd.grad(z, [x, *fs], gz, retain_graph=True)
    for a, b in zip(got, want):
        assert a.shape == b.shape and rel(a, b) <= BOUND[dt]
    again = torch.autograd.grad(z, [x, *fs], gz, retain_graph=True)
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    # a single factor's gradient, the chain cut short
    only = torch.autograd.grad(z, [fs[0]], gz)[0]
    assert rel(only, want[1]) <= BOUND[dt]


@pytest.mark.parametrize("mm", ["mkm", "kmm"])
def test_many_rows(mm):
    """Every workgroup takes several tiles and the partial sums of all of them are added: 2^18 rows of integers, exact."""
    import torch
    import fastkron_amd as fk
    g = torch.Generator().manual_seed(3)
    x = torch.randint(-2, 3, (2 ** 15, 64) if mm == "mkm" else (64, 2 ** 15), generator=g).float().cuda()
    fs = [torch.randint(-2, 3, s, generator=g).float().cuda().requires_grad_(True) for s in ((8, 8), (8, 8))]
    gz = torch.randint(-1, 2, x.shape, generator=g).float().cuda()
    z = fk.gemkm(x, fs) if mm == "mkm" else fk.gekmm(fs, x)
    got = torch.autograd.grad(z, fs, gz)
    _, want = reference(mm, x, fs, gz)
    for a, b in zip(got, want[1:]):
        assert torch.equal(a.cpu().double(), b)


@pytest.mark.parametrize("need", ["x", "factors"])
@pytest.mark.parametrize("mm", ["mkm", "kmm"])
def test_gradient_of_a_gradient(mm, need):
    """create_graph with gradients of X alone or of the factors alone: the norm of the gradient is differentiated, in float64
    against the dense product on the CPU."""
    import torch
    import fastkron_amd as fk
    x, fs, _ = operands(mm, 3, [(3, 2), (2, 4)], (), (), False, True, torch.float64)

    def second(x, fs, product):
        w = [t.requires_grad_(True) for t in ([x] if need == "x" else fs)]
        first = torch.autograd.grad((product(x, fs) ** 2).sum(), w, create_graph=True)
        return torch.autograd.grad(sum((g ** 2).sum() for g in first), w)
    got = second(x, fs, lambda x, fs: fk.gemkm(x, fs) if mm == "mkm" else fk.gekmm(fs, x))
    want = second(x.detach().cpu(), [f.detach().cpu() for f in fs], lambda x, fs: x @ torch.kron(*fs) if mm == "mkm" else torch.kron(*fs) @ x)
    for a, b in zip(got, want):
        assert rel(a, b) <= BOUND["float64"]


def test_backward_of_a_backward_pass():
    """create_graph: the backward pass is differentiated once more."""
    import torch
    import fastkron_amd as fk
    for mm in ("mkm", "kmm"):
        x, fs, _ = operands(mm, 3, [(3, 2), (2, 4)], (), (), False, False, torch.float64)
        x.requires_grad_(True)
        for f in fs:
            f.requires_grad_(True)
        fn = fk.MKM.apply if mm == "mkm" else fk.KMM.apply
        assert torch.autograd.gradgradcheck(fn, (x, *fs), eps=1e-6, atol=1e-5)


def library_gradients(mm, x, fs, gz):
    """Z and the gradients of X and of every factor through the C functions, operands stored row-major, no batch."""
    import ctypes
    import torch
    import fastkron_amd as fk
    from fastkron_amd import capi
    h = fk.default_handle()
    h.set_stream(torch.cuda.current_stream())
    mkm, dbl = int(mm == "mkm"), int(x.dtype == torch.float64)
    M = x.shape[0] if mkm else x.shape[1]
    shape = (M, len(fs), capi.arr_u32([f.shape[0 if mkm else 1] for f in fs]), capi.arr_u32([f.shape[1 if mkm else 0] for f in fs]))
    save, work = ctypes.c_size_t(), ctypes.c_size_t()
    assert h.lib.fastKronGradSizes(h.h, mkm, dbl, *shape, capi.OP_N, 0, 0, 1, ctypes.byref(save), ctypes.byref(work)) == 0
    new = lambda *s: torch.full(s, float("nan"), dtype=x.dtype, device="cuda")
    kept, scratch, z, gx, gf = new(save.value), new(work.value), torch.empty_like(gz), torch.empty_like(x), [torch.empty_like(f) for f in fs]
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    args = (h.h, mkm, dbl, *shape, ptr(x), capi.OP_N, 0, capi.arr_ptr([f.data_ptr() for f in fs]), capi.OP_N, 0, 1)
    assert h.lib.fastKronGradForward(*args, ptr(z), ptr(kept)) == 0
    assert h.lib.fastKronGradBackward(*args, ptr(gz), ptr(kept), ptr(gx), capi.arr_ptr([g.data_ptr() for g in gf]), ptr(scratch)) == 0
    torch.cuda.synchronize()
    return z, gx, gf


@pytest.mark.parametrize("dt", ["float32", "float64"])
@pytest.mark.parametrize("mm", ["mkm", "kmm"])
@pytest.mark.parametrize("Q", [17, 70, 281, 553])                   # one block, several, F beyond LDS in fp64, in either type
def test_infinities_stay_where_they_are(Q, mm, dt):
    """Blocks of 16 are padded: what stands beside the padding must not enter it as 0 * inf."""
    import torch
    x, fs, gz = operands(mm, 5, [(20, Q)], (), (), False, False, getattr(torch, dt))
    (fs[0] if mm == "mkm" else fs[0].t())[3, Q - 1] = float("inf")
    (x if mm == "mkm" else x.t())[2, 19] = float("-inf")
    _, gx, gf = library_gradients(mm, x, fs, gz)
    X, F, G = (t.cpu().double() if mm == "mkm" else t.cpu().double().t() for t in (x, fs[0], gz))
    for got, want in ((gx, G @ F.t()), (gf[0], X.t() @ G)):
        got = got.cpu().double() if mm == "mkm" else got.cpu().double().t()
        assert torch.equal(got.isinf(), want.isinf()) and torch.equal(got[got.isinf()], want[want.isinf()])
        fin = want.isfinite()
        assert float((got[fin] - want[fin]).norm() / want[fin].norm()) <= BOUND[dt]


@pytest.mark.parametrize("create_graph", [False, True])
@pytest.mark.parametrize("need", ["x", "factors", "all"])
@pytest.mark.parametrize("mm", ["mkm", "kmm"])
@pytest.mark.parametrize("fb", [(), (3,), (2, 3)])
def test_gradients_of_a_vector(fb, mm, need, create_graph):
    """X of one dimension; against a batch of factors its gradient is the sum over the entries, each with its own result."""
    import torch
    import fastkron_amd as fk
    g = torch.Generator().manual_seed(1)
    x = torch.randn(12, generator=g, dtype=torch.float64).cuda()
    fs = [torch.randn(fb + ((p, q) if mm == "mkm" else (q, p)), generator=g, dtype=torch.float64).cuda() for p, q in ((3, 2), (4, 5))]
    gz = torch.randn(fb + (10,), generator=g, dtype=torch.float64).cuda()
    _, want = reference(mm, x, fs, gz)
    needed = [need != "factors"] + [need != "x"] * 2
    for t, n in zip([x, *fs], needed):
        t.requires_grad_(n)
    z = fk.gemkm(x, fs) if mm == "mkm" else fk.gekmm(fs, x)
    got = torch.autograd.grad(z, [t for t, n in zip([x, *fs], needed) if n], gz, create_graph=create_graph)
    for a, b in zip(got, [w for w, n in zip(want, needed) if n]):
        assert a.shape == b.shape and rel(a.detach(), b) <= BOUND["float64"]


@pytest.mark.parametrize("need", ["x", "factors", "all"])
@pytest.mark.parametrize("mm", ["mkm", "kmm"])
@pytest.mark.parametrize("xb,fb", [((), ()), ((2, 1), (3,)), (None, (3,))])           # None: X of one dimension
def test_batches_of_gradients(xb, fb, mm, need):
    """is_grads_batched and jacobian(vectorize=True) against one gradient at a time."""
    import torch
    import fastkron_amd as fk
    x, fs, _ = operands(mm, 3 if xb is not None else 1, [(3, 2), (2, 4)], xb or (), fb, False, False, torch.float64)
    x = x.reshape(-1) if xb is None else x
    needed = [need != "factors"] + [need != "x"] * 2
    for t, n in zip([x, *fs], needed):
        t.requires_grad_(n)
    product = lambda *t: fk.gemkm(t[0], t[1:]) if mm == "mkm" else fk.gekmm(t[1:], t[0])
    z, w = product(x, *fs), [t for t, n in zip([x, *fs], needed) if n]
    gz = torch.randn((4,) + z.shape, dtype=z.dtype, device="cuda")
    one = [torch.autograd.grad(z, w, g, retain_graph=True) for g in gz]
    for i, a in enumerate(torch.autograd.grad(z, w, gz, is_grads_batched=True)):
        assert rel(a, torch.stack([g[i] for g in one]).cpu()) <= BOUND["float64"]
    at = lambda *t: product(*[t[needed[:i].count(True)] if n else u for i, (u, n) in enumerate(zip([x, *fs], needed))])
    jacobian = lambda v: torch.autograd.functional.jacobian(at, tuple(t.detach() for t in w), vectorize=v)
    for a, b in zip(jacobian(True), jacobian(False)):
        assert a.shape == b.shape and rel(a, b.cpu()) <= BOUND["float64"]


@pytest.mark.parametrize("mm", ["mkm", "kmm"])
def test_a_transposed_x_is_not_kept_as_a_copy(mm):
    """Between the passes a call holds its result and the steps' outputs, however X is stored."""
    import torch
    import fastkron_amd as fk

    def held(transposed, n):
        fs = [torch.randn(16, 16, device="cuda", requires_grad=True) for _ in range(n)]
        rows, cols = (512, 16 ** n) if mm == "mkm" else (16 ** n, 512)
        x = torch.randn(cols, rows, device="cuda").t() if transposed else torch.randn(rows, cols, device="cuda")
        before = torch.cuda.memory_allocated()
        z = fk.gemkm(x, fs) if mm == "mkm" else fk.gekmm(fs, x)
        return torch.cuda.memory_allocated() - before
    for n in (1, 3):
        assert held(True, n) == held(False, n)

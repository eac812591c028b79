"""The native host path of the PyTorch front end (csrc/frontend.cpp): operands that are stored in unusual ways against the
same call on plain copies (equal bits: the same kernels on the same values; where a transposed view takes another kernel,
TOL of gpu_util), refused operands, streams, and operands that come back from saved-tensor hooks stored another way."""
import numpy as np
import pytest

from tests.gpu_util import TOL, normwise

pytestmark = pytest.mark.gpu


def rand(*shape, dtype=None):
    import torch
    return torch.randn(*shape, dtype=dtype or torch.float32, device="cuda")


@pytest.mark.parametrize("mm", ["mkm", "kmm"])
def test_unusual_storage(mm):
    import torch
    import fastkron_amd as fk
    call = (lambda x, fs, **k: fk.gemkm(x, fs, **k)) if mm == "mkm" else (lambda x, fs, **k: fk.gekmm(fs, x, **k))
    torch.manual_seed(1)
    shape = (6, 30) if mm == "mkm" else (30, 6)
    fs = [rand(5, 5), rand(6, 6)]
    x = rand(*shape)
    want = call(x, fs)
    wide = rand(shape[0], 2 * shape[1])
    wide[:, ::2] = x
    assert torch.equal(call(wide[:, ::2], fs), want)                            # neither contiguous nor transposed
    assert normwise(call(x.t().contiguous().t(), fs).cpu(), want.cpu()) <= TOL[np.float32]
    mixed = [fs[0], fs[1].t().contiguous().t()]                                 # factors stored differently
    assert torch.equal(call(x, mixed), want)
    assert torch.equal(call(x, tuple(fs)), want) and torch.equal(call(torch.nn.Parameter(x, requires_grad=False), fs), want)
    y = rand(3, 1, *shape)                                                      # Y broadcast over a part of the batch
    xb = rand(3, 2, *shape)
    got = call(xb, fs, alpha=2.0, beta=0.5, y=y)
    for i in range(3):
        for j in range(2):
            assert normwise(got[i, j].cpu(), (2.0 * call(xb[i, j], fs) + 0.5 * y[i, 0]).cpu()) <= TOL[np.float32]
    v = rand(60)[::2]                                                           # a strided vector
    assert torch.equal(call(v, fs), call(v.contiguous(), fs)) and call(v, fs).shape == (30,)
    bf = [rand(4, 5, 5), rand(4, 6, 6)]                                         # shared X, factors per entry
    got = call(x, bf)
    for i in range(4):
        assert normwise(got[i].cpu(), call(x, [f[i] for f in bf]).cpu()) <= TOL[np.float32]


def test_refused_operands():
    import torch
    import fastkron_amd as fk
    x, fs = rand(4, 16), [rand(4, 4), rand(4, 4)]
    for bad, kind in [((x, []), ValueError), ((x, fs[0]), ValueError), (("x", fs), ValueError), ((x, [fs[0], 3]), ValueError),
                      ((x, [fs[0], rand(4)]), ValueError), ((x, [fs[0], fs[1].cpu()]), RuntimeError),
                      ((x, [fs[0], rand(2, 4, 4)]), ValueError), ((rand(3, 4, 16), [rand(2, 4, 4)] * 2), ValueError),
                      ((x, fs, 1.0, 1.0, rand(4, 15)), ValueError), ((x, fs, 1.0, 1.0, rand(2, 4, 16)), ValueError),
                      ((x, fs, 1.0, 1.0, rand(4, 16).double()), ValueError), ((x[:0], fs), fk.FastKronError),
                      ((rand(4, 1), [rand(1, 1)] * 65), fk.FastKronError), ((rand(4, 0), [rand(0, 4), rand(4, 4)]), fk.FastKronError)]:
        with pytest.raises(kind):
            fk.gemkm(*bad)
    f = [t.clone().requires_grad_(True) for t in fs]
    with pytest.raises(ValueError):
        fk.MKM.apply(rand(4, 15), *f)


def test_calls_follow_the_current_stream():
    import torch
    import fastkron_amd as fk
    x, fs = rand(512, 4096), [rand(16, 16) for _ in range(3)]
    want = fk.gemkm(x, fs)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.cuda._sleep(2_000_000)
        x2 = x * 2.0
        z = fk.gemkm(x2, fs)                                                    # has to wait for x2
    side.synchronize()
    assert torch.equal(z, fk.gemkm(x2, fs)) and normwise(z.cpu(), 2.0 * want.cpu()) <= TOL[np.float32]


@pytest.mark.parametrize("mm", ["mkm", "kmm"])
def test_saved_tensors_may_come_back_stored_another_way(mm):
    import torch
    import fastkron_amd as fk
    fn = fk.MKM.apply if mm == "mkm" else fk.KMM.apply
    x = rand(24, 7).t() if mm == "mkm" else rand(7, 24).t()                     # transposed views
    fs = [rand(6, 6).t().requires_grad_(True), rand(4, 4).t().requires_grad_(True)]
    gz = rand(*((7, 24) if mm == "mkm" else (24, 7)))
    want = torch.autograd.grad(fn(x, *fs), fs, gz)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.cuda().contiguous()):
        z = fn(x, *fs)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(z, fs, gz), want))


@pytest.mark.parametrize("mm", ["mkm", "kmm"])
@pytest.mark.parametrize("change", ["half", "double", "cpu", "short", "sparse"])
def test_the_kept_buffer_has_to_come_back_as_it_was(mm, change):
    """The one saved tensor of one dimension is the buffer that the forward pass keeps; the kernels would read beyond a
    buffer of another type, or through a host address."""
    import torch
    import fastkron_amd as fk
    fn = fk.MKM.apply if mm == "mkm" else fk.KMM.apply
    x = rand(*((7, 24) if mm == "mkm" else (24, 7)))
    fs = [rand(6, 6).requires_grad_(True), rand(4, 4).requires_grad_(True)]
    unpack = {"half": lambda t: t.half(), "double": lambda t: t.double(), "cpu": lambda t: t.cpu(), "short": lambda t: t[:-1],
              "sparse": lambda t: t.to_sparse()}[change]
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: (seen.append(t), unpack(t))[1] if t.ndim == 1 else t):
        z = fn(x, *fs)
    with pytest.raises(RuntimeError, match="forward pass"):
        torch.autograd.grad(z, fs, torch.ones_like(z))
    assert len(seen) == 1


def test_row_counts_beyond_32_bits():
    """The C API counts rows in 32 bits: a folded batch of more rows goes entry by entry, one entry of more is refused (before
    anything of its size is allocated)."""
    import torch
    import fastkron_amd as fk
    f = [torch.full((1, 1), 3.0, device="cuda")]
    with pytest.raises(fk.FastKronError):
        fk.gemkm(rand(1, 1).expand(2 ** 32 + 4, 1), f)
    with pytest.raises(fk.FastKronError):
        fk.gekmm(f, rand(1, 1).expand(1, 2 ** 32 + 4))
    with pytest.raises(fk.FastKronError):
        fk.MKM.apply(rand(1, 1).expand(2 ** 32 + 4, 1), f[0].clone().requires_grad_(True))
    if torch.cuda.mem_get_info()[0] < 110 << 30:
        pytest.skip("needs 110 GB")
    x = torch.ones((2 ** 20 + 1, 4096, 1), device="cuda")                       # 2^32 + 4096 rows, 17 GB
    x[-1, -1] = 2.0
    z = fk.gemkm(x, f)
    x *= 3.0
    same = torch.equal(z, x)
    del x, z
    torch.cuda.empty_cache()
    assert same


@pytest.mark.parametrize("mm,xb,fb,taken", [
    ("mkm", (), (0, 3), True), ("mkm", (0, 3), (0, 3), True), ("mkm", (0, 3), (1, 3), True), ("mkm", (0, 2, 0), (0, 2, 0), True),
    ("kmm", (), (0, 3), True), ("kmm", (0, 3), (), True), ("kmm", (2, 0, 3), (), True),
    ("mkm", (0, 3), (), False), ("mkm", (3, 0), (3, 0), False), ("kmm", (3, 0), (3, 0), False), ("mkm", (0,), (0,), False), ("kmm", (), (0,), False)])
@pytest.mark.parametrize("need", ["", "x", "factors", "all"])
def test_empty_batches(mm, xb, fb, taken, need):
    """No entry along an outer batch dimension: an empty result and gradients of zeros, with every kind of gradient.  An
    empty innermost dimension, or rows folded to none, are refused, as the library refuses M = 0."""
    import torch
    import fastkron_amd as fk
    rows = lambda a, b: (a, b) if mm == "mkm" else (b, a)
    x, fs = rand(*xb, *rows(3, 6)), [rand(*fb, *rows(3, 2)), rand(*fb, *rows(2, 4))]
    x.requires_grad_(need in ("x", "all"))
    for f in fs:
        f.requires_grad_(need in ("factors", "all"))
    call = lambda: fk.gemkm(x, fs) if mm == "mkm" else fk.gekmm(fs, x)
    if not taken:
        with pytest.raises(fk.FastKronError):
            call()
        return
    z = call()
    assert z.shape == tuple(torch.broadcast_shapes(xb, fb)) + rows(3, 8)
    w = [t for t in [x, *fs] if t.requires_grad]
    for t, g in zip(w, torch.autograd.grad(z, w, torch.ones_like(z)) if w else []):
        assert g.shape == t.shape and not g.any()


@pytest.mark.parametrize("mm", ["mkm", "kmm"])
def test_a_recorded_call_copies_its_operands_once(mm):
    """A strided X and strided factors are copied by the autograd function, not by the call that finds it has to be recorded
    as well: gemkm allocates what the autograd function alone does."""
    import torch
    import fastkron_amd as fk
    x = rand(64, 2 * 4096)[:, ::2] if mm == "mkm" else rand(4096, 2 * 64)[:, ::2]
    fs = [rand(16, 32)[:, ::2].requires_grad_(True) for _ in range(3)]

    def allocated(call):
        before = torch.cuda.memory_stats()["allocated_bytes.all.allocated"]
        call()
        return torch.cuda.memory_stats()["allocated_bytes.all.allocated"] - before
    call = (lambda: fk.gemkm(x, fs)) if mm == "mkm" else (lambda: fk.gekmm(fs, x))
    fn = fk.MKM.apply if mm == "mkm" else fk.KMM.apply
    call()
    assert allocated(call) == allocated(lambda: fn(x, *fs))


def test_other_threads_run_during_a_call(monkeypatch):
    """A call that tunes keeps the host busy for milliseconds; a thread that ticks every half of one goes on meanwhile."""
    import threading
    import time
    import torch
    import fastkron_amd as fk
    handle = fk.FastKron(tune=True)
    handle.set_tuned_db("")
    monkeypatch.setattr(fk, "_default", handle)
    x, fs = rand(500, 21 ** 3), [rand(21, 21) for _ in range(3)]
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.wait(0.0005):
            ticks.append(time.perf_counter())
    thread = threading.Thread(target=tick)
    thread.start()
    begin = time.perf_counter()
    fk.gemkm(x, fs)
    end = time.perf_counter()
    stop.set()
    thread.join()
    inside = [begin] + [t for t in ticks if begin <= t <= end] + [end]
    longest = max(b - a for a, b in zip(inside, inside[1:]))
    assert end - begin > 0.004 and longest < 0.5 * (end - begin), (end - begin, longest)


def test_threads_with_streams_of_their_own():
    """Each call sets the shared handle's stream: two threads must not get in between, products and gradients alike."""
    import threading
    import torch
    import fastkron_amd as fk
    shapes = [(64, [4] * 5), (33, [5] * 4), (100, [16] * 3), (7, [31, 31])]
    errors = []

    def work(i):
        m, ps = shapes[i]
        g = torch.Generator(device="cuda").manual_seed(i)
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            fs = [torch.randn(p, p, device="cuda", generator=g).requires_grad_(True) for p in ps]
            x = torch.randn(m, int(np.prod(ps)), device="cuda", generator=g)
            want = fk.gemkm(x, [f.detach() for f in fs])
            grads = torch.autograd.grad(fk.gemkm(x, fs), fs, x)
            for n in range(40):
                y = x * 1.0                                                     # written on this stream just before it is read
                if not torch.equal(fk.gemkm(y, [f.detach() for f in fs]), want):
                    errors.append((i, n, "product"))
                if not all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(fk.gemkm(y, fs), fs, y), grads)):
                    errors.append((i, n, "gradients"))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(shapes))]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not errors, errors

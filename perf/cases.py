"""Performance cases: what programs have this framework do, from single small products to operands of a gigabyte.

A case is a dict of plain values:
  api      "torch": the PyTorch front end (`fastkron_amd.gemkm` / `gekmm`, autograd included);
           "handle": the C entry points through a handle, arguments marshalled once, as a program that repeats a
           product on resident buffers does (temporaries and result buffer are the program's own).
  mm       "mkm": Z = alpha X (F_0 (x) ... (x) F_{n-1}) + beta Y;  "kmm": Z = alpha (F_0 (x) ...) X + beta Y
  m        rows (mkm) / columns (kmm) of X per batch entry
  factors  "PxQ" per factor, separated by blanks: P inputs become Q outputs
  dtype    "float32" / "float64"
  trx, trf X / the factors are transposed views of row-major buffers
  xb, fb   batch dimensions of X and of the factors, e.g. "2,1" ("" for none); "handle" takes one dimension, and
           fb "" then means factors shared by the batch
  epilogue alpha = 1.5 and beta = 0.5 with a Y, instead of the plain product
  grad     "" (no gradient), "x", "factors" or "all": forward and backward pass, gradients of these operands
"""
import math

import torch

import fastkron_amd
from fastkron_amd import capi


def _case(name, api, mm, m, factors, dtype, trx=False, trf=False, xb="", fb="", epilogue=False, grad=""):
    return dict(name=name, api=api, mm=mm, m=m, factors=factors, dtype=dtype, trx=trx, trf=trf, xb=xb, fb=fb,
                epilogue=epilogue, grad=grad)


def _same(p, q, n):
    return " ".join([f"{p}x{q}"] * n)


def listed():
    return [
        # one vector against a small product: what an iterative solver or a sampler calls in its innermost loop, the
        # time is the call's own
        _case("vector_8x8^3", "torch", "mkm", 1, _same(8, 8, 3), "float32"),
        # a step of conjugate gradients on a grid of 16^3 points: few right hand sides, double precision, the shift
        # (K + s I) v as the epilogue
        _case("solver_16x16^3_f64", "torch", "kmm", 16, _same(16, 16, 3), "float64", epilogue=True),
        # rows of 16^4: the configuration the headline metric is quoted on
        _case("rows_16x16^4", "handle", "mkm", 1024, _same(16, 16, 4), "float32"),
        # few large factors in double precision, bound by the matrix cores
        _case("rows_64x64^3_f64", "handle", "mkm", 256, _same(64, 64, 3), "float64"),
        # many columns, small factors, with the epilogue
        _case("columns_4x4^6", "handle", "kmm", 2048, _same(4, 4, 6), "float32", epilogue=True),
        # a strided batch with factors of its own per entry that shrink their rows
        _case("batch_32x16^3", "handle", "mkm", 512, _same(32, 16, 3), "float32", xb="8", fb="8", epilogue=True),
        # sizes that are no powers of two, and rectangular: feature maps, grids of measured extent
        _case("ragged_31x63^2", "torch", "mkm", 1003, _same(31, 63, 2), "float32"),
        # small odd factors over several dimensions
        _case("odd_5x5^6", "handle", "mkm", 1001, _same(5, 5, 6), "float32"),
        # transposed views and batches of different shapes, broadcast between X and the factors
        _case("views_8x8^5", "torch", "mkm", 32, _same(8, 8, 5), "float32", trx=True, trf=True, xb="2,1", fb="3"),
        # a training step of a layer of 1024 features whose weight is a Kronecker product: every gradient
        _case("train_layer_32x32^2", "torch", "mkm", 4096, _same(32, 32, 2), "float32", grad="all"),
        # gradients of covariance factors on a grid, double precision, a few probe vectors as columns
        _case("train_grid_8x8^5_f64", "torch", "kmm", 16, _same(8, 8, 5), "float64", grad="factors"),
        # a chain longer than one launch takes, a gigabyte of X
        _case("long_8x8^6", "handle", "mkm", 1024, _same(8, 8, 6), "float32"),
    ]


# Limits of a drawn case, well inside the largest listed one (2.1 GB and 26 GFLOP)
_DRAW_BYTES = 400e6
_DRAW_TRAIN_BYTES = 120e6
_DRAW_FLOPS = 12e9


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_factors(rng):
    """2 to 8 factors, K between 2^6 and 2^20: equal square ones over the range of sizes, odd ones among them, equal
    rectangular ones, and mixed chains."""
    kind = rng.random()
    while True:
        if kind < 0.6:
            p = rng.choice([2, 3, 4, 5, 6, 7, 8, 8, 9, 10, 12, 13, 16, 16, 20, 24, 27, 31, 32, 32, 48, 50, 64, 64, 96, 100, 128, 128])
            ps = [(p, p)] * rng.randint(2, 8)
        elif kind < 0.8:
            p, q = rng.choice([(2, 4), (4, 2), (8, 16), (16, 8), (8, 32), (32, 8), (32, 16), (16, 32), (12, 16), (31, 63), (63, 31),
                               (32, 64), (64, 32), (24, 48), (64, 16), (50, 40), (100, 64), (3, 5), (7, 5)])
            ps = [(p, q)] * rng.randint(2, 6)
        else:
            ps = [(p, p) if rng.random() < 0.6 else (p, max(2, p + rng.randint(-p // 2, p // 2)))
                  for p in (rng.choice([2, 3, 4, 5, 6, 7, 8, 10, 12, 16, 20, 24, 32, 50, 64]) for _ in range(rng.randint(2, 6)))]
        k, l = math.prod(p for p, _ in ps), math.prod(q for _, q in ps)
        if 64 <= k <= 2 ** 20 and l <= 2 ** 20:
            return " ".join(f"{p}x{q}" for p, q in ps)


def draw(rng):
    """One more case of the same ranges: sizes spread over their logarithm, from a vector to 400 MB."""
    while True:
        api = rng.choice(["handle", "torch", "torch"])
        grad = rng.choice(["", "", "", "all", "factors", "x"]) if api == "torch" else ""
        mm = rng.choice(["mkm", "kmm"])
        trx, trf, xb, fb = False, False, "", ""
        if rng.random() < 0.2:
            trx, trf = rng.choice([(True, False), (False, True), (True, True)])
        if rng.random() < 0.25:
            b = rng.randint(2, 12)
            if api == "handle":
                xb, fb = str(b), rng.choice(["", str(b)])
            else:
                xb, fb = rng.choice([(f"{b}", ""), (f"{b}", f"{b}"), (f"{b},1", "3"), ("", f"{b}"), (f"2,{b}", f"2,{b}")])
        case = _case("", api, mm, _log_int(rng, 1, 4096), _draw_factors(rng), rng.choice(["float32", "float32", "float64"]), trx, trf,
                     xb, fb, epilogue=not grad and rng.random() < 0.3, grad=grad)
        del case["name"]
        w = work(case)
        # every step's output counts: a chain may grow before it shrinks
        batch, _, _, _ = _dims(case)
        widest = max(_widths(case)) * case["m"] * batch * (4 if case["dtype"] == "float32" else 8)
        if max(w["bytes"], 2 * widest) <= (_DRAW_TRAIN_BYTES if grad else _DRAW_BYTES) and w["flops"] <= _DRAW_FLOPS:
            return case


def _batch(text):
    return tuple(int(n) for n in text.split(",")) if text else ()


def _shapes(case):
    return [tuple(int(v) for v in f.split("x")) for f in case["factors"].split()]


def _widths(case):
    """Columns of X and of every step's output, the last factor first."""
    fs = _shapes(case)
    w = [math.prod(p for p, _ in fs)]
    for p, q in reversed(fs):
        w.append(w[-1] // p * q)
    return w


def _dims(case):
    """(batch entries of the result, of X, of the factors, floats per element of batch)"""
    xb, fb = _batch(case["xb"]), _batch(case["fb"])
    return math.prod(torch.broadcast_shapes(xb, fb)), math.prod(xb), math.prod(fb), len(_shapes(case))


def prepare(case, seed):
    """Inputs as such programs hold them: X and Y normal, factors normal with variance 1 / P (outputs then have the
    size of the inputs); for the handle also the result buffer and the two temporaries."""
    dev = torch.device("cuda:0")
    dt = getattr(torch, case["dtype"])
    gen = torch.Generator(device=dev).manual_seed(seed)
    fs = _shapes(case)
    m, k, l = case["m"], math.prod(p for p, _ in fs), math.prod(q for _, q in fs)
    xb, fb = _batch(case["xb"]), _batch(case["fb"])
    mkm = case["mm"] == "mkm"

    def normal(shape, transposed, scale=1.0):
        if transposed:
            shape = shape[:-2] + (shape[-1], shape[-2])
        t = torch.randn(shape, generator=gen, device=dev, dtype=dt) * scale
        return t.mT if transposed else t

    x = normal(xb + ((m, k) if mkm else (k, m)), case["trx"])
    factors = [normal(fb + ((p, q) if mkm else (q, p)), case["trf"], p ** -0.5) for p, q in fs]
    zshape = tuple(torch.broadcast_shapes(xb, fb)) + ((m, l) if mkm else (l, m))
    y = normal(zshape, False) if case["epilogue"] else None
    alpha, beta = (1.5, 0.5) if case["epilogue"] else (1.0, 0.0)
    if case["api"] == "torch":
        state = dict(mm=case["mm"], x=x, fs=factors, y=y, alpha=alpha, beta=beta, grad=case["grad"])
        if case["grad"]:
            x.requires_grad_(case["grad"] in ("x", "all"))
            for f in factors:
                f.requires_grad_(case["grad"] in ("factors", "all"))
            state["gz"] = normal(zshape, False)
        return state
    h = fastkron_amd.default_handle()
    h.set_stream(torch.cuda.current_stream())
    ps, qs = [p for p, _ in fs], [q for _, q in fs]
    batch = math.prod(xb)
    _, te = h.sizes(m, ps, qs)
    z = torch.empty(zshape, device=dev, dtype=dt)
    t1, t2 = (torch.empty(batch * te, device=dev, dtype=dt) for _ in range(2))
    ops = dict(opX=capi.OP_T if case["trx"] else capi.OP_N, opFs=capi.OP_T if case["trf"] else capi.OP_N)
    if xb:
        call = h.prepared("xgemkm_strided_batched" if mkm else "xgekmm_strided_batched", m, ps, qs, x, m * k, factors,
                          [p * q if fb else 0 for p, q in fs], z, m * l, batch, alpha, beta, y, m * l if y is not None else 0,
                          t1, t2, **ops)
    else:
        call = h.prepared("xgemkm" if mkm else "xgekmm", m, ps, qs, x, factors, z, alpha, beta, y, t1, t2, **ops)
    return dict(mm=case["mm"], call=call, z=z, keep=(h, x, factors, y, t1, t2), grad="")


def run(state):
    if "call" in state:
        error = state["call"]()
        if error != capi.SUCCESS:
            raise fastkron_amd.FastKronError(error, state["mm"])
        return state["z"]
    x, fs = state["x"], state["fs"]
    if not state["grad"]:
        if state["mm"] == "mkm":
            return fastkron_amd.gemkm(x, fs, state["alpha"], state["beta"], state["y"])
        return fastkron_amd.gekmm(fs, x, state["alpha"], state["beta"], state["y"])
    z = fastkron_amd.gemkm(x, fs) if state["mm"] == "mkm" else fastkron_amd.gekmm(fs, x)
    wanted = ([x] if x.requires_grad else []) + [f for f in fs if f.requires_grad]
    return [z.detach(), *torch.autograd.grad(z, wanted, state["gz"])]


def work(case):
    """Compulsory bytes: operands once, results once.  Operations: 2 per multiply-add of every step, once for the
    product and once more for the gradients of X's chain and of the factors where they are asked for."""
    nb, nx, nf, _ = _dims(case)
    fs, w, m = _shapes(case), _widths(case), case["m"]
    k, l = w[0], w[-1]
    fbytes = nf * sum(p * q for p, q in fs)
    elems = nx * m * k + nb * m * l * (2 if case["epilogue"] else 1) + fbytes
    muls = nb * m * sum(a * q for a, (_, q) in zip(w, reversed(fs)))
    flops = 2 * muls
    if case["grad"]:
        elems += nb * m * l                                             # the gradient of Z
        if case["grad"] in ("x", "all"):
            elems += nx * m * k
        if case["grad"] in ("factors", "all"):
            elems += fbytes
        flops += 2 * muls * (2 if case["grad"] != "x" else 1)
    return {"bytes": elems * (4 if case["dtype"] == "float32" else 8), "flops": flops}


def tolerance(case):
    """Four times the largest relative error seen against 64-bit (for float64: reordered 64-bit) sums over the listed
    and 200 drawn cases: 1.8e-7 and 6.7e-16 for products, 6.1e-6 and 2.6e-14 where factor gradients are among the
    outputs (sums of random signs over up to a million rows, which cancel)."""
    f32 = case["dtype"] == "float32"
    if case["grad"] in ("factors", "all"):
        return {"rel": 2.4e-5 if f32 else 1.1e-13}
    return {"rel": 7.2e-7 if f32 else 2.7e-15}

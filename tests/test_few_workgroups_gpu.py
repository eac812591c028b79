"""Problems with few tiles, which take other branches than large ones: several waves per tile of the two-factor KMM kernel
(9x9 ... 16x16, kernels/kmm16x2_mfma.hip) and the plain step with its loads ahead (kernels/generic_step.hip).  Against
the oracle with TOL of gpu_util (normwise 1e-5 / 1e-12; sums of at most 3 x 129 terms: u * 387 = 2.3e-5 only if every
rounding had the same sign, sqrt(387) * u = 1.2e-6 with random ones)."""
import numpy as np
import pytest

from oracle import kron_oracle as ko
from tests.gpu_util import TOL, make_case, normwise, oracle_answer, run_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fk():
    import fastkron_amd
    h = fastkron_amd.FastKron()
    yield h
    h.close()


def check(fk, mm, M, Ps, Qs, dt, seed, **kw):
    alpha, beta = kw.pop("alpha", 1.0), kw.pop("beta", 0.0)
    y_is_z = kw.pop("y_is_z", False)
    X, Fs, Y = make_case(mm, M, Ps, Qs, dt, seed=seed, with_y=beta != 0.0, **{k: v for k, v in kw.items() if k in ("batch", "opX", "opFs")})
    want = oracle_answer(mm, M, Ps, Qs, X, Fs, Y, alpha, beta, **kw)
    got, e = run_gpu(fk, mm, M, Ps, Qs, X, Fs, Y, alpha, beta, y_is_z=y_is_z, **kw)
    assert e == 0 and normwise(got, want) <= TOL[dt], (fk.last_plan(), M, Ps, Qs, kw)


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
@pytest.mark.parametrize("P", [9, 10, 13, 16])
@pytest.mark.parametrize("M", [2, 17, 64, 600, 4200, 8300])      # 4, 2 and 1 waves per tile, incomplete last tiles
def test_two_factors_with_few_tiles(fk, M, P, dt):
    check(fk, ko.KMM, M, [P, P], [P, P], dt, 1)
    if M <= 600:
        check(fk, ko.KMM, M, [P, P], [P, P], dt, 2, alpha=1.5, beta=0.5, batch=3)
        check(fk, ko.KMM, M, [P, P], [P, P], dt, 3, alpha=1.5, beta=0.5, y_is_z=True, opFs=ko.OP_T)
    assert any("_2_16x256" in k for _, _, k in fk.last_plan())


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
@pytest.mark.parametrize("P", [1, 2, 7, 8, 9, 16, 17, 31, 33, 129])
@pytest.mark.parametrize("Q", [1, 3, 5, 16, 17])
def test_plain_step(fk, P, Q, dt):
    plain = "gekmm_hip_gfx950_256_%s_generic_1" % ("f" if dt is np.float32 else "d")
    fk.set_options(fusion=False)
    try:
        for mm, M in [(ko.KMM, 5), (ko.KMM, 300), (ko.MKM, 7)]:
            check(fk, mm, M, [3, P], [3, Q], dt, 4, alpha=1.5, beta=0.5)
            check(fk, mm, M, [3, P], [3, Q], dt, 5, batch=2, opX=ko.OP_T)
        if P < 17 and Q < 16:
            check(fk, ko.KMM, 60000, [3, P], [3, Q], dt, 6)            # more than four workgroups per CU: the other loop
            assert any(k == plain for _, _, k in fk.last_plan()), fk.last_plan()
    finally:
        fk.set_options(fusion=True)


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
@pytest.mark.parametrize("M,P,Q", [(70000, 33, 16), (70000, 65, 9), (70000, 129, 17), (8, 260, 300), (70000, 16, 17), (3, 1000, 3)])
def test_plain_step_on_either_side_of_the_rule_for_loads_ahead(fk, M, P, Q, dt):
    """Rows of more than one staged piece of 32 with the loads ahead (from 256 workgroups on) and without; TOL as above, the
    sums have at most 1000 terms: sqrt(1000) * u = 1.9e-6."""
    fk.set_options(fusion=False)
    try:
        check(fk, ko.KMM, M, [P], [Q], dt, 7, alpha=1.5, beta=0.5)
        if M < 100:
            check(fk, ko.MKM, M, [P], [Q], dt, 8, batch=2)
    finally:
        fk.set_options(fusion=True)


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f", "d"])
@pytest.mark.parametrize("P,Q", [(12, 13), (16, 400), (33, 90), (64, 300), (65, 16), (128, 70), (129, 33), (200, 13), (256, 512)])
def test_padded_step_stages_its_factor_in_any_number_of_batches(fk, P, Q, dt):
    """Factors of one and of many batches of staged elements, the first tile's loads ahead of them and behind, fewer tiles than
    waves and more; sums of at most 256 terms, sqrt(256) * u = 1e-6."""
    for mm, M in [(ko.MKM, 3), (ko.KMM, 3), (ko.KMM, 40), (ko.KMM, 3000 if P * Q < 20000 else 300), (ko.MKM, 700 if P * Q < 20000 else 50)]:
        check(fk, mm, M, [P], [Q], dt, 9, alpha=1.5, beta=0.5)
        check(fk, mm, M, [P], [Q], dt, 10, batch=2, opX=ko.OP_T, opFs=ko.OP_T)

"""GPU solves whose steps take their inner products in the hops' epilogues, at the
forms these have: a wavefront per direction and a lane per site, workgroups
partly filled, two FP32 right-hand sides per lane (fields beyond 256 MiB),
more workgroups than one finishing pass sums, with and without the clover
term; plain FP64 and every inner precision.  Each RHS's FP64 true residual
through the oracle operator, and as many iterations as the oracle's BiCGStab
takes in FP64 (to one: the sums are taken in another order)."""
import numpy as np
import pytest

from oracle import oracle
from qcu_mrhs_amd import api, fields

pytestmark = pytest.mark.gpu

D, S, H, B = 2, 1, 0, 4
KAPPA, CSW, TOL = 0.12, 1.1, 1e-10


def _solve(L, Nc, R, inner, clover, distinct, seed):
    gauge = fields.gauge_field(L, Nc, seed, kind="smooth", eps=0.6)
    b = fields.gaussian_sources(L, Nc, distinct, seed + 1)
    n = b.shape[1]
    api.initGridSize(L, Nc, R, D, inner)
    d_g = api.DeviceArray.from_complex(gauge.reshape(-1))
    api.loadQcuGauge(d_g, D)
    api.getDslash(api.DSLASH_CLOVER if clover else 0, 1.0 / (2 * KAPPA) - 4.0)
    if clover:
        api.set_clover_coefficient(CSW)
    api.set_solver_options(inner, 0.0, False)
    d_b = [api.DeviceArray.from_complex(v) for v in b]
    xs = [api.DeviceArray(n * 16) for _ in range(R)]
    for r in range(R):
        api.pushBackFermions(xs[r], d_b[r % distinct])
    try:
        info = api.qcuInvertEx(500, TOL)
        x = np.stack([xs[r].complex(n) for r in range(R - distinct, R)])
    finally:
        api.finalizeQcu()
    bm = fields.to_mrhs(np.stack([b[r % distinct] for r in range(R - distinct, R)]), Nc)
    xm = fields.to_mrhs(x, Nc)
    if clover:
        ax = oracle.clover_mat(xm, gauge, oracle.clover(gauge, L, Nc, CSW, KAPPA), L, Nc, distinct, KAPPA)
    else:
        ax = oracle.mat(xm, gauge, L, Nc, distinct, KAPPA)
    tr = oracle.norm(bm - ax, distinct) / oracle.norm(bm, distinct)
    print("case dots", L, Nc, R, inner, clover, info["iterations"], tr.max(), flush=True)
    assert info["converged"]
    assert tr.max() <= TOL * 1.05
    return info, gauge, b


@pytest.mark.parametrize("inner", [D, S, H, B])
@pytest.mark.parametrize("L,Nc,R,clover", [((4, 4, 4, 4), 3, 1, False), ((4, 2, 6, 4), 3, 5, False), ((6, 4, 4, 4), 4, 16, False),
                                           ((4, 4, 2, 6), 2, 37, False), ((4, 2, 4, 4), 3, 100, False), ((4, 2, 4, 6), 4, 33, False),
                                           ((4, 4, 2, 4), 3, 36, True), ((2, 4, 4, 2), 4, 70, True)])
def test_solves(L, Nc, R, clover, inner):
    _solve(L, Nc, R, inner, clover, R, 20 + R)


@pytest.mark.parametrize("Nc,R", [(3, 40), (2, 60)])
def test_two_rhs_per_lane(Nc, R):
    _solve((16, 16, 16, 16), Nc, R, S, False, 2, 50 + Nc)


@pytest.mark.parametrize("inner", [D, H])
def test_more_rows_than_one_pass(inner):
    _solve((16, 8, 12, 12), 2, 128, inner, False, 2, 70)


@pytest.mark.parametrize("L,R", [((4, 4, 4, 8), 4), ((4, 4, 4, 4), 36)])
def test_plain_double_iterations(L, R):
    info, gauge, b = _solve(L, 3, R, D, False, R, 90)
    iters = oracle.bicgstab(fields.to_mrhs(b, 3), gauge, L, 3, R, KAPPA, 500, TOL)[2]
    print("  oracle iterations", iters, flush=True)
    assert abs(info["iterations"] - iters) <= 1

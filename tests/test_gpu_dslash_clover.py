"""GPU parity of the hops that apply the clover blocks in their epilogue, at
RHS counts and lattices where the work does not divide evenly (a workgroup of
one site, several, a last one partly filled; two right-hand sides per lane for
FP32 fields beyond 256 MiB), both forms (A x + coef D in through mat_Qcu,
A^{-1} (coef D in + b) and the fused residual and omega through a solve),
against the FP64 oracle."""
import numpy as np
import pytest

from oracle import oracle
from qcu_mrhs_amd import api, fields

pytestmark = pytest.mark.gpu

D, S, H, B = 2, 1, 0, 4
MASS, CSW = -0.2, 1.3
KAPPA = 1.0 / (2 * (4 + MASS))


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def _setup(L, Nc, R, user, prec, seed):
    gauge = fields.gauge_field(L, Nc, seed, kind="smooth", eps=0.5)
    api.initGridSize(L, Nc, R, user, prec)
    d_g = api.DeviceArray.from_complex(gauge.reshape(-1))
    api.loadQcuGauge(d_g, D)
    api.getDslash(api.DSLASH_CLOVER, MASS)
    api.set_clover_coefficient(CSW)
    return gauge, oracle.clover(gauge, L, Nc, CSW, KAPPA), d_g


def _mat(L, Nc, R, prec, tol, distinct, seed):
    """R sources made of `distinct` ones in turn."""
    gauge, c, d_g = _setup(L, Nc, R, prec, prec, seed)
    b = fields.gaussian_sources(L, Nc, distinct, seed + 1)
    n = b.shape[1]
    stored = np.stack([api.from_storage(api.to_storage(v, prec), prec) for v in b])
    ins = [api.DeviceArray.from_complex(v, prec) for v in b]
    try:
        for dagger in (0, 1):
            outs = [api.DeviceArray(api.storage_bytes(n, prec)) for _ in range(R)]
            for r in range(R):
                api.pushBackFermions(outs[r], ins[r % distinct])
            api.mat_Qcu(dagger)
            ref = oracle.clover_mat(fields.to_mrhs(stored, Nc), gauge, c, L, Nc, distinct, KAPPA, dagger)
            ref = ref.reshape(-1, distinct)
            for r in range(R):
                got = fields.to_mrhs(outs[r].complex(n, prec)[None], Nc).reshape(-1)
                err = _rel(got, ref[:, r % distinct])
                assert err < tol, (r, err)
            print("case clover hop", L, Nc, R, prec, dagger, err, flush=True)
    finally:
        api.finalizeQcu()


@pytest.mark.parametrize("prec,tol", [(D, 1e-13), (S, 2e-6)])
@pytest.mark.parametrize("L,Nc,R", [((4, 2, 6, 4), 3, 36), ((2, 4, 2, 6), 2, 33), ((4, 2, 2, 4), 4, 40),
                                    ((2, 2, 4, 2), 3, 65), ((2, 2, 2, 4), 3, 127), ((2, 4, 2, 2), 2, 128)])
def test_operator(L, Nc, R, prec, tol):
    _mat(L, Nc, R, prec, tol, R, 40 + R)


def test_operator_two_per_lane():
    _mat((16, 16, 16, 16), 3, 40, S, 2e-6, 3, 77)


@pytest.mark.parametrize("inner", [D, S, H, B])
@pytest.mark.parametrize("L,Nc,R", [((4, 4, 2, 4), 3, 36), ((2, 4, 4, 2), 2, 127)])
def test_solve(L, Nc, R, inner):
    tol = 1e-10
    gauge, c, d_g = _setup(L, Nc, R, D, inner, 60 + R)
    api.set_solver_options(inner, 0.0, False)
    b = fields.gaussian_sources(L, Nc, R, 61)
    n = b.shape[1]
    d_b = [api.DeviceArray.from_complex(v) for v in b]
    xs = [api.DeviceArray(n * 16) for _ in range(R)]
    for r in range(R):
        api.pushBackFermions(xs[r], d_b[r])
    info = api.qcuInvertEx(5000, tol)
    x = np.stack([v.complex(n) for v in xs])
    api.finalizeQcu()
    bm = fields.to_mrhs(b, Nc)
    res = bm - oracle.clover_mat(fields.to_mrhs(x, Nc), gauge, c, L, Nc, R, KAPPA)
    tr = oracle.norm(res, R) / oracle.norm(bm, R)
    print("case clover solve", L, Nc, R, inner, info["iterations"], tr.max(), flush=True)
    assert info["converged"]
    assert tr.max() <= tol * 1.05 and info["true_rel_residual"] <= tol * 1.05

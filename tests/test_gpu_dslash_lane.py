"""GPU parity of the lane-per-(site, RHS) hopping kernel at the edges of its
launch shapes (eight hops per lane, and the directions split over four
wavefronts on small lattices): right-hand sides that fill no wavefront, one lane per site and
more lanes than a wavefront per site, sites that do not fill the last
workgroup, lattices of a single workgroup, and the form with two right-hand
sides per lane (fields beyond 256 MiB in FP32); xpay and the dagger on the
way.  Tolerances are those of the storage types used for every variant."""
import numpy as np
import pytest

from oracle import oracle
from qcu_mrhs_amd import api, fields

pytestmark = pytest.mark.gpu

D, S, H, B = 2, 1, 0, 4
TOL = {D: 1e-13, S: 2e-7, H: 2e-3, B: 1.5e-2}


@pytest.fixture(autouse=True)
def _reset_tune():
    yield
    api.dslash_tune("auto")


def _check(L, Nc, R, prec, parity, dagger, xpay, seed):
    gauge = fields.gauge_field(L, Nc, seed, kind="smooth", eps=0.6)
    g = fields.rng(seed + 1)
    n = fields.half_volume(L) * 4 * Nc * R
    vec = [g.standard_normal(n) + 1j * g.standard_normal(n) for _ in range(2)]
    # inputs as stored, so that only the kernel's arithmetic is compared
    st = lambda a: api.from_storage(api.to_storage(a, prec), prec)  # noqa: E731
    inp, x, gs = st(vec[0]), st(vec[1]), st(gauge.reshape(-1)).reshape(gauge.shape)
    d_in, d_x = api.DeviceArray.from_complex(inp, prec), api.DeviceArray.from_complex(x, prec)
    d_g = api.DeviceArray.from_complex(gauge.reshape(-1), prec)
    d_out = api.DeviceArray(api.storage_bytes(n, prec))
    coef = -0.7 if xpay else 1.0
    api.dslash_tune("lane_rhs")
    api.dslash_mrhs(d_out, d_in, d_g, L, Nc, R, parity, dagger, precision=prec, xpay=d_x if xpay else None, coef=coef)
    got = d_out.complex(n, prec)
    ref = coef * oracle.dslash(inp, gs, L, Nc, R, parity, dagger)
    if xpay:
        ref = x + ref
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    print("case lane", L, Nc, R, prec, parity, dagger, xpay, err, flush=True)
    assert err < TOL[prec]


@pytest.mark.parametrize("prec", [D, S, H, B])
@pytest.mark.parametrize("L,Nc,R", [((2, 2, 2, 2), 3, 1), ((4, 2, 6, 4), 3, 5), ((6, 4, 2, 10), 2, 17),
                                    ((4, 6, 4, 6), 4, 33), ((6, 6, 4, 4), 3, 70), ((4, 4, 4, 2), 4, 130),
                                    ((14, 6, 10, 6), 3, 3), ((8, 12, 8, 16), 3, 12), ((12, 6, 6, 8), 4, 1),
                                    ((4, 4, 4, 8), 2, 64), ((18, 16, 12, 22), 3, 5), ((24, 14, 18, 24), 2, 1)])
def test_lane_kernel_edges(prec, L, Nc, R):
    for k, (parity, dagger, xpay) in enumerate([(0, 0, False), (1, 1, True)]):
        _check(L, Nc, R, prec, parity, dagger, xpay, 900 + 7 * R + k)


@pytest.mark.parametrize("Nc,R,dagger", [(3, 28, 0), (2, 46, 1)])
def test_two_rhs_per_lane(Nc, R, dagger):
    _check((16, 16, 16, 32), Nc, R, S, 1, dagger, True, 950 + Nc)


@pytest.mark.parametrize("inner", [H, B, S])
@pytest.mark.parametrize("L,Nc,R", [((8, 8, 8, 8), 3, 16), ((12, 6, 10, 4), 2, 24), ((8, 6, 4, 20), 4, 20)])
def test_mixed_solve_on_lane_kernels(inner, L, Nc, R):
    """A reliable-update solve whose hops, fused omega (16 bits) and fused FP64
    residual run on the lane kernel, with sites that do not fill the last
    workgroup: the FP64 true residual through the oracle operator."""
    kappa, tol = 0.12, 1e-10
    gauge = fields.gauge_field(L, Nc, 970 + Nc, kind="smooth", eps=0.8)
    b = fields.gaussian_sources(L, Nc, R, 980 + R)
    api.initGridSize(L, Nc, R, D, inner)
    d_g = api.DeviceArray.from_complex(gauge.reshape(-1))
    api.loadQcuGauge(d_g, D)
    api.getDslash(0, 1.0 / (2 * kappa) - 4.0)
    bs = [api.DeviceArray.from_complex(b[r]) for r in range(R)]
    xs = [api.DeviceArray(b[r].nbytes) for r in range(R)]
    for r in range(R):
        api.pushBackFermions(xs[r], bs[r])
    info = api.qcuInvertEx(500, tol)
    x = np.stack([xs[r].complex(b[r].size) for r in range(R)])
    api.finalizeQcu()
    bm = fields.to_mrhs(b, Nc)
    res = bm - oracle.mat(fields.to_mrhs(x, Nc), gauge, L, Nc, R, kappa)
    rel = (oracle.norm(res, R) / oracle.norm(bm, R)).max()
    print("case lane solve", L, Nc, R, inner, info["iterations"], rel, flush=True)
    assert info["converged"] and info["reliable_updates"] >= 1
    assert rel <= 1.01 * tol and abs(info["true_rel_residual"] - rel) <= 0.01 * tol


@pytest.mark.parametrize("L,Nc,R,inner", [((8, 8, 8, 8), 3, 4, S), ((16, 12, 16, 20), 2, 24, S), ((12, 10, 14, 6), 4, 7, S),
                                          ((8, 6, 4, 4), 3, 16, H), ((8, 6, 4, 4), 3, 16, B)])
def test_operator_on_wider_vectors_keeps_its_rounding(L, Nc, R, inner):
    """start_dslash on double-precision vectors in a lower precision sums the
    hops in the order of the wave-per-site (16 bits: matrix-core) kernel: the
    same bits as that kernel chosen explicitly."""
    gauge = fields.gauge_field(L, Nc, 990 + Nc, kind="smooth", eps=0.8)
    half = fields.half_volume(L) * 4 * Nc
    g = fields.rng(991)
    b = g.standard_normal((R, half)) + 1j * g.standard_normal((R, half))
    api.initGridSize(L, Nc, R, D, inner)
    d_g = api.DeviceArray.from_complex(gauge.reshape(-1))
    api.loadQcuGauge(d_g, D)
    api.getDslash(0, 0.1)
    bs = [api.DeviceArray.from_complex(v) for v in b]
    got = []
    for variant in ("auto", "wave" if inner == S else "mfma"):
        xs = [api.DeviceArray(16 * half) for _ in range(R)]
        api.dslash_tune(variant)
        for r in range(R):
            api.pushBackFermions(xs[r], bs[r])
        api.start_dslash(1, 0)
        got.append(np.stack([x.complex(half) for x in xs]))
    api.finalizeQcu()
    print("case lane order", L, Nc, R, inner, flush=True)
    np.testing.assert_array_equal(got[0], got[1])

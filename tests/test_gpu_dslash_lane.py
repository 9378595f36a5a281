"""GPU parity of the lane-per-(site, RHS) hopping kernel at the edges of its
launch shape: right-hand sides that fill no wavefront, one lane per site and
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
                                    ((14, 6, 10, 6), 3, 3), ((8, 12, 8, 16), 3, 12), ((12, 6, 6, 8), 4, 1)])
def test_lane_kernel_edges(prec, L, Nc, R):
    for k, (parity, dagger, xpay) in enumerate([(0, 0, False), (1, 1, True)]):
        _check(L, Nc, R, prec, parity, dagger, xpay, 900 + 7 * R + k)


@pytest.mark.parametrize("Nc,R,dagger", [(3, 28, 0), (2, 46, 1)])
def test_two_rhs_per_lane(Nc, R, dagger):
    _check((16, 16, 16, 32), Nc, R, S, 1, dagger, True, 950 + Nc)

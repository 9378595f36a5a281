"""The hop for few right-hand sides on larger lattices, where variant 1 runs a
kernel without the links in LDS: results against the FP64 oracle on both
sides of the rule, and a call with fewer right-hand sides takes no longer than
one with twice as many (with the links of all its sites in LDS it did, by
half)."""
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


def _arrays(L, Nc, R, prec, seed):
    g = fields.rng(seed)
    n = fields.half_volume(L) * 4 * Nc * R
    st = lambda a: api.from_storage(api.to_storage(a, prec), prec)  # noqa: E731
    inp, x = (st(g.standard_normal(n) + 1j * g.standard_normal(n)) for _ in range(2))
    gauge = st(fields.gauge_field(L, Nc, seed + 1, kind="smooth", eps=0.6).reshape(-1))
    return inp, x, gauge


@pytest.mark.parametrize("prec", [D, S, H, B])
@pytest.mark.parametrize("variant", ["lane_rhs", "auto"])
@pytest.mark.parametrize("L,Nc,R", [((16, 16, 16, 24), 3, 1), ((16, 16, 16, 32), 2, 1), ((24, 14, 18, 24), 3, 2),
                                    ((16, 16, 16, 24), 4, 3), ((14, 14, 12, 18), 2, 5), ((12, 12, 12, 14), 3, 7)])
def test_matches_oracle(L, Nc, R, variant, prec):
    inp, x, gauge = _arrays(L, Nc, R, prec, 1500 + R)
    d_in, d_x, d_g = (api.DeviceArray.from_complex(v, prec) for v in (inp, x, gauge))
    d_out = api.DeviceArray(api.storage_bytes(inp.size, prec))
    api.dslash_tune(variant)
    for dagger, xpay in ((0, False), (1, True)):
        coef = -0.7 if xpay else 1.0
        api.dslash_mrhs(d_out, d_in, d_g, L, Nc, R, 1 - dagger, dagger, precision=prec, xpay=d_x if xpay else None, coef=coef)
        ref = coef * oracle.dslash(inp, gauge.reshape(4, 2, -1, Nc, Nc), L, Nc, R, 1 - dagger, dagger)
        if xpay:
            ref = x + ref
        err = np.linalg.norm(d_out.complex(inp.size, prec) - ref) / np.linalg.norm(ref)
        print("case few rhs", L, Nc, R, variant, prec, dagger, err, flush=True)
        assert err < TOL[prec]


@pytest.mark.parametrize("prec,Nc,R", [(S, 3, 1), (D, 3, 1), (H, 3, 1), (B, 4, 1), (S, 4, 2)])
def test_fewer_rhs_take_no_longer(prec, Nc, R):
    L = (24, 24, 24, 24)
    n = fields.half_volume(L) * 4 * Nc * 2 * R
    one = np.ones(1 << 16, dtype=np.complex128)
    full = lambda count: api.DeviceArray.from_complex(np.resize(one, count), prec)  # noqa: E731
    d_in, d_g = full(n), full(fields.half_volume(L) * 8 * Nc * Nc)
    d_out = api.DeviceArray(api.storage_bytes(n, prec))
    api.dslash_tune("lane_rhs")

    def us(r):
        run = lambda: api.dslash_mrhs(d_out, d_in, d_g, L, Nc, r, 0, 0, precision=prec)  # noqa: E731
        run()
        best = 1e30
        for _ in range(4):
            api.check(api.lib().qcuTimerStart())
            for _ in range(10):
                run()
            best = min(best, api.lib().qcuTimerStopMs() * 100)
        return best

    fewer, more = us(R), us(2 * R)
    print("case few rhs time", prec, Nc, R, fewer, more, flush=True)
    assert fewer < 1.05 * more

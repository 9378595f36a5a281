"""GPU parity of the clover build and block inverse where their lanes do not
divide evenly: site counts that leave a workgroup or wavefront partly filled,
extents of 2 (both neighbours of a site are the same one), every Nc, and
coefficients at which the off-diagonal entries lead, so that rows are
interchanged.  The term against the FP64 oracle; the inverse against LAPACK on
the term, within the bound of an elimination with partial pivoting
(16 n eps times the condition number of the block)."""
import numpy as np
import pytest

from oracle import oracle
from qcu_mrhs_amd import api, fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("csw", [1.1, 9.0])
@pytest.mark.parametrize("L,Nc", [((2, 2, 2, 2), 3), ((6, 2, 2, 4), 3), ((2, 6, 10, 2), 3), ((4, 6, 2, 4), 2),
                                  ((2, 4, 2, 6), 4), ((2, 2, 6, 2), 8)])
def test_ragged_sites_and_pivots(L, Nc, csw):
    kappa, n = 0.125, 2 * Nc
    print("case clover build", L, Nc, csw, flush=True)
    gauge = fields.gauge_field(L, Nc, 800 + Nc, kind="haar")
    ref = oracle.clover(gauge, L, Nc, csw, kappa)
    d_g = api.DeviceArray.from_complex(gauge.reshape(-1))
    d_c, d_i = api.DeviceArray(ref.size * 16), api.DeviceArray(ref.size * 16)
    api.clover_build(d_c, d_i, d_g, L, Nc, csw, kappa)
    got = d_c.complex(ref.size).reshape(ref.shape)
    assert np.abs(got - ref).max() < 1e-14 * max(1.0, csw)
    blocks, inv = got.reshape(-1, n, n), d_i.complex(ref.size).reshape(-1, n, n)
    exact = np.linalg.inv(blocks)
    err = np.linalg.norm(inv - exact, axis=(1, 2)) / np.linalg.norm(exact, axis=(1, 2))
    bound = 16 * n * np.finfo(np.float64).eps * np.linalg.cond(blocks)
    print("  inverse error / bound", (err / bound).max(), flush=True)
    assert (err < bound).all()
    # in place
    api.clover_build(d_c, d_c, d_g, L, Nc, csw, kappa)
    assert np.array_equal(d_c.complex(ref.size).reshape(-1, n, n), inv)

"""GPU parity of the learned preconditioner's FP32 matrix-core kernels at the
edges of their chunks: columns that do and do not fill the tiles of 16, one
and several chunks of right-hand sides, a last chunk with missing ones, every
Nc, lattices with fewer sites than workgroups.  Forward and gradients against
the FP64 oracle network within the FP32 tolerances of the other shapes."""
import numpy as np
import pytest

from oracle import lgnn as olgnn
from qcu_mrhs_amd import api, fields, lgnn

pytestmark = pytest.mark.gpu

RTOL_FWD, RTOL_GRAD, KAPPA = 1e-5, 1e-4, 0.13


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("L,Nc,R", [((2, 2, 2, 2), 3, 1), ((2, 4, 2, 4), 3, 21), ((2, 2, 4, 2), 3, 22), ((4, 2, 2, 6), 3, 16),
                                    ((2, 4, 2, 2), 2, 32), ((2, 2, 2, 4), 2, 33), ((2, 2, 4, 4), 4, 17),
                                    ((2, 4, 2, 2), 8, 9), ((6, 4, 4, 10), 3, 5), ((2, 2, 2, 2), 4, 50)])
def test_forward_and_gradients_at_chunk_edges(L, Nc, R):
    gauge = fields.gauge_field(L, Nc, 61 + Nc + R, kind="haar")
    api.initGridSize(L, Nc, R, 2, 2)
    d_g = api.DeviceArray.from_complex(gauge.reshape(-1))
    api.loadQcuGauge(d_g, 2)
    api.getDslash(0, 1.0 / (2 * KAPPA) - 4.0)
    g = np.random.default_rng(62 + R)
    shape = (fields.half_volume(L), 4, Nc, R)
    r, e = ((g.standard_normal(shape) + 1j * g.standard_normal(shape)).astype(np.complex64).astype(np.complex128)
            for _ in range(2))
    net = olgnn.Net.random(3, 63, scale=0.3)
    lgnn.set_weights(net.W1[:, 0].copy(), net.W2[0].copy())
    tr = olgnn.Transport(gauge, L, Nc)
    d_r, d_e = (api.DeviceArray.from_complex(v.reshape(-1), 1) for v in (r, e))
    ref, _ = net.forward(tr, r, L, Nc, R)
    for prec in (1, 2):
        d_in, d_out = api.DeviceArray.from_complex(r.reshape(-1), prec), api.DeviceArray(api.storage_bytes(r.size, prec))
        lgnn.apply(d_out, d_in, prec)
        err = _rel(d_out.complex(r.size, prec), ref.reshape(-1))
        print("case stencil", L, Nc, R, prec, err, flush=True)
        assert err < RTOL_FWD
    loss, g1, g2 = lgnn.loss_grad(d_r, d_e, 3)
    ref_loss, ref_g1, ref_g2 = net.loss_and_grad(tr, r, e, L, Nc, R)
    print("  loss", loss, ref_loss, "gradients", _rel(g1, ref_g1[:, 0]), _rel(g2, ref_g2[0]), flush=True)
    api.finalizeQcu()
    assert abs(loss - ref_loss) <= RTOL_FWD * abs(ref_loss)
    assert _rel(g1, ref_g1[:, 0]) < RTOL_GRAD and _rel(g2, ref_g2[0]) < RTOL_GRAD

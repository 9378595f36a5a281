"""FP32 application of the learned preconditioner where a workgroup of the
matrix-core mixing takes one to four sites: against the FP64 oracle network on
lattices whose last workgroup is partly filled, and a small lattice that pays
for its own sites (with one site per workgroup each workgroup fetched the
stencil anew, and 8^4 took more than half the time of a lattice 3.7 times its
size)."""
import time

import numpy as np
import pytest

from oracle import lgnn as olgnn
from qcu_mrhs_amd import api, fields, lgnn

pytestmark = pytest.mark.gpu

KAPPA = 0.13


def _network(L, Nc, R, seed):
    gauge = fields.gauge_field(L, Nc, seed, kind="haar")
    api.initGridSize(L, Nc, R, 2, 2)
    d_g = api.DeviceArray.from_complex(gauge.reshape(-1))
    api.loadQcuGauge(d_g, 2)
    api.getDslash(0, 1.0 / (2 * KAPPA) - 4.0)
    net = olgnn.Net.random(3, seed + 1, scale=0.3)
    lgnn.set_weights(net.W1[:, 0].copy(), net.W2[0].copy())
    g = fields.rng(seed + 2)
    n = fields.half_volume(L) * 4 * Nc * R
    r = (g.standard_normal(n) + 1j * g.standard_normal(n)).astype(np.complex64)
    return gauge, net, r, api.DeviceArray.from_complex(r, 1), api.DeviceArray(8 * n)


@pytest.mark.parametrize("L,Nc,R", [((6, 6, 6, 4), 3, 2), ((6, 6, 6, 10), 3, 2), ((6, 10, 6, 10), 2, 5), ((8, 6, 8, 10), 4, 1),
                                    ((6, 10, 6, 14), 3, 1)])
def test_matches_oracle(L, Nc, R):
    gauge, net, r, d_in, d_out = _network(L, Nc, R, 2000)
    try:
        lgnn.apply(d_out, d_in, 1)
        got = d_out.complex(r.size, 1)
    finally:
        api.finalizeQcu()
    ref, _ = net.forward(olgnn.Transport(gauge, L, Nc), r.astype(np.complex128).reshape(-1, 4, Nc, R), L, Nc, R)
    err = np.linalg.norm(got - ref.reshape(-1)) / np.linalg.norm(ref)
    print("case lgnn sites", L, Nc, R, err, flush=True)
    assert err < 1e-5


def test_small_lattice_pays_for_its_own_sites():
    us = []
    for L in ((8, 8, 8, 8), (6, 10, 14, 18)):
        _, _, _, d_in, d_out = _network(L, 3, 32, 2010)
        try:
            best = 1e30
            for k in range(40):
                api.synchronize()
                t = time.perf_counter()
                lgnn.apply(d_out, d_in, 1)
                best = min(best, time.perf_counter() - t)
        finally:
            api.finalizeQcu()
        us.append(best * 1e6)
    print("case lgnn sites time", us, flush=True)
    assert us[0] < 0.5 * us[1]

"""The stateless hop on two GPUs of one process, same lattice and precision:
what the library keeps per lattice lies in each GPU's own memory."""
import numpy as np
import pytest
import torch

from oracle import oracle
from qcu_mrhs_amd import api, fields

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two GPUs")]


@pytest.mark.parametrize("prec,tol", [(2, 1e-13), (1, 2e-7), (0, 2e-3)])
def test_each_device_has_its_own_tables(prec, tol):
    L, Nc, R = (4, 6, 4, 10), 3, 12
    gauge = fields.gauge_field(L, Nc, 2200, kind="smooth", eps=0.6)
    g = fields.rng(2201)
    n = fields.half_volume(L) * 4 * Nc * R
    inp = g.standard_normal(n) + 1j * g.standard_normal(n)
    ref = oracle.dslash(inp, gauge, L, Nc, R, 1, 0)
    try:
        for dev in (0, 1, 0):
            torch.cuda.set_device(dev)
            torch.cuda.synchronize()
            d_in, d_g = api.DeviceArray.from_complex(inp, prec), api.DeviceArray.from_complex(gauge.reshape(-1), prec)
            d_out = api.DeviceArray(api.storage_bytes(n, prec))
            api.dslash_mrhs(d_out, d_in, d_g, L, Nc, R, 1, 0, precision=prec)
            err = np.linalg.norm(d_out.complex(n, prec) - ref) / np.linalg.norm(ref)
            print("case two devices", dev, prec, err, flush=True)
            assert err < tol
    finally:
        torch.cuda.set_device(0)

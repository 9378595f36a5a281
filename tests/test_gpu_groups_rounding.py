"""Rounding of a batch's 16-bit hops on the lane kernels: FP32 from the stored
values on, so that each stored component is the exact result rounded once, as
in the batches' wave-per-site kernel."""
import numpy as np
import pytest

import internals as it
from oracle import oracle
from qcu_mrhs_amd import api, fields
from test_gpu_dslash_rounding import _half_ulp

pytestmark = pytest.mark.gpu

H, B = 0, 4


@pytest.mark.parametrize("scale_in,scale_g", [(1.0, 1.0), (2.5e4, 0.03)])
@pytest.mark.parametrize("prec", [H, B])
@pytest.mark.parametrize("L,Nc,sizes", [((4, 4, 6, 6), 3, (5, 12)), ((4, 4, 4, 6), 4, (33, 1)), ((6, 4, 4, 4), 2, (128, 3))])
def test_batch_hop_rounds_once(L, Nc, sizes, prec, scale_in, scale_g):
    n, Rt, g = fields.half_volume(L) * 4 * Nc, sum(sizes), fields.rng(1800)
    st = lambda a: api.from_storage(api.to_storage(a, prec), prec)  # noqa: E731
    inp, x = (st(scale_in * np.clip(g.standard_normal((n * Rt, 2)), -1.5, 1.5) @ [1, 1j]) for _ in range(2))
    gauge = st(scale_g * fields.gauge_field(L, Nc, 1801, kind="haar").reshape(-1))
    d_in, d_x, d_g = (api.DeviceArray.from_complex(v, prec) for v in (inp, x, gauge))
    d_out = api.DeviceArray(api.storage_bytes(n * Rt, prec))
    tab, rows = it.groups(L, Nc, sizes), it.SegRows()
    a = it.args(L, Nc, 0, prec, out=d_out.ptr, inp=d_in.ptr, gauge=d_g.ptr, xpay=d_x.ptr)
    a.coef = -0.75
    assert it.call("dslash_dots_rows", a.g, Nc, prec, tab, rows)
    d_part = api.DeviceArray(8 * rows.total)
    for dots in (False, True):
        if dots:
            assert it.call("launch_dslash_lane_dots_groups", a, it.OMEGA, None, tab, rows, d_part.ptr, 2, 2, None) == 0
        else:
            assert it.call("launch_dslash_lane_groups", a, tab, 2, 2, None) == 0
        api.synchronize()
        out = d_out.complex(n * Rt, prec)
        for k, R in enumerate(sizes):
            own = slice(n * tab.base[k], n * (tab.base[k] + R))
            ref = (x[own] - 0.75 * oracle.dslash(inp[own], gauge.reshape(4, 2, -1, Nc, Nc), L, Nc, R, 1, 0)).view(np.float64)
            assert np.abs(ref).max() < 6e4
            # FP32: 8 hops of 4 Nc products, each sum at most about 10 times the largest result
            slack = 16 * Nc * 2.0 ** -24 * 10 * np.abs(ref).max()
            err = np.abs(out[own].view(np.float64) - ref) / (_half_ulp(np.abs(ref) + slack, prec) + slack)
            print("case batch rounding", L, Nc, R, prec, scale_in, dots, err.max(), flush=True)
            assert (err <= 1).all()

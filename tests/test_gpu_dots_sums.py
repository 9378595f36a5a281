"""The inner products that the hops' epilogues form for a BiCGStab step are
sums in FP64 of products of the stored values, from the first product on, for
every storage type: the rows of partial sums that the kernels leave, added up,
against the same sums in numpy.  Forms with a lane per site, a wavefront per
direction, clover blocks, and the batches' one."""
import numpy as np
import pytest

import internals as it
from qcu_mrhs_amd import api, fields

pytestmark = pytest.mark.gpu

D, S, H, B = 2, 1, 0, 4
CSW, KAPPA = 1.2, 0.12


def _setup(L, Nc, count, prec, seed):
    g = fields.rng(seed)
    st = lambda a: api.from_storage(api.to_storage(a, prec), prec)  # noqa: E731
    vecs = [st(g.standard_normal(count) + 1j * g.standard_normal(count)) for _ in range(3)]  # in, x, r0
    gauge = fields.gauge_field(L, Nc, seed + 1, kind="smooth", eps=0.6)
    return vecs, [api.DeviceArray.from_complex(v, prec) for v in vecs], gauge, api.DeviceArray.from_complex(gauge.reshape(-1), prec)


def _compare(kind, sums, out, x, r0, R, n, what):
    """sums [R][4] against numpy's; n terms of two products each"""
    t, s, r = (v.reshape(n, R) for v in (out, x, r0))
    pairs = [(r, t)] if kind == it.ALPHA else [(t, s), (t, t)]
    for k, (a, b) in enumerate(pairs):
        p = (a.conj() * b)
        bound = 2 * n * 2.0 ** -53 * (np.abs(a.real * b.real) + np.abs(a.imag * b.imag) + np.abs(a.real * b.imag) + np.abs(a.imag * b.real)).sum(0)
        got = sums[:, 0] + 1j * sums[:, 1] if k == 0 else sums[:, 2]
        err = np.abs(got - (p.sum(0) if k == 0 else p.real.sum(0)))
        print("case dots sums", *what, kind, k, (err / bound).max(), flush=True)
        assert (err <= bound).all()


@pytest.mark.parametrize("prec", [D, S, H, B])
@pytest.mark.parametrize("L,Nc,R,clover", [((4, 4, 4, 4), 3, 4, False), ((4, 4, 6, 4), 2, 36, False), ((4, 2, 4, 6), 4, 33, False),
                                           ((4, 4, 2, 4), 3, 36, True), ((2, 4, 4, 2), 4, 70, True)])
def test_solver_forms(L, Nc, R, clover, prec):
    n = fields.half_volume(L) * 4 * Nc
    (inp, x, r0), (d_in, d_x, d_r0), gauge, d_g = _setup(L, Nc, n * R, prec, 1600 + R)
    d_out = api.DeviceArray(api.storage_bytes(n * R, prec))
    a = it.args(L, Nc, R, prec, 5, out=d_out.ptr, inp=d_in.ptr, gauge=d_g.ptr, xpay=d_x.ptr)
    a.coef = -KAPPA * KAPPA
    if clover:
        d_c = api.DeviceArray(2 * fields.half_volume(L) * 8 * Nc * Nc * 16)
        api.clover_build(d_c, None, api.DeviceArray.from_complex(gauge.reshape(-1)), L, Nc, CSW, KAPPA)
        d_b = api.DeviceArray.from_complex(d_c.complex(d_c.nbytes // 16)[d_c.nbytes // 32:], D if prec == D else S)
        a.clover, a.clover_in, a.xpay = d_b.ptr, d_x.ptr, None
    cap = it.call("dslash_dots_partials", a.g, Nc, R, prec)
    d_part, d_st = api.DeviceArray(8 * cap), api.DeviceArray(16 * it.NUM_SLOTS * R)
    for kind in (it.ALPHA, it.OMEGA):
        d_part.zero()
        d_st.upload(np.ones(it.NUM_SLOTS * R, dtype=np.complex128))
        assert it.call("launch_dslash_dots", a, kind, d_r0.ptr, d_part.ptr, cap, d_st.ptr, None) == 0
        api.synchronize()
        sums = d_part.download(np.float64).reshape(-1, R, 4).sum(0)
        _compare(kind, sums, d_out.complex(n * R, prec), x, r0, R, n, (L, Nc, R, prec, clover))


@pytest.mark.parametrize("prec", [S, H, B])
@pytest.mark.parametrize("L,Nc,sizes", [((4, 4, 6, 6), 3, (5, 12)), ((4, 4, 4, 6), 4, (33, 1)), ((6, 4, 4, 4), 2, (128, 3))])
def test_batch_form(L, Nc, sizes, prec):
    n, Rt = fields.half_volume(L) * 4 * Nc, sum(sizes)
    (inp, x, r0), (d_in, d_x, d_r0), gauge, d_g = _setup(L, Nc, n * Rt, prec, 1700 + Rt)
    d_out = api.DeviceArray(api.storage_bytes(n * Rt, prec))
    a = it.args(L, Nc, 0, prec, out=d_out.ptr, inp=d_in.ptr, gauge=d_g.ptr, xpay=d_x.ptr)
    a.coef = -KAPPA * KAPPA
    tab, rows = it.groups(L, Nc, sizes), it.SegRows()
    assert it.call("dslash_dots_rows", a.g, Nc, prec, tab, rows)
    d_part = api.DeviceArray(8 * rows.total)
    for kind in (it.ALPHA, it.OMEGA):
        d_part.zero()
        assert it.call("launch_dslash_lane_dots_groups", a, kind, d_r0.ptr, tab, rows, d_part.ptr, 2, 2, None) == 0
        api.synchronize()
        part, out = d_part.download(np.float64), d_out.complex(n * Rt, prec)
        for k, R in enumerate(sizes):
            sums = part[rows.off[k]:rows.off[k] + rows.n[k] * R * 4].reshape(-1, R, 4).sum(0)
            own = slice(n * tab.base[k], n * (tab.base[k] + R))
            _compare(kind, sums, out[own], x[own], r0[own], R, n, (L, Nc, sizes, prec))

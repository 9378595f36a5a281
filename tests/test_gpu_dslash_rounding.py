"""Rounding of the 16-bit hops of the lane kernels.  Variant 1 computes in FP32
from the stored inputs on, so each stored component is the exact result
rounded once (and projected entries beyond the range of FP16 are no
overflow); variant 5 also rounds the projected spinors to the storage type,
like the matrix cores.  Lattices on which a site's directions share one
wavefront and on which they have one each."""
import numpy as np
import pytest

from oracle import oracle
from qcu_mrhs_amd import api, fields

pytestmark = pytest.mark.gpu

H, B = 0, 4
SHAPES = [((4, 4, 4, 4), 3, 4), ((4, 2, 6, 4), 3, 5), ((6, 4, 2, 10), 2, 17), ((8, 6, 4, 6), 4, 33), ((8, 12, 8, 16), 3, 12),
          ((4, 4, 4, 2), 4, 130)]


@pytest.fixture(autouse=True)
def _reset_tune():
    yield
    api.dslash_tune("auto")


def _hop(variant, L, Nc, R, prec, scale_in, scale_g, dagger, xpay, seed):
    g = fields.rng(seed)
    n = fields.half_volume(L) * 4 * Nc * R
    st = lambda a: api.from_storage(api.to_storage(a, prec), prec)  # noqa: E731
    inp, x = (st(scale_in * np.clip(g.standard_normal((n, 2)), -1.5, 1.5) @ [1, 1j]) for _ in range(2))
    gauge = st(scale_g * fields.gauge_field(L, Nc, seed + 1, kind="haar").reshape(-1))
    d = [api.DeviceArray.from_complex(v, prec) for v in (inp, x, gauge)]
    d_out = api.DeviceArray(api.storage_bytes(n, prec))
    coef = -0.75 if xpay else 1.0
    api.dslash_tune(variant)
    api.dslash_mrhs(d_out, d[0], d[2], L, Nc, R, 1, dagger, precision=prec, xpay=d[1] if xpay else None, coef=coef)
    got = d_out.complex(n, prec).view(np.float64)
    ref = coef * oracle.dslash(inp, gauge.reshape(4, 2, -1, Nc, Nc), L, Nc, R, 1, dagger)
    return got, (x + ref if xpay else ref).view(np.float64)


def _half_ulp(a, prec):
    bits, least = (11, -14) if prec == H else (8, -126)
    e = np.maximum(np.floor(np.log2(np.maximum(np.abs(a), 1e-300))), least)
    return 0.5 * 2.0 ** (e - bits + 1)


@pytest.mark.parametrize("scale_in,scale_g", [(1.0, 1.0), (2.5e4, 0.03)])
@pytest.mark.parametrize("prec", [H, B])
@pytest.mark.parametrize("L,Nc,R", SHAPES)
def test_variant_1_rounds_once(L, Nc, R, prec, scale_in, scale_g):
    for dagger, xpay in ((0, False), (1, True)):
        print("case rounding", L, Nc, R, prec, scale_in, dagger, xpay, flush=True)
        got, ref = _hop("lane_rhs", L, Nc, R, prec, scale_in, scale_g, dagger, xpay, 1200 + R)
        assert np.abs(ref).max() < 6e4 and np.isfinite(got).all()
        # FP32: 8 hops of 4 Nc products, each sum at most about 10 times the largest result
        slack = 16 * Nc * 2.0 ** -24 * 10 * np.abs(ref).max()
        # a rounding step further up where the FP32 error crosses a power of two
        assert (np.abs(got - ref) <= _half_ulp(np.abs(ref) + slack, prec) + slack).all()


@pytest.mark.parametrize("prec,tol", [(H, 2e-3), (B, 1.5e-2)])
@pytest.mark.parametrize("L,Nc,R", SHAPES + [((2, 2, 2, 2), 3, 1), ((6, 6, 4, 4), 3, 70), ((14, 6, 10, 6), 3, 3),
                                             ((4, 4, 4, 8), 2, 64), ((18, 16, 12, 22), 3, 5)])
def test_variant_5(L, Nc, R, prec, tol):
    for dagger, xpay in ((0, False), (1, True)):
        got, ref = _hop("lane_16", L, Nc, R, prec, 1.0, 1.0, dagger, xpay, 1300 + R)
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        print("case variant 5", L, Nc, R, prec, dagger, err, flush=True)
        assert err < tol


@pytest.mark.parametrize("prec", [1, 2])
def test_variant_5_is_variant_1_in_wider_storage(prec):
    L, Nc, R = (4, 6, 4, 6), 3, 12
    a, _ = _hop("lane_16", L, Nc, R, prec, 1.0, 1.0, 0, True, 1400)
    b, _ = _hop("lane_rhs", L, Nc, R, prec, 1.0, 1.0, 0, True, 1400)
    np.testing.assert_array_equal(a, b)

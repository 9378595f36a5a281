"""The hop with fused inner products and two FP32 right-hand sides per lane,
which runs where the fields exceed the 256 MiB memory-side cache: the number
of rows of partial sums shows that this form ran, the stored result against
the FP64 oracle for the first and last right-hand sides, and the sums against
numpy within the FP64 summation bound; with and without clover blocks, whose
hops without inner products have the same form."""
import numpy as np
import pytest

import internals as it
from oracle import oracle
from qcu_mrhs_amd import api, fields
from test_gpu_dots_sums import CSW, KAPPA, _compare, _setup

pytestmark = pytest.mark.gpu

S = 1


def _blocks_times(blocks, v, Nc):
    """Blocks [Vh][2][2 Nc][2 Nc] on a vector [Vh][4][Nc][R]."""
    b, w = blocks.reshape(-1, 2 * Nc, 2 * Nc), v.reshape(-1, 2 * Nc, v.size // (blocks.size // (2 * Nc)))
    return np.matmul(b, w).reshape(-1)


@pytest.mark.parametrize("Nc,R,clover", [(2, 64, False), (3, 44, False), (2, 64, True), (3, 44, True)])
def test_two_per_lane(Nc, R, clover):
    L = (16, 16, 16, 16)
    g = it.geom(L)
    assert g.Vh * (8 * Nc * Nc + 8 * Nc * R) * 8 > 1.02 * 2 ** 28  # links and two vectors
    n = g.Vh * 4 * Nc
    (inp, x, r0), (d_in, d_x, d_r0), gauge, d_g = _setup(L, Nc, n * R, S, 2100)
    d_out = api.DeviceArray(8 * n * R)
    a = it.args(L, Nc, R, S, out=d_out.ptr, inp=d_in.ptr, gauge=d_g.ptr, xpay=d_x.ptr)
    a.coef = -0.02
    cap = it.call("dslash_dots_partials", g, Nc, R, S)
    d_part, d_st = api.DeviceArray(8 * cap), api.DeviceArray(16 * it.NUM_SLOTS * R)
    some = [0, 1, R - 2, R - 1]
    gs = api.from_storage(api.to_storage(gauge.reshape(-1), S), S).reshape(gauge.shape)
    pick = lambda v: v.reshape(n, R)[:, some].reshape(-1)  # noqa: E731
    hop = oracle.dslash(pick(inp), gs, L, Nc, len(some), 1, 0)
    ref = pick(x) - 0.02 * hop
    if clover:
        d_c = api.DeviceArray(2 * g.Vh * 8 * Nc * Nc * 16)
        api.clover_build(d_c, None, api.DeviceArray.from_complex(gauge.reshape(-1)), L, Nc, CSW, KAPPA)
        blocks = api.from_storage(api.to_storage(d_c.complex(d_c.nbytes // 16)[d_c.nbytes // 32:], S), S)
        d_b = api.DeviceArray.from_complex(blocks, S)
        a.clover, a.clover_in, a.xpay = d_b.ptr, d_x.ptr, None
        ref = _blocks_times(blocks, pick(x), Nc) - 0.02 * hop
        # without the products: A (coef D in + x)
        h = it.args(L, Nc, R, S, out=d_out.ptr, inp=d_in.ptr, gauge=d_g.ptr, xpay=d_x.ptr, clover=d_b.ptr)
        h.coef = -0.02
        assert it.call("launch_dslash_clover", h, None) == 0
        api.synchronize()
        want = _blocks_times(blocks, pick(x) - 0.02 * hop, Nc)
        err = np.linalg.norm(pick(d_out.complex(n * R, S)) - want) / np.linalg.norm(want)
        print("case clover two per lane", Nc, R, err, flush=True)
        assert err < 2e-6
    for kind in (it.ALPHA, it.OMEGA):
        d_part.zero()
        d_st.upload(np.ones(it.NUM_SLOTS * R, dtype=np.complex128))
        assert it.call("launch_dslash_dots", a, kind, d_r0.ptr, d_part.ptr, cap, d_st.ptr, None) == 0
        api.synchronize()
        rows = d_part.download(np.float64).reshape(-1, R, 4)
        assert (rows[:, 0, 0] != 0).sum() == -(-g.Vh // (256 // (R // 2)))
        out = d_out.complex(n * R, S)
        err = np.linalg.norm(pick(out) - ref) / np.linalg.norm(ref)
        print("case dots two per lane", Nc, R, clover, kind, err, flush=True)
        assert err < (2e-6 if clover else 2e-7)
        _compare(kind, rows.sum(0), out, x, r0, R, n, (L, Nc, R, S, clover))

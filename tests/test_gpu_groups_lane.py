"""Batches with the lane kernel chosen explicitly for the inner and the FP64
hops (qcuGroupsDslashTune): the number that the library reports for a batch's
kernel is one that it accepts, and the batch then runs it; groups of one
right-hand side to more than a workgroup finishes in one pass of the fused
inner products (more than 4096 rows: 128 right-hand sides, two sites per row)."""
import numpy as np
import pytest

from oracle import oracle
from qcu_mrhs_amd import api, fields

pytestmark = pytest.mark.gpu

LANE = 6


@pytest.fixture(autouse=True)
def _reset():
    yield
    api.check(api.lib().qcuGroupsDslashTune(0, 0))
    api.finalizeQcu()


def _solve(L, Nc, sizes, inner, seed, kappa=0.12, tol=1e-10):
    gauge = fields.gauge_field(L, Nc, seed, kind="smooth", eps=0.8)
    api.initGridSize(L, Nc, 4, 2, inner)
    d_g = api.DeviceArray.from_complex(gauge.reshape(-1))
    api.loadQcuGauge(d_g, 2)
    api.getDslash(0, 1.0 / (2 * kappa) - 4.0)
    api.set_solver_options(inner, 0.1, False)
    srcs = [fields.gaussian_sources(L, Nc, R, seed + 1 + k) for k, R in enumerate(sizes)]
    groups = [([api.DeviceArray(v.nbytes) for v in b], [api.DeviceArray.from_complex(v) for v in b]) for b in srcs]
    infos = api.invert_groups(groups, 3000, tol)
    for g, b, info, R in zip(groups, srcs, infos, sizes):
        x = np.stack([v.complex(b.shape[1]) for v in g[0]])
        bm = fields.to_mrhs(b, Nc)
        res = bm - oracle.mat(fields.to_mrhs(x, Nc), gauge, L, Nc, R, kappa)
        rel = (oracle.norm(res, R) / oracle.norm(bm, R)).max()
        print("case groups lane", L, Nc, R, inner, info["iterations"], rel, flush=True)
        assert info["converged"] and rel < 1.5 * tol
    return api.lib().qcuGroupsDslashVariant(), api.lib().qcuGroupsDslashVariant64()


@pytest.mark.parametrize("inner", [1, 0, 4])
@pytest.mark.parametrize("L,Nc,sizes", [((8, 6, 4, 10), 3, (1, 7, 40)), ((6, 4, 4, 6), 4, (17, 33)), ((4, 4, 6, 6), 2, (128, 3)),
                                        ((8, 8, 16, 18), 2, (128, 3))])
def test_lane_kernel(L, Nc, sizes, inner):
    api.check(api.lib().qcuGroupsDslashTune(LANE, LANE))
    assert _solve(L, Nc, sizes, inner, 1900 + Nc) == (LANE, LANE)


def test_reported_kernel_can_be_chosen():
    case = ((8, 8, 8, 8), 3, (12, 12), 1, 1950)
    for _ in range(2):
        chosen = _solve(*case)
        api.check(api.lib().qcuGroupsDslashTune(*chosen))
        api.finalizeQcu()
        assert _solve(*case) == chosen
        api.finalizeQcu()
        api.check(api.lib().qcuGroupsDslashTune(0, 0))


def test_other_shapes_keep_the_timed_choice():
    api.check(api.lib().qcuGroupsDslashTune(LANE, LANE))
    inner, fp64 = _solve((4, 4, 4, 4), 8, (3, 5), 1, 1960)
    assert inner in (2, 3, 5) and fp64 in (2, 3, 5)


def test_choice_is_by_what_an_iteration_runs():
    """The lane kernel's bare hop is slower here than the packed matrix-core
    one, its iteration, which needs no separate inner products, faster by a
    tenth: the batch takes it."""
    assert _solve((6, 10, 14, 18), 4, (3, 8, 17), 1, 1970)[0] == LANE

"""GPU batched solves whose lane kernel forms the step's inner products: groups
from one right-hand side to the widest, lattices that leave workgroups partly
filled, every inner precision.  Every group's FP64 true residual through the
oracle operator."""
import numpy as np
import pytest

from oracle import oracle
from qcu_mrhs_amd import api, fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inner", [1, 0, 4])
@pytest.mark.parametrize("L,Nc,sizes", [((8, 6, 4, 10), 3, (1, 7, 40)), ((4, 4, 6, 6), 2, (128, 3)), ((6, 4, 4, 6), 4, (17, 33)),
                                        ((8, 8, 8, 8), 3, (12, 12))])
def test_groups(L, Nc, sizes, inner):
    kappa, tol = 0.12, 1e-10
    gauge = fields.gauge_field(L, Nc, 300 + Nc, kind="smooth", eps=0.8)
    api.initGridSize(L, Nc, 4, 2, inner)
    d_g = api.DeviceArray.from_complex(gauge.reshape(-1))
    api.loadQcuGauge(d_g, 2)
    api.getDslash(0, 1.0 / (2 * kappa) - 4.0)
    api.set_solver_options(inner, 0.1, False)
    srcs = [fields.gaussian_sources(L, Nc, R, 310 + k) for k, R in enumerate(sizes)]
    groups = [([api.DeviceArray(v.nbytes) for v in b], [api.DeviceArray.from_complex(v) for v in b]) for b in srcs]
    try:
        infos = api.invert_groups(groups, 3000, tol)
        variant = api.lib().qcuGroupsDslashVariant()
        xs = [np.stack([x.complex(b.shape[1]) for x in g[0]]) for g, b in zip(groups, srcs)]
    finally:
        api.finalizeQcu()
    for b, x, info, R in zip(srcs, xs, infos, sizes):
        bm = fields.to_mrhs(b, Nc)
        res = bm - oracle.mat(fields.to_mrhs(x, Nc), gauge, L, Nc, R, kappa)
        rel = (oracle.norm(res, R) / oracle.norm(bm, R)).max()
        print("case groups", L, Nc, sizes, inner, "kernel", variant, R, info["iterations"], rel, flush=True)
        assert info["converged"] and rel < 1.5 * tol

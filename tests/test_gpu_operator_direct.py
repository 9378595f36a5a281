"""GPU parity of start_dslash and mat_Qcu on the caller's own vectors: lanes that
do not divide evenly, one and several right-hand sides per wavefront, a
wavefront per direction and a lane per site, with and without the clover term,
against the FP64 oracle; and the calls whose vectors cannot be read in place
while the results are written (output on input, shared and overlapping
buffers, vectors aligned to their entries only), which keep their results."""
import numpy as np
import pytest

from oracle import oracle
from qcu_mrhs_amd import api, fields

pytestmark = pytest.mark.gpu

D, S = 2, 1
KAPPA, CSW = 0.125, 1.3
TOL = {D: 1e-13, S: 2e-6}


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def _setup(L, Nc, R, prec, clover, seed):
    gauge = fields.gauge_field(L, Nc, seed, kind="smooth", eps=0.6)
    api.initGridSize(L, Nc, R, prec, prec)
    d_g = api.DeviceArray.from_complex(gauge.reshape(-1))
    api.loadQcuGauge(d_g, D)
    api.getDslash(api.DSLASH_CLOVER if clover else 0, 1.0 / (2 * KAPPA) - 4.0)
    if clover:
        api.set_clover_coefficient(CSW)
    return gauge, (oracle.clover(gauge, L, Nc, CSW, KAPPA) if clover else None), d_g


def _ref_mat(v, gauge, c, L, Nc, R, dagger):
    if c is None:
        return oracle.mat(v, gauge, L, Nc, R, KAPPA, dagger)
    return oracle.clover_mat(v, gauge, c, L, Nc, R, KAPPA, dagger)


@pytest.mark.parametrize("prec", [D, S])
@pytest.mark.parametrize("L,Nc,R,clover", [((2, 2, 2, 2), 3, 1, False), ((4, 2, 6, 4), 3, 5, True), ((6, 4, 2, 10), 2, 17, False),
                                           ((4, 2, 4, 6), 4, 3, True), ((4, 6, 4, 6), 4, 33, False), ((2, 4, 2, 6), 2, 37, True),
                                           ((2, 2, 2, 6), 3, 128, False), ((2, 2, 4, 2), 4, 100, True),
                                           ((16, 12, 14, 18), 3, 4, True), ((14, 10, 14, 10), 3, 5, False)])
def test_operator_and_hop(L, Nc, R, clover, prec):
    gauge, c, d_g = _setup(L, Nc, R, prec, clover, 30 + R)
    src = fields.gaussian_sources(L, Nc, R, 31)
    src = np.stack([api.from_storage(api.to_storage(v, prec), prec) for v in src])
    n = src.shape[1]
    try:
        for dagger in (0, 1):
            ins = [api.DeviceArray.from_complex(v, prec) for v in src]
            outs = [api.DeviceArray(api.storage_bytes(n, prec)) for _ in range(R)]
            for r in range(R):
                api.pushBackFermions(outs[r], ins[r])
            api.mat_Qcu(dagger)
            got = fields.to_mrhs(np.stack([o.complex(n, prec) for o in outs]), Nc)
            err = _rel(got, _ref_mat(fields.to_mrhs(src, Nc), gauge, c, L, Nc, R, dagger))
            parity, half = dagger, n // 2
            hin = src.reshape(R, 2, half)[:, 1 - parity]
            ins = [api.DeviceArray.from_complex(np.ascontiguousarray(v), prec) for v in hin]
            for r in range(R):
                api.pushBackFermions(outs[r], ins[r])
            api.start_dslash(parity, dagger)
            got = fields.to_mrhs(np.stack([o.complex(half, prec) for o in outs]), Nc)
            err2 = _rel(got, oracle.dslash(fields.to_mrhs(hin, Nc), gauge, L, Nc, R, parity, dagger))
            print("case operator", L, Nc, R, clover, prec, dagger, err, err2, flush=True)
            assert err < TOL[prec] and err2 < TOL[prec]
    finally:
        api.finalizeQcu()


@pytest.mark.parametrize("how", ["in place", "crossed", "overlapping", "misaligned", "shared input"])
@pytest.mark.parametrize("clover", [False, True])
def test_vectors_that_alias(how, clover):
    L, Nc, R, prec = (4, 6, 2, 4), 3, 3, S
    gauge, c, d_g = _setup(L, Nc, R, prec, clover, 91)
    src = fields.gaussian_sources(L, Nc, R, 92)
    if how == "shared input":
        src = np.stack([src[0]] * R)
    src = np.stack([api.from_storage(api.to_storage(v, prec), prec) for v in src])
    n = src.shape[1]
    nb = api.storage_bytes(n, prec)
    arena = api.DeviceArray(2 * R * nb + 64)
    skew = 8 if how == "misaligned" else 0
    at_in = [r * nb + skew for r in range(R)]
    at_out = [(R + r) * nb + skew for r in range(R)]
    if how == "in place":
        at_out = at_in
    elif how == "crossed":
        at_out = at_in[1:] + at_in[:1]
    elif how == "overlapping":
        at_out = [o + nb // 2 // 16 * 16 - R * nb for o in at_out]  # halfway into the inputs
    elif how == "shared input":
        at_in = [at_in[0]] * R
    try:
        buf = np.zeros(arena.nbytes, np.uint8)
        for r in range(R):
            buf[at_in[r]:at_in[r] + nb] = np.ascontiguousarray(api.to_storage(src[r], prec)).view(np.uint8).reshape(-1)
        arena.upload(buf)
        for r in range(R):
            api.pushBackFermions(arena.offset(at_out[r]), arena.offset(at_in[r]))
        api.mat_Qcu(0)
        raw = arena.download(np.uint8)
        got = np.stack([raw[o:o + nb].copy().view(np.complex64) for o in at_out]).astype(np.complex128)
        err = _rel(fields.to_mrhs(got, Nc), _ref_mat(fields.to_mrhs(src, Nc), gauge, c, L, Nc, R, 0))
        print("case", how, clover, err, flush=True)
        assert err < TOL[prec]
    finally:
        api.finalizeQcu()

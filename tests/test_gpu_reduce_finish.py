"""GPU reductions at the edges of the finishing kernel (a workgroup per RHS over
the rows of partials): one row, fewer rows than lanes, a whole number of them
and one more, the most there are; one RHS to the widest.  Against FP64 sums of
the same inputs; the bound is that of n products summed in any order."""
import numpy as np
import pytest

from qcu_mrhs_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 3, 64, 256])
@pytest.mark.parametrize("rows", [1, 2, 63, 255, 256, 257, 1024, 3000])
def test_rows_of_partials(rows, R):
    per_block = 256 // R * R
    n = max(1, rows * per_block // R * (1 if rows <= 256 else 8) - 1)
    g = np.random.default_rng(7 * rows + R)
    a, b = ((g.standard_normal(n * R) + 1j * g.standard_normal(n * R)) for _ in range(2))
    da, db, out = api.DeviceArray.from_complex(a), api.DeviceArray.from_complex(b), api.DeviceArray(16 * R)
    api.check(api.lib().qcuBlasDotc(out.ptr, da.ptr, db.ptr, n, R, 2))
    api.synchronize()
    prod = (a.conj() * b).reshape(n, R)
    err = np.abs(out.complex(R) - prod.sum(axis=0))
    print("case rows", rows, R, n, err.max(), flush=True)
    assert (err <= 4 * n * np.finfo(np.float64).eps * np.abs(prod).sum(axis=0)).all()

"""Size of a solver's buffer for the fused inner products: rows for every form
that can run, and no buffer where none exists (Nc = 8 in FP32 and FP64,
vectors of 4 GiB and more)."""
import pytest

import internals as it


@pytest.mark.parametrize("L,Nc,R,prec", [((8, 8, 8, 8), 8, 4, 2), ((8, 8, 8, 8), 8, 16, 1), ((64, 64, 64, 32), 4, 8, 2),
                                         ((64, 64, 64, 64), 3, 12, 1)])
def test_no_form_no_buffer(L, Nc, R, prec):
    assert it.call("dslash_dots_partials", it.geom(L), Nc, R, prec) == 0


@pytest.mark.parametrize("prec", [0, 1, 2, 4])
@pytest.mark.parametrize("L,Nc,R", [((8, 8, 8, 8), 3, 4), ((8, 8, 8, 8), 4, 1), ((12, 12, 12, 12), 2, 64), ((6, 4, 4, 4), 3, 33),
                                    ((24, 24, 24, 24), 3, 16), ((4, 4, 4, 4), 4, 256)])
def test_rows_for_every_form(L, Nc, R, prec):
    g = it.geom(L)
    # at most 256 lanes of (site, RHS) per workgroup, or 64 with a wavefront per direction (up to 131072 lanes)
    rows = g.Vh * R // 256
    if R <= 64 and (64 // R) * R >= 48 and g.Vh * R <= (131072 if R <= 4 else 65536):
        rows = -(-g.Vh // (64 // R))
    assert it.call("dslash_dots_partials", g, Nc, R, prec) >= (rows + 512) * R * 4


def test_matrix_cores_in_16_bits():
    g = it.geom((8, 8, 8, 8))
    assert it.call("dslash_dots_partials", g, 8, 4, 0) >= (g.Vh // 4 + 512) * 16

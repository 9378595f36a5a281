"""The automatic choice of a 16-bit hop's kernel, where the lane kernel and the
matrix cores were timed against each other: matrix cores (3) on small
lattices whose fields stay in the caches, lanes (5) beyond; a kernel named in
the call stays."""
import pytest

import internals as it

SITES = {"8^4": (8, 8, 8, 8), "8^3x16": (8, 8, 8, 16), "12^4": (12, 12, 12, 12), "16^4": (16, 16, 16, 16),
         "16^3x32": (16, 16, 16, 32), "24^4": (24, 24, 24, 24), "24^3x48": (24, 24, 24, 48)}


@pytest.mark.parametrize("prec", [0, 4])
@pytest.mark.parametrize("lattice,Nc,R,want", [
    # up to 1.45 times the matrix cores' time on lanes
    ("12^4", 4, 16, 3), ("12^4", 4, 12, 3), ("12^4", 4, 8, 3), ("8^4", 4, 48, 3), ("8^3x16", 4, 17, 3), ("8^3x16", 4, 12, 3),
    ("8^4", 3, 48, 3), ("8^3x16", 3, 17, 3), ("12^4", 3, 16, 3), ("16^3x32", 4, 16, 3), ("8^3x16", 2, 17, 3),
    # and down to half of it
    ("12^4", 4, 4, 5), ("8^3x16", 4, 64, 5), ("16^4", 4, 8, 5), ("24^4", 4, 16, 5), ("12^4", 3, 20, 5), ("12^4", 3, 8, 5),
    ("16^4", 3, 12, 5), ("24^3x48", 3, 16, 5), ("24^3x48", 3, 32, 5), ("8^3x16", 2, 20, 5), ("12^4", 2, 17, 5)])
def test_16_bit_hop(lattice, Nc, R, want, prec):
    a = it.args(SITES[lattice], Nc, R, prec)
    assert it.call("dslash_resolve", a).variant == want
    a.clover = 1  # the fused clover forms are the lane kernel's
    assert it.call("dslash_resolve", a).variant == 5
    a.tune.variant = 8 - want
    assert it.call("dslash_resolve", a).variant == 8 - want

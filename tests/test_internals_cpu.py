"""The structure mirrors of tests/internals.py against the library, on the
host: each field that a launch reads changes what the host-side functions
return."""
import ctypes

import internals as it


def test_layouts():
    assert [ctypes.sizeof(c) for c in (it.Geom, it.DslashArgs, it.SegTab, it.SegRows)] == [24, 120, 128, 136]
    L, D, H = (8, 12, 16, 20), 2, 0
    t = it.call("dslash_resolve", it.args(L, 3, 12, D))
    assert t.variant == 1 and L[1] % t.by == 0 and L[2] % t.bz == 0 and (t.by, t.bz) != (0, 0)
    a = it.args(L, 3, 12, H, 2)
    a.tune.by, a.tune.bz, a.tune.spw = 3, 8, 2
    t = it.call("dslash_resolve", a)
    assert (t.variant, t.by, t.bz, t.spw) == (2, 3, 8, 2)
    # the fused clover form: 16 bits only as variant 5, not with keep_order, not where the directions are split
    big = (16, 16, 16, 32)
    for variant, keep, lattice, want in ((5, False, big, True), (1, False, big, False), (5, True, big, False),
                                         (5, False, (4, 4, 4, 4), False)):
        a = it.args(lattice, 3, 12, H, variant, keep_order=keep)
        assert it.call("dslash_lane_clover_fused", a, a.tune) == want


def test_group_rows():
    L, sizes, rows = (4, 4, 6, 6), (5, 12), it.SegRows()
    assert it.call("dslash_dots_rows", it.geom(L), 3, 0, it.groups(L, 3, sizes), rows)
    for k, R in enumerate(sizes):
        assert rows.n[k] == -(-288 // rows.sites[k]) and rows.sites[k] * R <= 256
    assert rows.off[0] == 0 and rows.off[1] == rows.n[0] * 5 * 4 and rows.total == rows.off[1] + rows.n[1] * 12 * 4

"""Tile cycles of many tiles: a rect of just over 1024 (from where a cycle is
ended by a kernel of its own), and learned cycles that list more tiles than the
list kernel has blocks, so that a block takes several.  Bit for bit the
separate passes', state, scalars and closure counts, in runs that end in the
first and in the second cycle of a pair and in odd launches."""
import numpy as np
import pytest

import pennant_amd as pa
from pennant_amd import decks as wd

pytestmark = pytest.mark.gpu

STATE = ("px", "pu", "zr", "ze", "zp", "zetot", "zwrate", "zvol")
SCAL = ("time", "dt", "dtrec", "cycle", "dtnew", "dvovmax", "dtnext", "done", "numsbad_pred", "numsbad_corr")
RECT = 460                                       # 33 x 33 tiles of 14 x 14 zones


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def state(text, mode, tiles, steps, mlp=None, squeeze=0.0):
    with pa.Problem(text) as pb:
        pb.set_tuning("tiles", tiles)
        assert pb.get_tuning("tiles") == tiles
        if mlp is not None:
            pb.set_closure(mlp)
        if squeeze:
            pb.set("pu", -squeeze * pb.get("px"))
        for n in steps:
            pb.run(n, mode)
        return {f: pb.get(f) for f in STATE}, pb.scalars(), pb.closure_stats() if mlp is not None else None


def compare(text, mode, steps, mlp=None, squeeze=0.0):
    a = state(text, mode, 1, steps, mlp, squeeze)
    b = state(text, mode, 0, steps, mlp, squeeze)
    for f in STATE:
        assert np.array_equal(bits(a[0][f]), bits(b[0][f])), (steps, f)
    for k in SCAL:
        assert bits(a[1][k]) == bits(b[1][k]), (steps, k)
    assert a[2] == b[2], steps
    return a


@pytest.mark.parametrize("cstop", [20, 21])
@pytest.mark.parametrize("mode", [pa.MODE_FUSED, pa.MODE_MIXED])
def test_a_rect_of_over_1024_tiles(mode, cstop):
    for steps in ([100], [3, 2, 100]):
        st = compare(wd.sedov_rect(RECT, cstop=cstop), mode, steps)
        assert st[1]["cycle"] == cstop and st[1]["done"] == 1


@pytest.mark.parametrize("cstop", [6, 7])
@pytest.mark.parametrize("mesh", ["rect", "pie"])
def test_more_listed_tiles_than_blocks(mesh, cstop):
    """Every zone of a converging flow compresses, so every tile is listed:
    1089 of a rect, 841 of a pie."""
    from pennant_amd.closure import Mlp
    from pennant_amd.train_closure import DEFAULT_OUT
    m = Mlp.load(DEFAULT_OUT)
    if mesh == "rect":
        text, zones = wd.sedov_rect(RECT, cstop=cstop), RECT * RECT
    else:
        text, zones = wd.noh_pie(400, 400, cstop=cstop, dtinit=1e-5), 400 * 399
    for steps in ([100], [3, 100]):
        st = compare(text, pa.MODE_LEARNED, steps, m, squeeze=0.5 if mesh == "rect" else 0.0)
        assert st[1]["cycle"] == cstop and st[1]["done"] == 1
        # gated zones over all cycles; a tile has at most 196, the list kernel 512 blocks
        assert sum(st[2]) > cstop * 512 * 196, (st[2], zones)
    m.close()

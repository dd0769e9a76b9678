"""The tile cycle of structured meshes (tuning key "tiles", on by default): a
whole cycle in one kernel over tiles of 14 x 14 zones and their ring.

Checked bit for bit at the edges of tiles (meshes of 1, 13, 14, 15, 28 and 29
zones a row, one-row and two-row pies, origins with few and with many
corners): the FP64 form against the oracle, the mixed and learned forms
against the separate passes; runs that end in the first and in the second
cycle of a pair, and launches of odd and even length.
"""
import numpy as np
import pytest

import pennant_amd as pa
from pennant_amd import decks as wd
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

STATE = ("px", "pu", "zr", "ze", "zp", "zetot", "zwrate", "zvol")
SCAL = ("time", "dt", "dtrec", "cycle", "dtnew", "dvovmax", "dtnext", "done", "numsbad_pred", "numsbad_corr")

DECKS = {
    "rect1": lambda c: wd.sedov_rect(1, cstop=c),
    "rect13": lambda c: wd.sedov_rect(13, cstop=c),
    "rect14": lambda c: wd.sedov_rect(14, cstop=c),
    "rect15": lambda c: wd.sedov_rect(15, cstop=c, bc_far=True),
    "rect28x29": lambda c: wd.leblanc_rect(28, 29, cstop=c),
    "pie2x3": lambda c: wd.noh_pie(2, 3, cstop=c, dtinit=1e-4),
    "pie15x14": lambda c: wd.noh_pie(15, 14, cstop=c, dtinit=1e-4),
    "pie16x29": lambda c: wd.noh_pie(16, 29, cstop=c, dtinit=1e-4),
    "pie30x80": lambda c: wd.noh_pie(30, 80, cstop=c, dtinit=1e-4),
    "pie2x600": lambda c: wd.noh_pie(2, 600, cstop=c, dtinit=1e-4),
}


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def state(text, mode, tiles, steps, mlp=None):
    with pa.Problem(text) as pb:
        pb.set_tuning("tiles", tiles)
        assert pb.get_tuning("tiles") == tiles
        if mlp is not None:
            pb.set_closure(mlp)
        for n in steps:
            pb.run(n, mode)
        return {f: pb.get(f) for f in STATE}, pb.scalars(), pb.closure_stats() if mlp is not None else None


@pytest.mark.parametrize("cstop", [16, 21])
@pytest.mark.parametrize("name", sorted(DECKS))
def test_fp64_tiles_match_the_oracle(name, cstop):
    text = DECKS[name](cstop)
    o = Oracle(text)
    ran = o.run(cstop)            # to cstop, or to tstop where that comes first
    for steps in ([100], [1, 2, 17, 100]):
        st, sc, _ = state(text, pa.MODE_FUSED, 1, steps)
        assert sc["cycle"] == ran and sc["done"] == 1
        for f in STATE:
            assert np.array_equal(bits(st[f]), bits(o.get(f))), (name, steps, f)


@pytest.mark.parametrize("mode", [pa.MODE_MIXED, pa.MODE_LEARNED])
@pytest.mark.parametrize("name", sorted(DECKS))
def test_mixed_tiles_match_the_separate_passes(name, mode):
    from pennant_amd.closure import Mlp
    from pennant_amd.train_closure import DEFAULT_OUT
    m = Mlp.load(DEFAULT_OUT) if mode == pa.MODE_LEARNED else None
    text = DECKS[name](33)
    for steps in ([100], [3, 2, 100]):
        a = state(text, mode, 1, steps, m)
        b = state(text, mode, 0, steps, m)
        for f in STATE:
            assert np.array_equal(bits(a[0][f]), bits(b[0][f])), (name, steps, f)
        for k in SCAL:
            assert bits(a[1][k]) == bits(b[1][k]), (name, steps, k)
        assert a[2] == b[2], (name, steps)


def test_tiles_stop_on_bad_sides_as_the_separate_passes():
    """A step far too long inverts zones: the same cycle, counts and state (a
    NaN that it leaves is a NaN in both; its sign, which the arithmetic leaves
    open, is not compared)."""
    text = wd.noh_pie(16, 15, cstop=50, dtinit=2.0, tstop=1e3).replace("cfl 0.6", "cfl 1e6\ncflv 1e6")
    got = []
    for tiles in (1, 0):
        with pa.Problem(text) as pb:
            pb.set_tuning("tiles", tiles)
            with pytest.raises(pa.PennantError):
                pb.run(50, pa.MODE_FUSED)
            got.append(({f: pb.get(f) for f in STATE}, pb.scalars()))
    for k in SCAL:
        assert bits(got[0][1][k]) == bits(got[1][1][k]), k
    for f in STATE:
        a, b = got[0][0][f], got[1][0][f]
        nan = np.isnan(a)
        assert np.array_equal(nan, np.isnan(b)), f
        assert np.array_equal(bits(a[~nan]), bits(b[~nan])), f


@pytest.mark.parametrize("mode", [pa.MODE_FUSED, pa.MODE_MIXED])
def test_batch_tiles_match_single_runs(mode):
    """Rect and pie meshes at the edges of tiles in one arena (non-zero zone,
    side and point offsets), stopping at different cycles."""
    names = sorted(DECKS)
    texts = [DECKS[n](20 + k) for k, n in enumerate(names)]
    for steps in ([60], [1, 2, 3, 60]):
        with pa.Batch(texts) as b:
            assert b.get_tuning("tiles") == 1
            for n in steps:
                b.run(n, mode)
            for i, t in enumerate(texts):
                st, sc, _ = state(t, mode, 0, [100])
                got = b.scalars(i)
                for k in SCAL:
                    assert bits(got[k]) == bits(sc[k]), (names[i], steps, k)
                for f in STATE:
                    assert np.array_equal(bits(b.get(i, f)), bits(st[f])), (names[i], steps, f)


def test_a_mesh_that_does_not_qualify():
    with pa.Problem(wd.noh_pie(1, 7, cstop=3, dtinit=1e-4)) as pb:      # triangles only
        assert pb.get_tuning("tiles") == 0
        assert pb.run(5, pa.MODE_FUSED) == 3
    with pa.Batch([wd.sedov_rect(8, cstop=3), wd.noh_pie(1, 7, cstop=3, dtinit=1e-4)]) as b:
        assert b.get_tuning("tiles") == 0
        b.run(5, pa.MODE_FUSED)

"""The separate passes of the fused cycle (tuning "tiles" 0) at every launch
shape and with computed and read maps, also on the structured meshes whose
cycles run as tiles by default: odd cycles, captures, the pipelined cycle, the
learned form of a batch and the autotuners' other shapes take them there too.
FP64 against the oracle, the mixed and learned forms against the default shape,
bit for bit."""
import numpy as np
import pytest

import pennant_amd as pa
from pennant_amd import decks as wd
from golden_decks import ref_deck
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

STATE = ("px", "pu", "zr", "ze", "zp", "zetot", "zwrate", "zvol")


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def passes(text, mode, cycles, mlp=None, **tuning):
    with pa.Problem(text) as pb:
        pb.set_tuning("tiles", 0)
        assert pb.get_tuning("tiles") == 0
        for k, v in tuning.items():
            pb.set_tuning(k, v)
        if mlp is not None:
            pb.set_closure(mlp)
        n = pb.run(cycles, mode)
        return n, {f: bits(pb.get(f)) for f in STATE}, bits(pb.scalars()["dtrec"]), \
            pb.closure_stats() if mlp is not None else None


def same(a, b, tag):
    assert a[0] == b[0] > 0, tag
    for f in STATE:
        assert np.array_equal(a[1][f], b[1][f]), (tag, f)
    assert a[2:] == b[2:], tag


def one_by_five(cstop):
    lines = [ln for ln in wd.sedov_rect(1, cstop=cstop).splitlines() if not ln.startswith("meshparams")]
    return "\n".join(lines) + "\nmeshparams 1 5 1.0 1.0\n"


@pytest.mark.parametrize("k1,maxb,xcd", [(0, 1, 1), (0, 7, 1), (0, 8, 1), (0, 16, 0), (0, 512, 1),
                                         (1, 1, 1), (1, 5, 1), (1, 24, 1), (1, 4096, 0)])
def test_fp64_launch_shapes(k1, maxb, xcd):
    for text in (wd.noh_pie(40, 24, cstop=12, dtinit=1e-4), wd.sedov_rect(37, cstop=12)):
        o = Oracle(text)
        o.run(100)
        n, st, dtrec, _ = passes(text, pa.MODE_FUSED, 100, k1_layout=k1, max_blocks=maxb, xcd=xcd)
        assert n == 12 and dtrec == bits(o.scalars()["dtrec"])
        for f in STATE:
            assert np.array_equal(st[f], bits(o.get(f))), f


@pytest.mark.parametrize("maxb,xcd", [(1, 1), (7, 0), (48, 1), (4096, 0)])
def test_mixed_launch_shapes(maxb, xcd):
    for text in (wd.noh_pie(40, 24, cstop=30, dtinit=1e-4), wd.sedov_rect(37, cstop=30)):
        same(passes(text, pa.MODE_MIXED, 100), passes(text, pa.MODE_MIXED, 100, max_blocks=maxb, xcd=xcd), text[:40])


@pytest.mark.parametrize("pipeline", [0, 1])
@pytest.mark.parametrize("mode", [pa.MODE_FUSED, pa.MODE_MIXED])
def test_computed_and_read_maps(mode, pipeline):
    for text in (wd.sedov_rect(37, cstop=40), wd.leblanc_rect(64, 8, cstop=40), ref_deck("sedov"), one_by_five(40)):
        a = passes(text, mode, 30, rect_maps=1, pipeline=pipeline)
        same(a, passes(text, mode, 30, rect_maps=0, pipeline=pipeline), text[:40])
        if mode == pa.MODE_FUSED:
            o = Oracle(text)
            o.run(a[0])
            for f in STATE:
                assert np.array_equal(a[1][f], bits(o.get(f))), f


def test_learned_list_slices():
    """One list slice per XCD band, or a single one: a triangle run and a quad
    run of 50 units."""
    from pennant_amd.closure import Mlp
    from pennant_amd.train_closure import DEFAULT_OUT
    m = Mlp.load(DEFAULT_OUT)
    text = wd.noh_pie(128, 100, cstop=500, dtinit=1e-4)
    ref = passes(text, pa.MODE_LEARNED, 40, m, max_blocks=2048, xcd=1)
    assert ref[3][0] > 0
    for cap, xcd in ((48, 1), (16, 1), (13, 1), (48, 0)):
        same(ref, passes(text, pa.MODE_LEARNED, 40, m, max_blocks=cap, xcd=xcd), (cap, xcd))
    m.close()


def batch_state(texts, mode, **tuning):
    with pa.Batch(texts) as b:
        b.set_tuning("tiles", 0)
        assert b.get_tuning("tiles") == 0
        for k, v in tuning.items():
            b.set_tuning(k, v)
        b.run(25, mode)
        return [(b.scalars(i)["cycle"], [bits(b.get(i, f)) for f in STATE]) for i in range(len(texts))]


@pytest.mark.parametrize("mode", [pa.MODE_FUSED, pa.MODE_MIXED])
def test_batch_shapes_and_maps(mode):
    """Rect problems after pie problems in the arena: every grid, computed and
    read maps, against the single runs' passes."""
    texts = [wd.noh_pie(40, 24, cstop=30, dtinit=1e-4), wd.sedov_rect(37, cstop=20), wd.noh_pie(3, 9, cstop=30),
             wd.leblanc_rect(64, 8, cstop=23), one_by_five(30)]
    want = [passes(t, mode, 25) for t in texts]
    for tuning in ({}, {"rect_maps": 0}, {"max_blocks": 1, "xcd": 0}, {"max_blocks": 7, "xcd": 1},
                   {"max_blocks": 64, "xcd": 1}, {"max_blocks": 65535, "xcd": 0}):
        for i, (cycle, st) in enumerate(batch_state(texts, mode, **tuning)):
            assert cycle == want[i][0], (tuning, i)
            for f, x in zip(STATE, st):
                assert np.array_equal(x, want[i][1][f]), (tuning, i, f)

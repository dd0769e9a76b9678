"""Task-mode cycles (four launches for the thirty steps of doCycle) against the
same steps through the task entry points, one launch per task: every field and
scalar bit for bit, at the edges of the zone tiles (64 quads or triangles) and
of the point blocks, at origins of 2 to 5, 64, 65, 255 to 257 and 300 corners, for
runs of single cycles and of captured ones, up to the stop condition and past
it.
"""
import numpy as np
import pytest

import pennant_amd as pa
from pennant_amd import decks as wd

pytestmark = pytest.mark.gpu

FIELDS = ("px pxp px0 pu pu0 pf pap pmaswt zx zxp zuc zarea zvol zareap zvolp zvol0 zdl zm zr zrp ze "
          "zetot zw zwrate zp zss zdu ztmp ex exp ssurfp sfp sfq sft cqe1 cqe2 sarea svol sareap svolp "
          "elen smf carea cevol cdu cdiv ccos crmu cw").split()
SCAL = ("time", "dt", "dtrec", "cycle", "dtnew", "dvovmax", "dtnext", "done", "numsbad_pred", "numsbad_corr")

DECKS = {
    "rect1x1": lambda c: wd.leblanc_rect(1, 1, cstop=c),
    "rect21x3": lambda c: wd.leblanc_rect(21, 3, cstop=c),
    "rect64x1": lambda c: wd.leblanc_rect(64, 1, cstop=c),
    "rect13x5": lambda c: wd.leblanc_rect(13, 5, cstop=c),
    "sedov37": lambda c: wd.sedov_rect(37, cstop=c, bc_far=True),
    "pie4x3": lambda c: wd.noh_pie(4, 3, cstop=c, dtinit=1e-4),
    "pie5x2": lambda c: wd.noh_pie(5, 2, cstop=c, dtinit=1e-4),
    "pie255x2": lambda c: wd.noh_pie(255, 2, cstop=c, dtinit=1e-4),
    "pie256x3": lambda c: wd.noh_pie(256, 3, cstop=c, dtinit=1e-4),
    "pie257x2": lambda c: wd.noh_pie(257, 2, cstop=c, dtinit=1e-4),
    "pie300x5": lambda c: wd.noh_pie(300, 5, cstop=c, dtinit=1e-4),
    # radial zones x sectors (the origin's corners)
    "pie3x4": lambda c: wd.noh_pie(3, 4, cstop=c, dtinit=1e-4),
    "pie2x5": lambda c: wd.noh_pie(2, 5, cstop=c, dtinit=1e-4),
    "pie2x64": lambda c: wd.noh_pie(2, 64, cstop=c, dtinit=1e-4),
    "pie2x65": lambda c: wd.noh_pie(2, 65, cstop=c, dtinit=1e-4),
    "pie2x255": lambda c: wd.noh_pie(2, 255, cstop=c, dtinit=1e-4),
    "pie3x256": lambda c: wd.noh_pie(3, 256, cstop=c, dtinit=1e-4),
    "pie2x257": lambda c: wd.noh_pie(2, 257, cstop=c, dtinit=1e-4),
    "pie5x300": lambda c: wd.noh_pie(5, 300, cstop=c, dtinit=1e-4),
}


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def same(a, b, what):
    """Equal bits; a NaN equals a NaN (its sign is left open)."""
    a, b = np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64)
    ok = (bits(a) == bits(b)) | (np.isnan(a) & np.isnan(b))
    assert ok.all(), (what, np.argwhere(~ok)[:4])


@pytest.mark.parametrize("name", sorted(DECKS))
def test_cycles_match_the_task_entry_points(name):
    text = DECKS[name](19)
    with pa.Problem(text) as one:
        while not one.scalars()["done"]:
            for k in range(30):
                assert one.step(k) == 0
            one.end_cycle()
        for runs in ([100], [1, 2, 16, 100]):
            with pa.Problem(text) as pb:
                for n in runs:
                    pb.run(n, pa.MODE_TASKS)
                sp, so = pb.scalars(), one.scalars()
                for k in SCAL:
                    assert bits(sp[k]) == bits(so[k]), (name, runs, k)
                for f in FIELDS:
                    same(pb.get(f), one.get(f), (name, runs, f))


def test_cycles_stop_on_bad_sides():
    """A step far too long inverts zones: no cycle runs after the one that
    found it, alone or in a captured run."""
    text = wd.noh_pie(16, 15, cstop=50, dtinit=2.0, tstop=1e3).replace("cfl 0.6", "cfl 1e6\ncflv 1e6")
    with pa.Problem(text) as one:
        while not one.scalars()["done"]:
            for k in range(30):
                rc = one.step(k)
                assert rc == 0 or k in (18, 29)      # the bad-side checks
            try:
                one.end_cycle()
            except pa.PennantError:
                break
        so = one.scalars()
        assert so["numsbad_pred"] + so["numsbad_corr"] > 0
        for runs in ([50], [1] * 15):
            with pa.Problem(text) as pb:
                with pytest.raises(pa.PennantError):
                    for n in runs:
                        pb.run(n, pa.MODE_TASKS)
                sp = pb.scalars()
                for k in SCAL:
                    assert bits(sp[k]) == bits(so[k]), (runs, k)
                for f in FIELDS:
                    same(pb.get(f), one.get(f), (runs, f))

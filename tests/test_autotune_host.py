"""The autotuners' decisions, on a HIP runtime without a device: which cycles
they time, what they leave behind, and that a snapshot that cannot be taken is
an error with nothing run."""
from fake_hip import run_fake  # noqa: F401


def test_a_failed_snapshot_runs_nothing(run_fake):
    """Every allocation and every copy of the snapshot in turn fails: the call
    returns the error, no kernel has run, the tuning and the memory in use are
    what they were, and the next launch is not told of the error."""
    run_fake("""
def check(h, tune, launch, tuning):
    for what in ("malloc", "copy"):
        for k in range(1, 13):
            launch(2, pa.MODE_MIXED)
            before, live = [tuning(key) for key in ("tiles", "xcd", "max_blocks", "graph")], fake.live
            clear()
            fake.fail_bytes = 0
            setattr(fake, "fail_" + what, k)
            ms = ctypes.c_double()
            rc = tune(h, pa.MODE_MIXED, 4, ctypes.byref(ms))
            setattr(fake, "fail_" + what, 0)
            assert rc == 2, (what, k, rc)
            assert names() == [], (what, k, names())
            assert [tuning(key) for key in ("tiles", "xcd", "max_blocks", "graph")] == before
            assert fake.live == live, (what, k)
            launch(2, pa.MODE_MIXED)

L = pa.lib()
with pa.Problem(wd.sedov_rect(20, cstop=100)) as pb:
    check(pb._h, L.pennant_autotune, pb.launch, pb.get_tuning)
    pb.set_tuning("pipeline", 1)                # the look-ahead is current before each call
    check(pb._h, L.pennant_autotune, pb.launch, pb.get_tuning)
with pa.Batch([wd.sedov_rect(20, cstop=100), wd.noh_pie(6, 5, cstop=100)]) as b:
    check(b._h, L.pennant_batch_autotune, b.launch, b.get_tuning)
""")


def test_an_odd_number_of_cycles_times_tiles(run_fake):
    """Tiles run in pairs.  With a cycle's time its number of kernels (four as
    separate passes, one as tiles and one more a run), the time of an odd number
    of cycles is that of tile cycles alone, scaled, and tiles are kept."""
    run_fake("""
for cycles in (1, 3, 4, 7):
    even = cycles + cycles % 2
    with pa.Problem(wd.sedov_rect(20, cstop=100)) as pb:
        best = pb.autotune(pa.MODE_FUSED, cycles)
        assert best == (even + 1) * cycles / even, (cycles, best)
        assert pb.get_tuning("tiles") == 1
    with pa.Batch([wd.sedov_rect(20, cstop=100), wd.leblanc_rect(15, 7, cstop=100)]) as b:
        best = b.autotune(pa.MODE_FUSED, cycles)
        assert best == (2 * even + 1) * cycles / even, (cycles, best)
        assert b.get_tuning("tiles") == 1
""")


def test_tiles_are_decided_for_the_form_that_was_timed(run_fake):
    """Where tiles lose they are off for that form's cycles and on for the
    others'; where they cannot be timed (the learned form of a batch, a capture
    buffer) they are left as they were; and the FP64 form's choices leave the
    mixed cycle's pipelining as it was."""
    run_fake("""
from pennant_amd.closure import Mlp
mlp = Mlp(0)
def tiles(h, mode):
    clear()
    h.launch(2, mode)
    return any("6k_tileI" in n or "k_tile_batch" in n for n in names())

FORMS = (pa.MODE_FUSED, pa.MODE_MIXED, pa.MODE_LEARNED)
text = wd.sedov_rect(20, cstop=100)
for form in FORMS:
    with pa.Problem(text) as pb:
        pb.set_closure(mlp)
        assert pb.get_tuning("tiles") == 1
        slow("6k_tileI")
        pb.autotune(form, 4)
        slow("")
        assert pb.get_tuning("tiles") == 0
        pb.set_tuning("pipeline", 0)
        assert [tiles(pb, f) for f in FORMS] == [f != form for f in FORMS], form
        pb.set_tuning("tiles", 1)
        pb.set_tuning("k1_layout", 0)
        assert [tiles(pb, f) for f in FORMS] == [True] * 3

with pa.Problem(text) as pb:                 # a capture buffer: not timed
    class Buf: ptr = 4096
    pb.set_capture(Buf, 16)
    pb.autotune(pa.MODE_MIXED, 4)
    pb.set_capture(None, 0)
    pb.set_tuning("pipeline", 0)
    assert pb.get_tuning("tiles") == 1 and tiles(pb, pa.MODE_MIXED)

with pa.Problem(text) as pb:                 # the FP64 form says nothing of pipelining
    pb.set_tuning("pipeline", 1)
    pb.autotune(pa.MODE_FUSED, 4)
    assert pb.get_tuning("pipeline") == 1 and tiles(pb, pa.MODE_FUSED)

with pa.Problem(text) as pb:                 # the FP64 form's layout is no other form's
    pb.set_tuning("k1_layout", 1)
    assert not tiles(pb, pa.MODE_FUSED) and tiles(pb, pa.MODE_MIXED)

with pa.Batch([text, wd.noh_pie(6, 5, cstop=100)]) as b:
    b.set_closure(mlp)
    b.autotune(pa.MODE_LEARNED, 4)
    assert b.get_tuning("tiles") == 1 and tiles(b, pa.MODE_MIXED) and tiles(b, pa.MODE_FUSED)
    slow("k_tile_batch")
    b.autotune(pa.MODE_MIXED, 4)
    slow("")
    assert b.get_tuning("tiles") == 0 and not tiles(b, pa.MODE_MIXED) and tiles(b, pa.MODE_FUSED)
""")

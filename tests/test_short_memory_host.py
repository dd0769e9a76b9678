"""Problems and batches where device memory is short, on a HIP runtime without a
device: without memory for what only makes a cycle or a creation faster (the
tile cycle's second state, the arena of a small problem) they are created all
the same and run as separate passes or on arrays of their own."""
from fake_hip import run_fake  # noqa: F401


def test_no_memory_for_the_second_state(run_fake):
    run_fake("""
def passes(h):
    clear()
    h.launch(4, pa.MODE_FUSED)
    return len(names()) >= 16 and not any("tile" in n for n in names())

n = 560                                      # above the arena's limit: an allocation for each array
second = 8 * (4 * (n + 1) ** 2 + 5 * n * n)
fake.fail_bytes, fake.fail_malloc = second, 2    # the first as large: the corner records
with pa.Problem(wd.sedov_rect(n, cstop=100)) as pb:
    assert fake.fail_malloc == 0
    assert pb.get_tuning("tiles") == 0 and passes(pb)
    pb.autotune(pa.MODE_MIXED, 2)

decks = [wd.sedov_rect(20, cstop=100), wd.leblanc_rect(15, 7, cstop=100)]
second = 8 * (4 * (21 ** 2 + 16 * 8) + 5 * (400 + 105))
fake.fail_bytes, fake.fail_malloc = second, 4    # the corner records, the problems' arenas, this
with pa.Batch(decks) as b:
    assert fake.fail_malloc == 0
    assert b.get_tuning("tiles") == 0 and passes(b)
assert fake.live == 0
""")


def test_no_arena(run_fake):
    run_fake("""
fake.fail_bytes, fake.fail_malloc = 1 << 20, 1
with pa.Problem(wd.sedov_rect(90, cstop=100)) as pb:
    assert fake.fail_malloc == 0
    pb.launch(4, pa.MODE_FUSED)
    assert pb.get_tuning("tiles") == 1
assert fake.live == 0
""")

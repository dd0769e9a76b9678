"""How the closure network's row kernel is launched, on a HIP runtime without a
device (which refuses 2^32 threads or more in a launch, as the real one does)."""
from fake_hip import run_fake  # noqa: F401


def test_forward_takes_any_number_of_rows(run_fake):
    """Below, at and above the rows of one launch; the pointers are not read."""
    run_fake("""
from pennant_amd.closure import Mlp
m = Mlp(0)
for n in (1, 32, 33, 2 ** 30, 2 ** 30 + 1, 2 ** 31 - 1, 2 ** 31, 2 ** 32 + 5):
    clear()
    assert pa.lib().pennant_mlp_forward(m._h, 1 << 12, n, 1 << 12, 0) == 0, n
    assert len(names()) == -(-n // 2 ** 30) and all("k_rows" in k for k in names()), n
""")


def test_training_ends_waited_for(run_fake):
    """An error left by another call is reported before the first step, and one
    in the middle of the steps after the kernels that read the caller's tuples
    and the rows' lists have ended."""
    run_fake("""
from pennant_amd.closure import Mlp
m = Mlp(0)
def train(steps):
    clear()
    return pa.lib().pennant_mlp_train(m._h, 1 << 12, 100, steps, 64, 1e-3, 7, None)
assert train(6) == 0 and len(names()) == 18
fake.error = 2
assert train(6) == 2 and names() == [], names()
fake.fail_wait = 2
assert train(6) == 999 and len(names()) == 9 and fake.queued == 0, (names(), fake.queued)
fake.error = 0
assert train(6) == 0 and len(names()) == 18
""")

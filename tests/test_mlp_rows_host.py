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

"""An error that an earlier HIP call of the program left behind (a failed
allocation, say), on a HIP runtime without a device: cycles report it before
their first kernel, not between the kernels of a cycle, whose half would then
have run; the call after it runs."""
from fake_hip import run_fake  # noqa: F401


def test_cycles_report_it_before_their_first_kernel(run_fake):
    run_fake("""
L = pa.lib()
for text in (wd.sedov_rect(20, cstop=100), wd.sedov_rect(500, cstop=100), wd.noh_pie(9, 7, cstop=100)):
    with pa.Problem(text) as pb:
        pb.set_tuning("graph", 0)
        for mode in (pa.MODE_TASKS, pa.MODE_FUSED, pa.MODE_MIXED):
            for n in (2, 20):
                pb.launch(n, mode)
                clear()
                fake.error = 2
                assert L.pennant_launch_cycles(pb._h, n, mode) == 2, (mode, n)
                assert not any("k_tile" in k or "k_cycle" in k for k in names()), names()
                pb.launch(n, mode)
with pa.Batch([wd.sedov_rect(20, cstop=100), wd.noh_pie(9, 7, cstop=100)]) as b:
    for mode in (pa.MODE_FUSED, pa.MODE_MIXED):
        b.launch(2, mode)
        clear()
        fake.error = 2
        assert L.pennant_batch_launch_cycles(b._h, 2, mode) == 2, mode
        assert names() == [], names()
        b.launch(2, mode)
""")

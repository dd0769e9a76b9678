"""How cycles in pieces are launched, on a HIP runtime without a device."""
from fake_hip import run_fake  # noqa: F401


def test_one_piece_takes_the_launches_of_a_problem(run_fake):
    """A run in one piece launches what a problem's separate passes launch; a
    run in several one kernel a phase."""
    run_fake("""
for text in (wd.sedov_rect(20, cstop=100), wd.noh_pie(9, 7, cstop=100)):
    for mode in (pa.MODE_FUSED, pa.MODE_MIXED):
        with pa.Problem(text) as pb:
            pb.set_tuning("tiles", 0)
            clear()
            pb.run(5, mode)
            want = names()
        with pa.Pieces(text, 1) as p:
            clear()
            p.run(5, mode)
            assert names() == want, (names(), want)
        with pa.Pieces(text, 4) as p:
            clear()
            p.run(5, mode)
            assert sum("k_pred_pieces" in n for n in names()) == 5 and len(names()) == 30, names()
""")

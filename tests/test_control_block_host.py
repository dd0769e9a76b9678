"""The control block's copy to the host, which every synchronisation makes, on a
HIP runtime without a device: a whole number of 16 bytes (others are copied by a
slower kernel)."""
from fake_hip import run_fake  # noqa: F401


def test_the_copy_of_a_synchronisation(run_fake):
    run_fake("""
with pa.Problem(wd.sedov_rect(5, cstop=9)) as pb:
    pb.sync()
    assert fake.copied >= 96 and fake.copied % 16 == 0, fake.copied
with pa.Batch([wd.sedov_rect(5, cstop=9)] * 3) as b:
    b.sync()
    assert fake.copied >= 288 and fake.copied % 48 == 0, fake.copied
""")

"""A run in one piece, whose cycles are launched as a problem's: the problem's
state and scalars bit for bit, over changes of form and reads of the fields in
between."""
import numpy as np
import pytest

import pennant_amd as pa
from pennant_amd import decks as wd

pytestmark = pytest.mark.gpu

STATE = ("px", "pu", "zr", "ze", "zp", "zetot", "zwrate", "zvol")


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


@pytest.mark.parametrize("text", [wd.sedov_rect(29, cstop=70), wd.noh_pie(70, 81, cstop=60, dtinit=1e-4)],
                         ids=["rect", "pie"])
def test_one_piece_is_one_problem(text):
    with pa.Problem(text) as one, pa.Pieces(text, 1) as pp:
        one.set_tuning("tiles", 0)
        for n, mode in ((3, pa.MODE_MIXED), (20, pa.MODE_FUSED), (17, pa.MODE_MIXED), (1, pa.MODE_FUSED),
                        (100, pa.MODE_MIXED)):
            assert one.run(n, mode) == pp.run(n, mode)
            a, b = one.scalars(), pp.scalars()
            assert all(bits(a[k]) == bits(b[k]) for k in a), (n, mode)
            for f in STATE:
                assert np.array_equal(bits(one.get(f)), bits(pp.get(f))), (n, mode, f)

"""Lines above 512 cells in y and z, whose workgroups take neighbouring lines of
one segment (and, where the lines are no multiple of them, lines of two), and
compact lines of two blocks with more than two rows a lane, against the oracle
with the bars of test_gpu_sweep_forms.py."""
import pytest

import nuc3d_amd as G
from test_gpu_sweep_forms import test_rhs_matches_oracle as check

pytestmark = pytest.mark.gpu

CASES = [
    # n, rank grid, scheme, viscous scheme, splitting
    ((11, 1022, 13), (1, 2, 1), G.CRWENO5, G.CD6, G.LF),       # 4 lines a workgroup, two waves a line
    ((13, 11, 1022), (1, 1, 2), G.CRWENO5, G.CD8, G.AUSM),     # 2 lines
    ((11, 600, 13), (1, 2, 1), G.HCCS, G.CD6, G.LF),
    ((13, 11, 600), (1, 1, 2), G.HCCS, G.CD8, G.AUSM),
    ((11, 13, 766), (1, 1, 2), G.HCCS77, G.CD6, G.AUSMP),
    ((12, 10, 768), (1, 1, 6), G.CRWENO5, G.CD6, G.LF),        # a rank grid inside segments
    ((11, 1024, 13), (1, 1, 1), G.WENO5JS, G.CD6, G.LF),       # one wave a line
    ((13, 11, 765), (1, 1, 1), G.WENO7JS, G.CD8, G.AUSM),
    ((128, 66, 200), (2, 1, 2), G.HCCS, G.CD6, G.LF),
    ((200, 128, 12), (2, 2, 1), G.CRWENO5, G.CD8, G.AUSM),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}-s{c[2]}-v{c[3]}-r{c[4]}")
def test_rhs_matches_oracle(case):
    check(case)

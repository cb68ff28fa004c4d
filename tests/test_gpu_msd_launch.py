"""MSD launches at the edges of the rules that choose them: more blocks than one
launch can hold."""
import numpy as np
import pytest

from analisi_amd import capi
from gpu_util import make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("skip", [1, 4])
def test_blocks_in_ranges(skip):
    """290,000 blocks of 240 values: finishing them takes more than 2^32 threads."""
    nb, n, nt = 290000, 4, 60
    ot, dt = make_case(43, 60, 12, 9.0, [1.0 / nt] * nt, 0.1)
    primo = [b % 5 for b in range(nb)]
    b = capi.DeviceBlocks(dt, primo, [n] * nb, msd=True, msd_skip=skip, msd_tmax=4, use_graph=False)
    b.run()
    per = b.msd_results()[2]
    for p in range(5):
        one = capi.msd(dt, skip, 4, False, False, n, p)
        assert (per[p::5] == one).all()

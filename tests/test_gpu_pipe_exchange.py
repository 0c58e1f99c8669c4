"""The pipelined sweep's exchange at the workgroup counts where it changes: every workgroup sums all partials (up to 16),
one workgroup reduces four slots (17 to 31), two slots (from 32), and as many workgroups as there are compute units."""
import pytest

import _oracle as orc
import test_gpu_pipe as tp
from _data import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("workgroups", [15, 16, 17, 18, 31, 32, 33, 63, 64, 65, 128, 255, 256])
@pytest.mark.parametrize("layout", [orc.DENSE, orc.RAGGED], ids=["dense", "ragged"])
def test_exchange_at_its_borders(gpu_lib, layout, workgroups):
    pr = make_problem(16 * workgroups - 3, 150, seed=500 + workgroups, causal_frac=0.2)   # slices of 16 individuals
    o, h = tp.pair(pr, layout, workgroups=workgroups)
    assert h.stats()["workgroups"] == workgroups
    tp.sweeps(o, h, layout)
    h.close()

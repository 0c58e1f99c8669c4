"""The dense table's column sums on the device: formed from value counts while the running sum stays in one binade,
added one by one where it leaves it. Equal bit for bit to the host builder, which adds every individual in order."""
import numpy as np
import pytest

import bayesrrcmd_amd as brr

pytestmark = pytest.mark.gpu


# around the 64 individuals of a lane and the 4,096 of a wave's trip; common and rare variants (long stretches of
# equal values, sums that stay at zero for long), a column of one value, ties (a mean with few bits), all missing
@pytest.mark.parametrize("n", [2, 63, 64, 65, 127, 4095, 4096, 4097, 8193, 30011])
@pytest.mark.parametrize("miss", [0.0, 0.02, 0.7])
def test_ordered_sums(gpu_lib, n, miss):
    rng = np.random.default_rng(n)
    cols = []
    for p in (0.5, 0.1, 0.003, 0.0):
        for _ in range(3):
            d = rng.binomial(2, p, n)
            c = np.where(d == 2, 0, np.where(d == 1, 2, 3)).astype(np.uint8)
            c[rng.random(n) < miss] = 1
            cols.append(c)
    cols.append(np.tile(np.array([0, 3], dtype=np.uint8), n)[:n])          # mean 1: squares are 1
    cols.append(np.tile(np.array([2, 3, 3, 3], dtype=np.uint8), n)[:n])    # mean 1/4
    cols.append(np.repeat(np.array([3, 0], dtype=np.uint8), [n - n // 3, n // 3]))
    cols.append(np.full(n, 1, dtype=np.uint8))
    cb = (n + 3) // 4
    codes = np.zeros((len(cols), 4 * cb), dtype=np.uint8)
    codes[:, :n] = np.stack(cols)
    q = codes.reshape(len(cols), cb, 4)
    bed = q[..., 0] | q[..., 1] << 2 | q[..., 2] << 4 | q[..., 3] << 6
    with np.errstate(all="ignore"):
        want = brr.build_dense(bed, n)
    with brr.HipSweep(n, len(cols), 4, layout=brr.LAYOUT_DENSE_2BIT) as h:
        h.load_bed(brr.bed_file_image(bed), brr.LAYOUT_DENSE_2BIT)
        got = h.marker_tables()
    same = got.view(np.uint64) == np.asarray(want).view(np.uint64)
    assert np.all(same | (np.isnan(got) & np.isnan(want)))

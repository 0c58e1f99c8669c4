"""The dense table's column sums where additions are ties: values half a unit of the running sum off, whose rounding
depends on the last bit that the additions before left. Columns are chosen on the host for that, in sizes that a wave
sums. Equal bit for bit to the host builder, which adds every individual in order."""
import math

import numpy as np
import pytest

import bayesrrcmd_amd as brr

pytestmark = pytest.mark.gpu


def squares(n, n1, n2, nm):
    """The addends of a column's squared norm by code (0: dosage 2, 1: missing, 2: dosage 1, 3: dosage 0), as the builder
    forms them when no call is missing; with missing calls its column mean is a sum in order, so they are estimates."""
    mean = (n1 + 2.0 * n2) / (n - nm)
    cm = (n1 + 2.0 * n2 + nm * mean) / n
    return [(2.0 - cm) ** 2, (mean - cm) ** 2, (1.0 - cm) ** 2, cm * cm]


def ties(codes, x):
    """Additions that are ties, and 64-individual stretches with one after the sum's first 512 individuals."""
    acc, count, late = 0.0, 0, set()
    for i, c in enumerate(codes):
        v = x[c]
        if acc > v > 0.0:
            unit = math.ulp(acc)
            if math.fmod(v, unit) == 0.5 * unit:
                count += 1
                if i >= 512:
                    late.add(i // 64)
        acc += v
    return count, len(late)


def tied_at(x, counts, n):
    """A value that a tenth of the individuals have is a tie while the sum is that of 600 to n individuals."""
    mean = sum(v * c for v, c in zip(x, counts)) / n
    for e in range(int(math.log2(600 * mean)), int(math.log2(n * mean)) + 1):
        unit = math.ulp(2.0 ** e)
        for v, c in zip(x, counts):
            if c > n // 10 and math.fmod(v, unit) == 0.5 * unit:
                return True
    return False


@pytest.mark.parametrize("n", [8193, 20011])
@pytest.mark.parametrize("missing", [False, True], ids=["complete", "missing"])
def test_sums_with_ties(gpu_lib, n, missing):
    rng = np.random.default_rng(n + missing)
    cols, seen = [], 0
    while len(cols) < 40:
        p = rng.uniform(0.02, 0.5)
        n2, n1 = int(n * p * p), int(2 * n * p * (1 - p)) + int(rng.integers(0, 64))
        nm = int(rng.integers(1, n // 20)) if missing else 0
        seen += 1
        assert seen < 100_000
        counts = (n2, nm, n1, n - n1 - n2 - nm)
        if counts[3] <= 0 or not tied_at(squares(n, n1, n2, nm), counts, n):
            continue
        c = np.repeat(np.array([0, 1, 2, 3], dtype=np.uint8), counts)
        cols.append(rng.permutation(c))
    found = [ties(c, squares(n, int((c == 2).sum()), int((c == 0).sum()), int((c == 1).sum()))) for c in cols]
    if not missing:
        assert sum(late >= 8 for _, late in found) >= 20, found     # long stretches of ties in most columns
    cb = (n + 3) // 4
    codes = np.zeros((len(cols), 4 * cb), dtype=np.uint8)
    codes[:, :n] = np.stack(cols)
    q = codes.reshape(len(cols), cb, 4)
    bed = q[..., 0] | q[..., 1] << 2 | q[..., 2] << 4 | q[..., 3] << 6
    want = brr.build_dense(bed, n)
    with brr.HipSweep(n, len(cols), 4, layout=brr.LAYOUT_DENSE_2BIT) as h:
        h.load_bed(brr.bed_file_image(bed), brr.LAYOUT_DENSE_2BIT)
        got = h.marker_tables()
    assert np.array_equal(got.view(np.uint64), np.asarray(want).view(np.uint64))

"""Fingerprint histogram bins where the single-precision estimate cannot
decide: distances on and next to bin edges, equal clusters, the top value,
for few and many bins, against the reference's arithmetic (gen_flat_hists and
get_bin, calc_histograms.cpp:251-259, 351-489) in numpy.  Counts are equal."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [2, 3, 4])
@pytest.mark.parametrize("nbin", [1, 7, 100, 1024, 1025, 8192])
def test_bins(model_dir, nb, nbin):
    import chimes_calculator_amd as cc
    m = cc.GpuModel(os.path.join(model_dir, "co_2b3b4b.txt"))
    P = nb * (nb - 1) // 2
    maxd = (P * 4.0) ** 0.5 + 1.0
    binw = maxd / nbin
    rng = np.random.default_rng(nbin + nb)
    e1 = rng.uniform(-1, 1, (300, P))
    e2 = rng.uniform(-1, 1, (520, P))
    # one coordinate apart by whole bins, some nudged by an ulp; the top value
    k = rng.integers(0, max(1, int(2.0 / binw)), 200)
    e1[:200] = 0.0
    e2[:200] = 0.0
    e2[:200, 0] = k * binw
    e2[50:100, 0] = np.nextafter(e2[50:100, 0], 10.0)
    e2[100:150, 0] = np.nextafter(e2[100:150, 0], -10.0)
    e2[200, :] = 0.0
    e2[200, 0] = maxd
    e1[200:, 1:] *= 0.03  # every distance below maxd
    e1[200:, 0] = 0.3 + 0.1 * e1[200:, 0]
    s = np.zeros((300, 520))
    for q in range(P):
        d = e1[:, None, q] - e2[None, :, q]
        s = s + d * d
    tot = np.sqrt(s)
    b = np.floor(tot / binw).astype(int)
    b[tot == maxd] -= 1
    assert b.min() >= 0 and b.max() < nbin
    counts, ns, _ = m.fp_histogram(nb, e1, e2, nbin=nbin)
    assert np.array_equal(counts, np.bincount(b.reshape(-1), minlength=nbin)) and ns == 300 * 520
    m.close()

"""FP32-mixed one-cluster-per-lane kernels where their tiles end: batches whose
triplet and quadruplet lists are shorter than a wavefront, a little past one
workgroup, and past the size at which a wavefront takes four tiles (groups of
every type tuple in between, every dimension the kernel takes), against the
FP64 evaluation of the same batch.

Tolerance: FP32 polynomials and inner sums are within a few 1e-7 of FP64 per
term; the model's terms add to forces of order 1 and the worst cancellation
seen over the reference force fields is below 1e-5 of the largest force, so
1e-5 of the largest component holds the rounding and is far below a missed,
doubled or misplaced cluster.  A configuration's bits are the same alone and
inside the batch (exact sums).
"""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# list slots from which a wavefront takes four tiles: 4096 workgroups of four
# wavefronts, four tiles of 64 each
FOUR_TILES = 256 * 4096 * 4


@pytest.mark.parametrize("model,nconf,natoms", [
    ("co_2b3b4b", 1, 8),        # a few clusters
    ("co_2b3b4b", 3, 37),
    ("co_2b3b4b", 420, 256),    # past 4096 workgroups of four tiles in the triplet list
    ("carbon_16_10_4", 2, 125),
])
def test_tiles(model_dir, model, nconf, natoms):
    import chimes_calculator_amd as cc
    from chimes_calculator_amd import workloads as W
    m = cc.GpuModel(os.path.join(model_dir, model + ".txt"))
    rng = np.random.default_rng(natoms)
    el = ("C", "O") if model.startswith("co") else ("C", "C")
    cfgs = [W.co_config(rng, natoms, 3.2 if nconf > 100 else 2.0, 0.5, elements=el) for _ in range(nconf)]
    v = cc.get_variants()
    cc.set_variants(2, 2)
    try:
        E, F, S = cc.eval_batch(m, cfgs, precision=cc.MIXED)
        if nconf > 100:
            assert min(m.counts()[1:]) > FOUR_TILES
        e1, f1, s1 = cc.eval_batch(m, cfgs[-1:], precision=cc.MIXED)
    finally:
        cc.set_variants(*v)
    E0, F0, S0 = cc.eval_batch(m, cfgs)
    assert np.array_equal(e1, E[-1:]) and np.array_equal(f1[0], F[-1]) and np.array_equal(s1[0], S[-1])
    F, F0 = np.concatenate(F), np.concatenate(F0)
    assert np.abs(E - E0).max() <= 1e-5 * np.abs(E0).max()
    assert np.abs(F - F0).max() <= 1e-5 * np.abs(F0).max()
    assert np.abs(S - S0).max() <= 1e-5 * np.abs(S0).max()
    m.close()


@pytest.mark.parametrize("D3,D4", [(d, 0) for d in range(2, 14)] + [(3, 2), (3, 3), (3, 4)])
def test_every_dimension(tmp_path, D3, D4):
    """Every instance of the kernel over a list past the four-tile length,
    its last tile partial, against the FP64 evaluation (tolerance as above),
    and with equal bits against single configurations, whose lists take one
    tile per wavefront."""
    import chimes_calculator_amd as cc
    from chimes_calculator_amd import workloads as W
    md = W.Model("c%d_%d" % (D3, D4), ["C"], (6, D3, D4), (4.5, 4.0, 3.5 if D4 else 0.0), {frozenset(("C",)): 0.6},
                 seed=D3)
    m = cc.GpuModel(md.write(str(tmp_path / "c.txt")))
    rng = np.random.default_rng(D3)
    base = [W.co_config(rng, 256, 3.2, 1.0, elements=("C", "C")) for _ in range(16)] \
        + [W.co_config(rng, 61, 3.0, 1.0, elements=("C", "C"))]
    cfgs = (base * 17)[:200 if not D4 else 280]
    v = cc.get_variants()
    cc.set_variants(2, 2)
    try:
        E, F, S = cc.eval_batch(m, cfgs, precision=cc.MIXED)
        n = m.counts()[2 if D4 else 1]
        assert n > FOUR_TILES and n % 64
        for k in (0, 16, len(cfgs) - 1):
            e, f, s = cc.eval_batch(m, cfgs[k:k + 1], precision=cc.MIXED)
            assert e[0] == E[k] and np.array_equal(f[0], F[k]) and np.array_equal(s[0], S[k]), k
    finally:
        cc.set_variants(*v)
    E0, F0, S0 = cc.eval_batch(m, cfgs)
    F, F0 = np.concatenate(F), np.concatenate(F0)
    assert np.abs(E - E0).max() <= 1e-5 * np.abs(E0).max()
    assert np.abs(F - F0).max() <= 1e-5 * np.abs(F0).max()
    assert np.abs(S - S0).max() <= 1e-5 * np.abs(S0).max()
    m.close()

"""Batches above 16384 atoms take other list kernels than small ones (one
wavefront per neighbour owner, four placement owners per wavefront).  Every
sum is exact and each owner's image order is canonical, so a configuration's
bits are the same in the batch and alone: compared with equality for owners
with few and with more than 64 images, and for models with few and many
cluster groups."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("what", ["co", "crowded", "groups"])
def test_batch_equals_alone(model_dir, tmp_path, what):
    import chimes_calculator_amd as cc
    from chimes_calculator_amd import workloads as W
    rng = np.random.default_rng(7)
    if what == "co":
        pf = os.path.join(model_dir, "co_2b3b4b.txt")
        cfgs = [W.co_config(rng, int(n), 2.5, 0.5) for n in rng.integers(8, 300, 125)]
    elif what == "crowded":  # about 155 images an owner
        pf = os.path.join(model_dir, "carbon_wide.txt")
        base = [W.dense_carbon(natoms=n, seed=n) for n in (48, 64, 71)]
        cfgs = [base[k % 3] for k in range(280)]
    else:  # 11 triplet and 16 quadruplet groups
        m = W.Model("cho", ["C", "H", "O"], (6, 3, 2), (4.5, 4.0, 3.5),
                    {frozenset((a, b)): 0.5 for a in "CHO" for b in "CHO"}, seed=3)
        pf = m.write(str(tmp_path / "cho.txt"))
        cfgs = []
        for n in rng.integers(8, 300, 125):
            pos, ty, cell = W.co_config(rng, int(n), 2.0, 0.6)
            cfgs.append((pos, ["H" if rng.random() < 0.3 else t for t in ty], cell))
    assert sum(len(c[0]) for c in cfgs) > 16384
    m = cc.GpuModel(pf)
    E, F, S = cc.eval_batch(m, cfgs)
    for k in (0, 1, 2, len(cfgs) // 2, len(cfgs) - 1):
        e, f, s = cc.eval_batch(m, [cfgs[k]])
        assert e[0] == E[k] and np.array_equal(f[0], F[k]) and np.array_equal(s[0], S[k]), k
    m.close()

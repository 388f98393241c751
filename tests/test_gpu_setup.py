"""The one-launch set-up of small batches at the edges of its range: around
1024 atoms, several configurations, a box with more cells than it takes, and
replicated small cells.  The same configuration beside a large one goes
through the separate launches; the bits are equal (exact sums, canonical
lists)."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,box,small", [
    ([2], None, False), ([2, 3, 5], None, True), ([1023], None, False), ([1024], None, False), ([1025], None, False),
    ([500, 524], None, False), ([500, 525], None, False), ([8] * 40, None, False),
    ([64], 40.0, False), ([64], 150.0, False),
])
def test_setup_paths(model_dir, sizes, box, small):
    import chimes_calculator_amd as cc
    from chimes_calculator_amd import workloads as W
    m = cc.GpuModel(os.path.join(model_dir, "co_2b3b4b.txt"))
    rng = np.random.default_rng(sum(sizes))
    cfgs = []
    for n in sizes:
        pos, ty, cell = W.co_config(rng, n, 2.2, 0.5)
        cfgs.append((pos, ty, cell if box is None else np.diag([box] * 3)))
    big = W.co_config(rng, 1100, 2.2, 0.5)
    E, F, S = cc.eval_batch(m, cfgs, small=small)
    E1, F1, S1 = cc.eval_batch(m, cfgs + [big], small=small)
    for k in range(len(cfgs)):
        assert E[k] == E1[k] and np.array_equal(F[k], F1[k]) and np.array_equal(S[k], S1[k]), k
    m.close()

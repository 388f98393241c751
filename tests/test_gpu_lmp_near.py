"""The pair style's per-step selection of the listed clusters within the
cutoffs, at the sizes where it can go wrong: no list entry within the cutoffs,
a handful, and lists past one and several workgroup spans of 2048 entries
(the lengths are asserted), against the oracle's loops over the whole lists.

Tolerance: both sides evaluate the same FP64 terms and differ by roundings of
a few ulp per term, so 1e-10 of the largest component is far above the error
and far below any missed or doubled cluster.
"""
import numpy as np
import pytest

from chimes_calculator_amd import workloads as W
from lmp_setup import LmpSystem
from oracle_bindings import LmpOracle

pytestmark = pytest.mark.gpu


SPAN = 2048


@pytest.mark.parametrize("natoms,box,skin,spans,inside", [
    (4, 13.0, 1.0, (0, 0), False),     # far apart: empty lists
    (3, 11.0, 3.5, (1, 0), False),     # one entry, outside
    (12, 11.0, 3.0, (1, 1), False),    # entries of both bodies, none inside
    (40, 11.0, 1.5, (1, 1), True),
    (64, 11.0, 1.5, (2, 2), True),     # past one span
    (110, 11.0, 1.0, (7, 5), True),    # several spans, both bodies
])
def test_near_selection(tmp_path, natoms, box, skin, spans, inside):
    from chimes_calculator_amd import GpuModel, LmpPair
    pf = W.MODELS["co_2b3b4b"].write(str(tmp_path / "co.txt"))
    rng = np.random.default_rng(natoms)
    ns = int(np.ceil(natoms ** (1.0 / 3.0)))
    a = box / ns
    sites = (np.stack(np.meshgrid(*[np.arange(ns)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) * a
    x = sites[rng.choice(len(sites), natoms, replace=False)] + rng.uniform(-0.15, 0.15, (natoms, 3)) * a
    typ = rng.integers(1, 3, natoms).astype(np.int32)
    O = LmpOracle(pf)
    S = LmpSystem(x, typ, np.arange(1, natoms + 1, dtype=np.int32), np.zeros(3), np.full(3, box), [0, 1], O.rc2(),
                  skin)
    trips, quads = O.build_lists(S)
    assert tuple(-(-len(c) // SPAN) for c in (trips, quads)) == spans
    p = S.x[np.asarray(trips, int).reshape(-1, 3)]
    d = np.stack([p[:, a] - p[:, b] for a, b in ((0, 1), (0, 2), (1, 2))])
    assert (np.sqrt((d * d).sum(-1)) < 4.0).all(0).any() == inside
    model = GpuModel(pf)
    P = LmpPair(model, {1: W.MASS["C"], 2: W.MASS["O"]})
    out = P.compute(S.x, S.type, S.tag, S.ilist, S.numneigh, S.nbr_off, S.nbr, ago=0, skin=skin)
    R = O.compute(S, trips, quads)
    for name, got, ref in zip(("f", "eng", "virial", "eatom", "vatom"), out,
                              (R.f, R.eng, R.virial, R.eatom, R.vatom)):
        got, ref = np.asarray(got, float), np.asarray(ref, float)
        assert np.abs(got - ref).max() <= 1e-10 * max(np.abs(ref).max(), 1e-300), (name, len(trips), len(quads))
    P.close()
    model.close()

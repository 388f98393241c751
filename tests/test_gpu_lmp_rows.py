"""The pair style's list kernels where their bit rows end: owners whose filtered
rows hold just below, at and above 64 and 256 candidates and the most of 512
(word and working-set edges, the large form included), in both forms, list
entries compared exactly with the oracle's.  Candidate counts and row lengths
are asserted."""
import numpy as np
import pytest

from chimes_calculator_amd import workloads as W
from lmp_setup import LmpSystem
from oracle_bindings import LmpOracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natoms,rc4,shell", [
    (2, 3.5, 0), (64, 3.5, 0), (65, 3.5, 0), (66, 0.9, 0),  # one wavefront per owner, up to 64 candidates
    (2, 3.5, 90), (64, 3.5, 90), (65, 3.5, 90), (66, 0.9, 90),  # the row-wise form: 63, 64, 65 candidates
    (129, 2.0, 0), (257, 1.2, 0), (258, 1.2, 0), (259, 1.2, 0), (513, 0.8, 0),
])
def test_rows(tmp_path, natoms, rc4, shell):
    from chimes_calculator_amd import GpuModel, LmpPair
    # natoms atoms in a ball of 2.2 A about the one of the lowest tag, which so
    # has natoms - 1 candidates; shell: atoms that lengthen its row beyond the
    # many-body cutoffs
    m = W.Model("ball", ["C"], (4, 3, 3), (5.0, 4.0, rc4), {frozenset(("C",)): 0.05}, seed=natoms)
    pf = m.write(str(tmp_path / "ball.txt"))
    rng = np.random.default_rng(natoms)
    v = rng.normal(size=(natoms + shell, 3))
    r = np.where(np.arange(natoms + shell) < natoms, 2.2 * rng.random(natoms + shell) ** (1.0 / 3.0), 4.5)
    r[0] = 0.0
    x = 10.0 + v / np.linalg.norm(v, axis=1)[:, None] * r[:, None]
    tag = np.concatenate([[1], rng.permutation(natoms + shell - 1) + 2]).astype(np.int32)
    O = LmpOracle(pf)
    S = LmpSystem(x, np.ones(len(x), np.int32), tag, np.zeros(3), np.full(3, 20.0), [0], O.rc2(), 0.0, shuffle_seed=1)
    keep = 1 if shell else 3 if natoms > 100 else natoms  # owners: the lists of a few low tags are long enough
    S.ilist = np.argsort(S.tag[: S.nlocal])[:keep].astype(np.int32)
    rows = [S.nbr[S.nbr_off[i]:S.nbr_off[i + 1]] for i in S.ilist]
    S.inum, S.nbr = keep, np.concatenate(rows).astype(np.int32)
    S.nbr_off = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    near = np.linalg.norm(S.x[rows[0]] - S.x[S.ilist[0]], axis=1) < 4.0
    assert near.sum() == natoms - 1 and len(rows[0]) == natoms + shell - 1
    assert (len(S.nbr) > 80 * S.inum) == (shell > 0 or natoms > 100)
    trips, quads = O.build_lists(S)
    model = GpuModel(pf)
    P = LmpPair(model, {1: W.MASS["C"]})
    P.build_mb_neighlists(S.x, S.tag, S.ilist, S.numneigh, S.nbr_off, S.nbr, skin=0.0)
    g3, g4 = P.mb_lists()
    assert np.array_equal(g3, trips) and np.array_equal(g4, quads), (len(trips), len(quads))
    P.close()
    model.close()


@pytest.mark.parametrize("ball,orders", [(0, (4, 3, 3)), (64, (4, 3, 3)), (65, (4, 3, 3)), (66, (4, 3, 3)),
                                         (66, (4, 3, 0)), (258, (4, 3, 3)), (513, (4, 3, 0))])
def test_short_rows(tmp_path, ball, orders):
    """Rows of a few entries on average, which the one-wavefront list form
    takes, beside a ball whose centre, of the lowest tag, has ball - 1
    candidates: the most that form holds, and the owners it leaves to both
    working sets of the row-wise form."""
    from chimes_calculator_amd import GpuModel, LmpPair
    rc4 = 2.0 if ball < 100 else 0.8
    m = W.Model("short", ["C"], orders, (5.0, 4.0, rc4 if orders[2] else 0.0), {frozenset(("C",)): 0.05}, seed=ball)
    pf = m.write(str(tmp_path / "short.txt"))
    rng = np.random.default_rng(ball)
    grid = (np.stack(np.meshgrid(*[np.arange(6)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) * 8.0
    grid = grid[np.linalg.norm(grid - 28.0, axis=1) > 7.0]
    x = np.concatenate([g + rng.uniform(-0.6, 0.6, (k, 3)) for g, k in zip(grid, rng.integers(1, 6, len(grid)))])
    tag = rng.permutation(len(x)).astype(np.int32) + 1 + ball
    if ball:
        v = rng.normal(size=(ball, 3))
        r = 2.2 * rng.random((ball, 1)) ** (1.0 / 3.0)
        r[0] = 0.0
        x = np.concatenate([28.0 + v / np.linalg.norm(v, axis=1)[:, None] * r, x])
        tag = np.concatenate([1 + np.arange(ball, dtype=np.int32), tag])
    O = LmpOracle(pf)
    S = LmpSystem(x, np.ones(len(x), np.int32), tag, np.zeros(3), np.full(3, 48.0), [0], O.rc2(), 0.0, shuffle_seed=2)
    keep = np.concatenate([np.arange(min(ball, 3)), np.arange(ball, len(x))]).astype(np.int32)
    rows = [S.nbr[S.nbr_off[i]:S.nbr_off[i + 1]] for i in keep]
    S.ilist, S.inum, S.nbr = keep, len(keep), np.concatenate(rows).astype(np.int32)
    S.nbr_off = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    assert len(S.nbr) <= 80 * S.inum
    if ball:
        near = np.linalg.norm(S.x[rows[0]] - S.x[0], axis=1) < 4.0
        assert near.sum() == ball - 1 and (S.tag[rows[0][near]] > 1).all()
    trips, quads = O.build_lists(S)
    assert len(trips) > 50 and (len(quads) > 0) == (orders[2] > 0)
    model = GpuModel(pf)
    P = LmpPair(model, {1: W.MASS["C"]})
    P.build_mb_neighlists(S.x, S.tag, S.ilist, S.numneigh, S.nbr_off, S.nbr, skin=0.0)
    g3, g4 = P.mb_lists()
    assert np.array_equal(g3, trips) and np.array_equal(g4, quads), (len(trips), len(quads))
    P.close()
    model.close()


@pytest.mark.parametrize("natoms", [2, 64, 65, 66, 129, 300])
def test_pair_rows(tmp_path, natoms):
    """1-/2-body forces and every tally of owners with up to natoms - 1
    partners: the queue's batches of 64 and, past 256 atoms, contributions that
    find the workgroup's table full.  Tolerance: the same FP64 terms on both
    sides, a few ulp of rounding each, so 1e-10 of the largest component."""
    from chimes_calculator_amd import GpuModel, LmpPair
    m = W.Model("ball2", ["C"], (6, 0, 0), (5.0, 0.0, 0.0), {frozenset(("C",)): 0.05}, seed=natoms)
    pf = m.write(str(tmp_path / "ball2.txt"))
    rng = np.random.default_rng(natoms)
    v = rng.normal(size=(natoms, 3))
    x = 10.0 + v / np.linalg.norm(v, axis=1)[:, None] * 2.4 * rng.random((natoms, 1)) ** (1.0 / 3.0)
    O = LmpOracle(pf)
    S = LmpSystem(x, np.ones(natoms, np.int32), rng.permutation(natoms).astype(np.int32) + 1, np.zeros(3),
                  np.full(3, 20.0), [0], O.rc2(), 1.0, shuffle_seed=1)
    R = O.compute(S, np.zeros((0, 3), np.int32), np.zeros((0, 4), np.int32))
    model = GpuModel(pf)
    P = LmpPair(model, {1: W.MASS["C"]})
    out = P.compute(S.x, S.type, S.tag, S.ilist, S.numneigh, S.nbr_off, S.nbr, ago=0, skin=1.0)
    for name, got, ref in zip(("f", "eng", "virial", "eatom", "vatom"), out,
                              (R.f, R.eng, R.virial, R.eatom, R.vatom)):
        got, ref = np.asarray(got, float), np.asarray(ref, float)
        assert np.abs(got - ref).max() <= 1e-10 * max(np.abs(ref).max(), 1e-300), name
    P.close()
    model.close()

"""DILU sweeps of structured boxes against the oracle, bit for bit, over the
shapes where a tile's schedule changes: tiles of every width the schedule
picks, partial tiles on either edge, lines shorter than a group of steps,
every sequential axis, boxes of one tile and of many, a single row of cells."""
import numpy as np
import pytest

import oracle_bind as ob

pytestmark = pytest.mark.gpu

SHAPES = [(3, 2, 2), (40, 1, 1), (7, 5, 1), (64, 64, 1), (200, 130, 1), (11, 9, 5), (33, 17, 9), (17, 33, 70),
          (20, 90, 31), (90, 66, 3), (150, 40, 40)]


def box(n, seed, symmetric=False):
    """Random diagonally dominant matrix on the faces of an n box."""
    rng = np.random.default_rng(seed)
    N = int(np.prod(n))
    c = np.arange(N)
    ijk = (c % n[0], (c // n[0]) % n[1], c // (n[0] * n[1]))
    has = np.stack([ijk[a] + 1 < n[a] for a in range(3)], axis=1)
    cell, axis = np.nonzero(has)
    nb = cell + np.take((1, n[0], n[0] * n[1]), axis)
    upper = -rng.uniform(0.1, 2.0, len(cell))
    lower = upper.copy() if symmetric else -rng.uniform(0.1, 2.0, len(cell))
    diag = 0.3 - np.bincount(cell, upper, N) - np.bincount(nb, lower, N)
    return dict(nCells=N, nFaces=len(cell), symmetric=symmetric, lAddr=cell.astype(np.int32),
                uAddr=nb.astype(np.int32), lower=lower, upper=upper, diag=diag, source=rng.standard_normal(N),
                psi=rng.standard_normal(N))


# boxes of several flat or nearly flat tiles, whose inboxes have sides that no
# neighbour delivers to
FLAT = [(300, 66, 1), (70, 300, 1), (1, 90, 150), (200, 130, 2), (64, 200, 3), (3, 70, 400)]


@pytest.mark.parametrize("n", SHAPES + FLAT, ids=lambda n: "x".join(map(str, n)))
def test_sweeps_match_oracle(gpu, n):
    # two boxes in one system, so that tiles of both are swept by one launch
    regions = [box(n, 1), box((n[0], n[2], n[1]), 2, symmetric=True)]
    O = ob.OracleSystem.from_arrays(regions, [])
    A = gpu.CoupledFvMatrix(0)
    A.add_system(regions, [])
    A.commit()
    rD = O.dilu_factor()
    assert np.array_equal(A.dilu_factor(), np.concatenate(rD))
    rng = np.random.default_rng(3)
    for _ in range(2):
        r = [rng.standard_normal(R["nCells"]) for R in regions]
        assert np.array_equal(A.precondition(r), np.concatenate(O.dilu_precondition(rD, r)))
    # the fused p and s updates, in a solve that starts and ends on its own
    psi, perf = O.solve(tol=1e-10, maxIter=40)
    got = A.solve(tolerance=1e-10, maxIter=40)[0]
    assert got.n_iterations == perf["nIterations"] and got.final_residual == perf["finalResidual"]
    assert np.array_equal(np.concatenate(A.psi(0)), np.concatenate(psi))
    A.close()


def _committed(gpu, regions):
    A = gpu.CoupledFvMatrix(0)
    A.add_system(regions, [])
    A.commit()
    return A


def test_wait_limit_is_of_one_wait(gpu):
    # two flat tiles of 60000 steps: the second waits for a few steps of the
    # first at a time, some 3000 polls in the whole sweep
    regions = [box((60000, 66, 1), 4)]
    A = _committed(gpu, regions)
    assert len(set(A.dilu_tiles())) > 1
    rD = A.dilu_factor()
    r = [np.random.default_rng(5).standard_normal(R["nCells"]) for R in regions]
    w = A.precondition(r)
    A.set_wait_limit(1000)
    assert np.array_equal(A.dilu_factor(), rD)
    assert np.array_equal(A.precondition(r), w)
    A.close()


def test_expired_wait_fails_the_call(gpu):
    # a tile waits for its neighbour's first 64 steps: more than one poll
    regions = [box((300, 130, 1), 6)]
    A = _committed(gpu, regions)
    A.dilu_factor()
    r = [np.random.default_rng(7).standard_normal(R["nCells"]) for R in regions]
    w = A.precondition(r)
    A.set_wait_limit(1)
    # the sweep's wait, then the factor's, whose values must not be kept
    for call in (lambda: A.precondition(r), A.dilu_factor):
        with pytest.raises(Exception, match="wait expired"):
            call()
        A.set_wait_limit(1 << 20)
        assert np.array_equal(A.precondition(r), w)
        A.set_wait_limit(1)
    for polls in (0, (1 << 20) + 1):
        with pytest.raises(Exception, match="polls must be"):
            A.set_wait_limit(polls)
    A.close()


@pytest.mark.parametrize("n", [(3, 2, 2), (12, 9, 7), (33, 17, 9), (17, 33, 70), (20, 90, 31)],
                         ids=lambda n: "x".join(map(str, n)))
def test_spmv_of_values_that_are_not_finite(gpu, n):
    # a face with a zero coefficient still multiplies its neighbour's value,
    # and a cell without a neighbour multiplies nothing
    R = box(n, 8)
    rng = np.random.default_rng(9)
    for side in ("lower", "upper"):
        R[side][rng.random(R["nFaces"]) < 0.3] = 0.0
    O = ob.OracleSystem.from_arrays([R], [])
    A = _committed(gpu, [R])
    x = rng.standard_normal(R["nCells"])
    x[rng.random(len(x)) < 0.05] = 0.0
    assert np.array_equal(A.spmv([x]), np.concatenate(O.amul([x])))
    for k, v in enumerate((np.inf, -np.inf, np.nan)):
        bad = np.random.default_rng(10 + k).choice(len(x), max(1, len(x) // 300), replace=False)
        y = x.copy()
        # the corners too: cells that lack neighbours on three sides
        y[np.concatenate([bad, [0, len(x) - 1]])] = v
        want = np.concatenate(O.amul([y]))
        assert np.array_equal(A.spmv([y]), want, equal_nan=True)
    A.close()

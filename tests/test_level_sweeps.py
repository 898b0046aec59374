"""DILU factor and sweeps of regions without box structure against the oracle,
bit for bit: level groups narrower and wider than a workgroup, dependencies
that lie further back than the LDS ring, every record width, a chain beside
them, and the FP32 sweeps."""
import numpy as np
import pytest

import oracle_bind as ob
from test_box_sweeps import box

pytestmark = pytest.mark.gpu


def renumbered(R, perm):
    inv = np.argsort(perm)
    a, b = perm[R["lAddr"]], perm[R["uAddr"]]
    swap = a > b
    lo, up = np.where(swap, R["upper"], R["lower"]), np.where(swap, R["lower"], R["upper"])
    a, b = np.minimum(a, b), np.maximum(a, b)
    o = np.lexsort((b, a))
    return dict(R, lAddr=a[o].astype(np.int32), uAddr=b[o].astype(np.int32), lower=lo[o], upper=up[o],
                **{f: R[f][inv] for f in ("diag", "source", "psi")})


def front(n, jitter, seed=4):
    """A box numbered along its diagonal front."""
    c = np.arange(int(np.prod(n)))
    key = c % n[0] + (c // n[0]) % n[1] + c // (n[0] * n[1]) + np.random.default_rng(seed).uniform(0, jitter, len(c))
    perm = np.empty(len(c), dtype=np.int64)
    perm[np.argsort(key, kind="stable")] = c
    return renumbered(box(n, seed), perm)


def shuffled(n, seed=5):
    return renumbered(box(n, seed), np.random.default_rng(seed).permutation(int(np.prod(n))))


def graph(N, most, seed=6):
    """A random graph with up to `most` lower and upper neighbours per cell."""
    rng = np.random.default_rng(seed)
    up = np.zeros(N, dtype=int)
    faces = set()
    for c in range(1, N):
        for l in rng.integers(max(0, c - 200), c, most):
            if up[l] < most and (l, c) not in faces:
                faces.add((int(l), c))
                up[l] += 1
    f = np.array(sorted(faces), dtype=np.int32)
    u, lo = -rng.uniform(0.1, 1.0, len(f)), -rng.uniform(0.1, 1.0, len(f))
    diag = 0.5 - np.bincount(f[:, 0], u, N) - np.bincount(f[:, 1], lo, N)
    return dict(nCells=N, nFaces=len(f), symmetric=False, lAddr=f[:, 0].copy(), uAddr=f[:, 1].copy(), lower=lo, upper=u,
                diag=diag, source=rng.standard_normal(N), psi=rng.standard_normal(N))


def ladder(widths, seed=8):
    """Levels of the given widths: each cell has a lower neighbour in the
    level before its own (at most six to one), and most of those from the 20th
    level on one among the first cells as well."""
    rng = np.random.default_rng(seed)
    start = np.concatenate([[0], np.cumsum(widths)])
    faces, up = set(), np.zeros(start[-1], dtype=int)
    for lv in range(1, len(widths)):
        for i in range(widths[lv]):
            c = int(start[lv]) + i
            before = int(start[lv - 1]) + (i % widths[lv - 1])
            far = int(rng.integers(0, start[min(20, lv)]))
            for l in (before, far) if lv >= 20 and up[far] < 5 else (before,):
                faces.add((l, c))
                up[l] += 1
    f = np.array(sorted(faces), dtype=np.int32)
    u, lo = -rng.uniform(0.1, 1.0, len(f)), -rng.uniform(0.1, 1.0, len(f))
    N = int(start[-1])
    diag = 0.5 - np.bincount(f[:, 0], u, N) - np.bincount(f[:, 1], lo, N)
    return dict(nCells=N, nFaces=len(f), symmetric=False, lAddr=f[:, 0].copy(), uAddr=f[:, 1].copy(), lower=lo, upper=u,
                diag=diag, source=rng.standard_normal(N), psi=rng.standard_normal(N))


def layers(width, n, most):
    """n levels of `width` cells, each cell with `most` lower neighbours in
    the level before."""
    c = np.arange(width)
    f = np.concatenate([np.stack([(lv - 1) * width + (c + 7 * j) % width, lv * width + c], axis=1)
                        for lv in range(1, n) for j in range(most)])
    f = f[np.lexsort((f[:, 1], f[:, 0]))].astype(np.int32)
    rng = np.random.default_rng(9)
    u, lo = -rng.uniform(0.1, 1.0, len(f)), -rng.uniform(0.1, 1.0, len(f))
    N = n * width
    diag = 0.5 - np.bincount(f[:, 0], u, N) - np.bincount(f[:, 1], lo, N)
    return dict(nCells=N, nFaces=len(f), symmetric=False, lAddr=f[:, 0].copy(), uAddr=f[:, 1].copy(), lower=lo, upper=u,
                diag=diag, source=rng.standard_normal(N), psi=rng.standard_normal(N))


def strip():
    """Three blocks side by side, numbered one after the other: a chain."""
    n = (60, 20, 1)
    c = np.arange(1200)
    i, j = c % 60, c // 60
    b = i // 20
    return renumbered(box(n, 7), b * 400 + j * 20 + i % 20)


WIDE_AMONG_NARROW = [900] * 25 + [30] * 40 + [150, 800, 4000, 9000] + [100] * 30 + [500, 2500, 9500, 500]
KINDS = {"beyond_the_ring": ["spread"], "spread_levels": ["spread", "spread"], "spread_twelve_neighbours": ["spread"],
         "spread_beside_others": ["spread", "chain", "box", "levels", "spread"],
         "with_chain_and_box": ["chain", "box", "levels"]}   # of the regions, if not all level groups

CASES = {
    "narrow_levels": lambda: [front((23, 11, 9), 0.9)],
    "levels_over_a_workgroup": lambda: [front((60, 45, 40), 0.5), front((40, 33, 9), 2.5)],
    "beyond_the_ring": lambda: [shuffled((40, 40, 30))],
    # a wide level, then levels that most waves of the workgroup have no part
    # in, with rows read back long after they have left the ring
    "far_rows_of_narrow_levels": lambda: [ladder([1000] + [300] * 110), ladder([2000, 700] + [64] * 300 + [300] + [900] * 5)],
    "wide_among_narrow_levels": lambda: [ladder(WIDE_AMONG_NARROW)],
    # spread over the device: a level of a few slices, of one row, of many
    "spread_levels": lambda: [layers(6000, 4, 3), ladder([5000, 5000, 1, 5, 25, 125, 600, 3000, 15000, 17001])],
    "spread_twelve_neighbours": lambda: [layers(5000, 3, 12)],
    "spread_beside_others": lambda: [shuffled((40, 40, 30)), strip(), box((30, 17, 15), 8), front((12, 12, 12), 0.9),
                                     layers(6000, 5, 2)],
    "six_neighbours": lambda: [shuffled((13, 11, 7))],
    "twelve_neighbours": lambda: [graph(1500, 12), front((17, 9, 8), 0.5)],
    "with_chain_and_box": lambda: [strip(), box((30, 17, 5), 8), front((12, 12, 12), 0.9)],
}


@pytest.mark.parametrize("name", list(CASES))
def test_level_sweeps_match_oracle(gpu, name):
    regions = CASES[name]()
    O = ob.OracleSystem.from_arrays(regions, [])
    A = gpu.CoupledFvMatrix(0)
    A.add_system(regions, [])
    A.commit()
    rD = O.dilu_factor()
    assert np.array_equal(A.dilu_factor(), np.concatenate(rD))
    rng = np.random.default_rng(3)
    r = [rng.standard_normal(R["nCells"]) for R in regions]
    w = np.concatenate(O.dilu_precondition(rD, r))
    assert np.array_equal(A.precondition(r), w)
    # FP32 records: rounding of the coefficients and of the recurrence
    w32 = A.precondition_fp32(np.concatenate(r).astype(np.float32))
    assert np.linalg.norm(w32 - w) < 1e-5 * np.linalg.norm(w)
    psi, perf = O.solve(tol=1e-10, maxIter=30)
    got = A.solve(tolerance=1e-10, maxIter=30)[0]
    assert got.n_iterations == perf["nIterations"]
    assert np.array_equal(np.concatenate(A.psi(0)), np.concatenate(psi))
    # every wave, tile, group and spread region appears in the trace of both sweeps
    for sweep in A.trace_dilu():
        assert len(sweep) == A.layout_info(0)["waves"]
        assert np.all(sweep[:, 1] >= sweep[:, 0]) and np.all(sweep[:, 0] >= 0) and np.all(sweep[:, 3] > 0)
    A.close()

"""Box tiles in batches whose records are wider than a box needs (another
region's cells have more neighbours), and mixed precision on every schedule of
regions without box structure, against the oracle."""
import numpy as np
import pytest

import oracle_bind as ob
from test_box_sweeps import box
from test_gpu_parity import _masked_dilu, rel
from test_level_sweeps import front, graph, ladder, layers, shuffled, strip

pytestmark = pytest.mark.gpu

# systems of a batch: lists of regions
BATCHES = {
    # several tiles per box, K = 6 and 12
    "tiles_six": lambda: [[box((30, 33, 17), 1), shuffled((13, 11, 7))], [box((70, 130, 1), 2)]],
    "tiles_twelve": lambda: [[box((20, 33, 18), 3), graph(1500, 12), box((17, 9, 25), 4, symmetric=True)]],
    # one tile per box
    "lone_six": lambda: [[box((40, 8, 6), 5), box((50, 7, 1), 6)], [shuffled((13, 11, 7))]],
    "lone_twelve": lambda: [[box((90, 5, 4), 7)], [graph(1500, 12), box((8, 8, 90), 8)]],
    # chains, level groups (with rows beyond the LDS ring) and spread levels
    "chain": lambda: [[strip(), strip()]],
    "level_groups": lambda: [[front((23, 11, 9), 0.9)], [ladder([1000] + [300] * 110), shuffled((13, 11, 7))]],
    "spread": lambda: [[shuffled((40, 40, 30))], [layers(6000, 4, 3), strip(), box((30, 17, 15), 9)]],
}


@pytest.mark.parametrize("name", list(BATCHES))
def test_batches_match_oracle(gpu, name):
    batch = BATCHES[name]()
    oracles = [ob.OracleSystem.from_arrays(regions, []) for regions in batch]
    A = gpu.CoupledFvMatrix(0)
    for regions in batch:
        A.add_system(regions, [])
    A.commit()
    rng = np.random.default_rng(3)
    for q, (regions, O) in enumerate(zip(batch, oracles)):
        rD = O.dilu_factor()
        assert np.array_equal(A.dilu_factor(sys=q), np.concatenate(rD))
        off, tiles = O.offsets(), A.dilu_tiles(sys=q)
        keep = []
        for g, R in enumerate(O.regions):
            t = tiles[off[g]:off[g + 1]]
            tl, tu = t[R["lAddr"]], t[R["uAddr"]]
            keep.append(~((tl >= 0) & (tu >= 0) & (tl != tu)))
        for _ in range(2):
            r = [rng.standard_normal(R["nCells"]) for R in regions]
            w = np.concatenate(O.dilu_precondition(rD, r))
            assert np.array_equal(A.precondition(r, sys=q), w)
            # FP32 records: rounding of the coefficients and of the recurrence
            assert rel(A.precondition_inner(np.concatenate(r), "DILU", sys=q).astype(np.float64), w) < 1e-5
            assert rel(A.precondition_inner(np.concatenate(r), "tileDILU", sys=q).astype(np.float64),
                       _masked_dilu(O, keep, r)) < 1e-5
    perf = A.solve(tolerance=1e-10, maxIter=300)
    for q, O in enumerate(oracles):
        psi, want = O.solve(tol=1e-10, maxIter=300)
        assert perf[q].n_iterations == want["nIterations"] and want["converged"]
        assert np.array_equal(np.concatenate(A.psi(q)), np.concatenate(psi))
    for inner in ("tileDILU", "DILU"):
        A.reset_psi()
        perf = A.solve(tolerance=1e-10, maxIter=300, precision="mixed", innerPreconditioner=inner)
        for q, O in enumerate(oracles):
            psi, _ = O.solve(tol=1e-10, maxIter=300)
            assert perf[q].converged and rel(np.concatenate(A.psi(q)), np.concatenate(psi)) <= 1e-8
    A.close()

"""Batches whose box sweeps are in flight together: the rule that keeps their
tiles from starving each other, and several batches solved at once."""
import os
import subprocess
import threading

import numpy as np
import pytest

from test_box_sweeps import box

HERE = os.path.dirname(os.path.abspath(__file__))


def test_gate_rule(tmp_path):
    exe = str(tmp_path / "gate")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-o", exe, os.path.join(HERE, "sweep_gate_check.cpp")],
                   check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout


@pytest.mark.gpu
def test_batches_of_many_tiles_at_once(gpu):
    # 432 tiles each: an XCD holds 96 and gets 54 of each of the four
    def batch(seed):
        A = gpu.CoupledFvMatrix(0)
        for q in range(48):
            A.add_system([box((24, 24, 24), 100 * seed + q)], [])
        A.commit()
        assert sum(len(set(A.dilu_tiles(q))) for q in range(48)) > 384
        return A
    batches = [batch(s) for s in range(4)]

    def solve(A):
        A.reset_psi()
        its = [p.n_iterations for p in A.solve(solver="BiCGStab", tolerance=1e-10, maxIter=40)]
        return its, [np.concatenate(A.psi(q)) for q in range(48)]
    alone = [solve(A) for A in batches]
    got = [None] * 4

    def run(k):
        for _ in range(3):
            got[k] = solve(batches[k])
    threads = [threading.Thread(target=run, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(4):
        assert got[k] is not None and got[k][0] == alone[k][0]
        assert all(np.array_equal(a, b) for a, b in zip(got[k][1], alone[k][1]))
        batches[k].close()

"""The curl update's threads walk along i on FP64 grids from a million cells;
the last walk of a grid is short where its planes do not divide.  Bitwise the
oracle's there, and alone like in a batch with a grid that does not walk.
"""
import pytest

import gamera_op as go
from parity import exact_mismatches, run_oracle


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n", [
    (go.SINUSOID_BLAST, (102, 99, 101)),   # 103 planes: a walk of three last
    (go.SINUSOID_SPHERE, (8, 360, 360)),   # 9 planes: a walk of one last
    (go.DIPOLE_SHELL, (129, 88, 90))])     # 130 planes: two last
def test_walk_matches_oracle(kind, n):
    print("ct walk", kind, n, flush=True)
    P = go.Problem(kind, 64, *n)
    try:
        S = go.Solver(P, 0)
        Q = go.Solver(P, 0)
        O = run_oracle(P, 2)
        P.reseed(64)
        P.device_open(0)
        P.device_step(2)
        P.device_fetch()
        assert exact_mismatches(P, O) == 0
    finally:
        P.close()
    P = go.Problem(go.DIPOLE_SHELL, 65, 16, 12, 16)
    small = go.Solver(P, 0)
    P.close()
    B = go.Batch()
    try:
        B.add(Q)
        B.add(small)
        B.step(2)
        S.step(2)
        (p0, b0), (p1, b1) = S.state(), Q.state()
        assert all((x == y).all() for x, y in zip(p0 + b0, p1 + b1))
    finally:
        B.close()
        for s in (S, Q, small):
            s.close()

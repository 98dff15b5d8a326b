"""Marches of a merged launch at every length the rule gives.

Grids of 5e4 to 3e5 cells whose marched extents the length does not divide (FP64 and
FP32-bulk faces per thread beside each).  Bitwise the oracle's in FP64; in
FP32-bulk bitwise what the launches apart and a batch give.
"""
import numpy as np
import pytest

import gamera_op as go
from parity import exact_mismatches, run_oracle

SIZES = [(go.DIPOLE_SHELL, (40, 31, 45)),       # 4 and 2
         (go.SINUSOID_SPHERE, (41, 40, 39)),    # 5 and 2
         (go.SINUSOID_BLAST, (61, 43, 37)),     # 8 and 4
         (go.WALL_BOX, (45, 52, 50)),           # 9 and 4
         (go.VARYING_B0_BOX, (40, 50, 71)),     # 10 and 4
         (go.SINUSOID_SPHERE, (131, 125, 8)),   # 11 and 5, packed k tiles
         (go.SINUSOID_SPHERE, (56, 55, 57)),    # 12 and 6
         (go.SINUSOID_SPHERE, (67, 66, 68))]    # 12 and 10, the edge fields apart


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n", SIZES)
def test_fp64_matches_oracle(kind, n):
    print("merge length", kind, n, flush=True)
    P = go.Problem(kind, 72, *n, full_b0=True)
    try:
        O = run_oracle(P, 3)
        P.device_open(0)
        P.device_step(3)
        P.device_fetch()
        assert exact_mismatches(P, O) == 0
        assert P.device_scalars()["time"] == O.scalar("time_sim")
    finally:
        P.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n", SIZES)
def test_fp32_merged_apart_and_batched(kind, n):
    print("merge length, FP32-bulk", kind, n, flush=True)
    P = go.Problem(kind, 73, *n)
    S = [go.Solver(P, 1) for _ in range(3)]
    P.close()
    B = go.Batch()
    try:
        S[1].set_tuning(go.TUNE_MERGE, 0)
        B.add(S[2])
        S[0].step(4)
        S[1].step(4)
        B.step(4)
        (p0, b0), (p1, b1), (p2, b2) = (s.state() for s in S)
        for x, y, z in zip(p0 + b0, p1 + b1, p2 + b2):
            assert np.array_equal(x, y) and np.array_equal(x, z)
    finally:
        B.close()
        for s in S:
            s.close()

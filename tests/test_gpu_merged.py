"""Merged launches of small grids, and packed k tiles.

A small grid stepped alone runs all sweeps in one launch and all edge fields in
another; a march length asked for (set_tuning) or a batch runs them apart.  Both
must be bitwise the oracle's in FP64 and bitwise each other's in FP32-bulk, at
the k extents where the k sweep changes form: 6 faces per row (the smallest),
31 to 33 around the last packed width, 64 and 65 around the tile, and a row of
one tile and leftover columns.
"""
import numpy as np
import pytest

import gamera_op as go
from parity import exact_mismatches, run_oracle

SIZES = [(go.SINUSOID_SPHERE, (6, 7, 5)), (go.SINUSOID_SPHERE, (8, 5, 7)),
         (go.SINUSOID_BLAST, (9, 6, 8)), (go.SINUSOID_SPHERE, (7, 6, 15)),
         (go.SINUSOID_SPHERE, (6, 5, 30)), (go.DIPOLE_SHELL, (8, 6, 31)),
         (go.SINUSOID_SPHERE, (5, 6, 32)), (go.SINUSOID_SPHERE, (5, 6, 63)),
         (go.VARYING_B0_BOX, (6, 5, 64)), (go.WALL_BOX, (9, 8, 70))]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n", SIZES)
def test_merged_and_apart_match_oracle(kind, n):
    steps = 4
    print("merged", kind, n, flush=True)
    P = go.Problem(kind, 61, *n, full_b0=True)
    try:
        O = run_oracle(P, steps)
        for apart in (False, True):
            P.reseed(61)
            P.device_open(0)
            if apart:
                P.set_tuning(go.TUNE_CHUNK, 2)
                P.set_tuning(go.TUNE_EMF_CHUNK, 2)
            P.device_step(steps)
            P.device_fetch()
            assert exact_mismatches(P, O) == 0, apart
            assert P.device_scalars()["time"] == O.scalar("time_sim")
    finally:
        P.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n", SIZES)
def test_fp32_merged_apart_and_batched(kind, n):
    P = go.Problem(kind, 62, *n)
    S = [go.Solver(P, 1) for _ in range(3)]
    P.close()
    B = go.Batch()
    try:
        S[1].set_tuning(go.TUNE_CHUNK, 2)
        S[1].set_tuning(go.TUNE_EMF_CHUNK, 2)
        B.add(S[2])
        S[0].step(5)
        S[1].step(5)
        B.step(5)
        (p0, b0), (p1, b1), (p2, b2) = (s.state() for s in S)
        for x, y, z in zip(p0 + b0, p1 + b1, p2 + b2):
            assert np.array_equal(x, y) and np.array_equal(x, z)
    finally:
        B.close()
        for s in S:
            s.close()

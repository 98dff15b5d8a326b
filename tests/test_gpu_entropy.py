"""The entropy channel is carried from the first p_S that is not 0.

A single cell with p_S != 0 (a corner, the cell next to the leftover k faces
of a 64-face tile, a cell inside) must make every stage carry the channel: the
device then matches the oracle as in test_gpu_failure.py (rho, v, p and face B
bitwise, p_S through the device's pow to relative L1 <= 1e-12).  In a batch the
members that carry it and those that do not keep their solo results.
"""
import numpy as np
import pytest

import gamera_op as go
from parity import active_slices, run_oracle


@pytest.mark.gpu
@pytest.mark.parametrize("n,at", [((12, 8, 10), (4, 4, 4)), ((8, 12, 64), (11, 15, 67)),
                                  ((16, 12, 8), (10, 9, 8))])
def test_one_cell(n, at):
    print("entropy in one cell", n, at, flush=True)
    P = go.Problem(go.SINUSOID_SPHERE, 51, *n, full_b0=True)
    try:
        P.gas(5)[at] = 0.25
        O = run_oracle(P, 6)
        P.device_open(0)
        P.device_step(6)
        P.device_fetch()
        cell, faces = active_slices(P)
        for f in range(5):
            assert np.array_equal(P.gas(f)[cell], O.gas[f][cell]), f
        for f in range(3):
            assert np.array_equal(P.gem(f)[faces[f]], O.gem[f][faces[f]]), f
        d, o = P.gas(5)[cell], O.gas[5][cell]
        assert np.count_nonzero(o) > 1 and np.array_equal(d == 0.0, o == 0.0)
        assert np.abs(d - o).sum() <= 1e-12 * np.abs(o).sum()
        flux = P.debug_fetch(2, 5)[cell]
        assert np.count_nonzero(flux) > 0
    finally:
        P.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_batch_members_keep_their_own(precision):
    alone, members = [], []
    for kind, seed, n in [(go.SINUSOID_SPHERE, 52, (16, 12, 8)), (go.ENTROPY_BOX, 53, (16, 12, 8)),
                          (go.DIPOLE_SHELL, 54, (12, 8, 16))]:
        P = go.Problem(kind, seed, *n)
        alone.append(go.Solver(P, precision))
        members.append(go.Solver(P, precision))
        P.close()
    B = go.Batch()
    try:
        for S in members:
            B.add(S)
        B.step(7)
        for q, (a, m) in enumerate(zip(alone, members)):
            a.step(7)
            (pa, ba), (pm, bm) = a.state(), m.state()
            assert all(np.array_equal(x, y) for x, y in zip(pa + ba, pm + bm)), q
            assert (np.abs(pm[5]).max() > 0.0) == (q == 1)
    finally:
        B.close()
        for S in alone + members:
            S.close()

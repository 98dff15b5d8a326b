"""What the prologue's scan must find, and what it may cost.

The entropy channel is carried from the first step if p_S is not 0 anywhere.  The scan's blocks walk many rows on grids of more than 2048
blocks of 256 points (100x70x70: 108 planes of 24): a single cell in the first,
the last and a later walked row must be found.  What carries the channel is seen
from the outside: p_S of one cell has spread to its neighbours after a step.
"""
import ctypes
import time

import numpy as np
import pytest

import gamera_op as go


def arrays(P):
    return [np.array(P.gas(f)) for f in range(6)], [np.array(P.gem(f)) for f in range(3)]


def set_state(S, prim, bface, prev=None):
    """gk_set_state + gk_prologue; prev: (primitives, face B) of the level before"""
    def ptrs(a):
        return (ctypes.c_void_p * len(a))(*[x.ctypes.data for x in a])

    hist = [ptrs(a) for a in prev] if prev else [None, None]
    assert S.op.gk_set_state(S.handle, ptrs(prim), ptrs(bface), *hist) == 0
    t0 = time.perf_counter()
    assert S.op.gk_prologue(S.handle, ctypes.c_double(1e-3 if prev else 0.0)) == 0
    return time.perf_counter() - t0


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_one_cell_in_a_walked_row_is_found(precision):
    n = (100, 70, 70)
    P = go.Problem(go.SINUSOID_SPHERE, 81, *n)
    S = go.Solver(P, precision)
    prim, bface = arrays(P)
    P.close()
    try:
        for at in [(4, 4, 4), (103, 73, 73), (90, 41, 66), (99, 4, 73)]:
            print("p_S at", at, flush=True)
            prim[5][:] = 0.0
            prim[5][at] = 0.25
            set_state(S, prim, bface)
            S.step(1)
            ps = S.state()[0][5][4:-5, 4:-5, 4:-5]
            assert np.count_nonzero(ps) > 1
    finally:
        S.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_previous_level_alone_moves_nothing(precision):
    """A restart whose p_S is not 0 in the level before only, which the scan does
    not read: every face state lies between the current cells of the face.  The
    twin has one more cell with p_S, at the current level and out of reach of the
    first, which makes it carry the channel."""
    n = (40, 24, 16)
    P = go.Problem(go.SINUSOID_SPHERE, 82, *n)
    S, T = go.Solver(P, precision), go.Solver(P, precision)
    prim, bface = arrays(P)
    P.close()
    try:
        prev = [x.copy() for x in prim]
        prev[5][10, 12, 10] = 0.25
        set_state(S, prim, bface, (prev, bface))
        twin = [x.copy() for x in prim]
        twin[5][34, 12, 10] = 0.25
        set_state(T, twin, bface, (prev, bface))
        S.step(2)
        T.step(2)
        (ps, bs), (pt, bt) = S.state(), T.state()
        assert all(np.array_equal(x, y) for x, y in zip(ps[:5] + bs, pt[:5] + bt))
        near = (slice(4, 22), slice(4, 28), slice(4, 20))  # two steps reach 8 cells at most
        assert np.array_equal(ps[5][near], pt[5][near])
        assert np.count_nonzero(pt[5]) > 1 and np.count_nonzero(ps[5]) == 0
    finally:
        S.close()
        T.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_back_to_zero(precision):
    """A solver whose p_S was not 0 and is set to 0 steps like a fresh one."""
    n = (16, 12, 40)
    P = go.Problem(go.ENTROPY_BOX, 83, *n)
    S = go.Solver(P, precision)
    prim, bface = arrays(P)
    P.gas(5)[:] = 0.0
    F = go.Solver(P, precision)
    P.close()
    try:
        S.step(5)
        assert np.abs(S.state()[0][5]).max() > 0.0
        prim[5][:] = 0.0
        set_state(S, prim, bface)
        S.step(4)
        F.step(4)
        (ps, bs), (pf, bf) = S.state(), F.state()
        assert all(np.array_equal(x, y) for x, y in zip(ps + bs, pf + bf))
        assert not ps[5].any()
    finally:
        S.close()
        F.close()


@pytest.mark.gpu
def test_scan_costs_the_same_whatever_it_finds():
    """The prologue reads the same bytes with and without p_S: its best time of
    nine may differ by launch jitter (0.3 ms launches of which the scan is a
    seventh), not by a factor."""
    P = go.Problem(go.SINUSOID_SPHERE, 84, 128, 128, 128)
    S = go.Solver(P, 0)
    prim, bface = arrays(P)
    P.close()
    try:
        best = []
        for value in (0.0, 0.25):
            prim[5][:] = value
            best.append(min(set_state(S, prim, bface) for _ in range(9)))
        print("prologue ms without and with p_S", [x * 1e3 for x in best], flush=True)
        assert best[1] < 1.4 * best[0]
    finally:
        S.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("batched", [False, True])
def test_switched_on_in_mid_run(precision, batched):
    """A regular state without p_S that turns non-finite in its first step (eight
    planes of negative pressure: no real sound speed on either side of their
    faces): from then on the channel is carried.  The twin
    carries it from the start, for a cell with p_S out of reach: every field
    of the solver, its NaN among them, is the twin's."""
    n = (60, 16, 12)
    P = go.Problem(go.SINUSOID_SPHERE, 85, *n)
    S, T = go.Solver(P, precision), go.Solver(P, precision)
    prim, bface = arrays(P)
    P.close()
    B = go.Batch() if batched else None
    try:
        prim[4][8:16] = -1.0
        set_state(S, prim, bface)
        prim[5][48, 10, 9] = 0.25
        set_state(T, prim, bface)
        if batched:
            B.add(S)
            B.add(T)
        near = (slice(4, 32), slice(4, 20), slice(4, 16))
        for step in range(3):
            if batched:
                with pytest.raises(go.GkNonFinite):
                    B.step(1)
            else:
                for s in (S, T):
                    with pytest.raises(go.GkNonFinite):
                        s.step(1)
            (ps, bs), (pt, bt) = S.state(), T.state()
            for x, y in zip(ps[:5] + bs, pt[:5] + bt):
                assert np.array_equal(x, y, equal_nan=True), step
            assert np.array_equal(ps[5][near], pt[5][near], equal_nan=True), step
            assert np.isnan(ps[5][near]).any() and (pt[5][44:52] > 0.0).any()
    finally:
        if batched:
            B.close()
        S.close()
        T.close()

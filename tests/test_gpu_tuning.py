"""Launch shapes: what can be read from one solver can be set on another.

A small grid runs its sweeps and its edge fields merged.  Which form runs shows
in the stages that are timed: k_sweep_j and k_emf_k exist only apart.
"""
import itertools

import pytest

import gamera_op as go

PARAMS = [go.TUNE_CHUNK, go.TUNE_EMF_CHUNK, go.TUNE_EMF_STAGE, go.TUNE_MERGE]


def stages(S):
    S.enable_timing(True)
    S.step(1)
    S.enable_timing(False)
    return {k for k, v in S.kernel_times().items() if v > 0.0}


def merged(S):
    """(sweeps, edge fields) in one launch each"""
    names = stages(S)
    return "k_sweep_j" not in names, "k_emf_k" not in names


@pytest.fixture
def make():
    made = []

    def solver(precision=0, n=(16, 12, 10), kind=go.SINUSOID_SPHERE):
        P = go.Problem(kind, 71, *n)
        S = go.Solver(P, precision)
        P.close()
        made.append(S)
        return S

    yield solver
    for S in made:
        S.close()


@pytest.mark.gpu
@pytest.mark.parametrize("merge", [3, 2, 1, 0])
def test_values_read_and_set_again(make, merge):
    A = make()
    assert A.get_tuning(go.TUNE_MERGE) == 3 and merged(A) == (True, True)
    A.set_tuning(go.TUNE_MERGE, merge)
    want = merged(A)
    assert want == (bool(merge & 1), bool(merge & 2))
    values = [A.get_tuning(p) for p in PARAMS]
    for order in itertools.permutations(PARAMS):
        B = make()
        for p in order:
            B.set_tuning(p, values[p])
        assert [B.get_tuning(p) for p in PARAMS] == values, order
        assert merged(B) == want, order


@pytest.mark.gpu
def test_a_length_alone_takes_the_launches_apart(make):
    S = make(1)
    S.set_tuning(go.TUNE_CHUNK, 4)
    assert S.get_tuning(go.TUNE_MERGE) == 2 and merged(S) == (False, True)
    S.set_tuning(go.TUNE_EMF_CHUNK, 4)
    assert S.get_tuning(go.TUNE_MERGE) == 0 and merged(S) == (False, False)


@pytest.mark.gpu
def test_bits_a_grid_does_not_have_are_refused(make):
    S = make(0, (70, 68, 66))  # 314160 cells: its sweeps merge, its edge fields do not
    assert S.get_tuning(go.TUNE_MERGE) == 1
    for bad in (-1, 2, 3, 4):
        with pytest.raises(go.GkError):
            S.set_tuning(go.TUNE_MERGE, bad)
    assert S.get_tuning(go.TUNE_MERGE) == 1
    S.set_tuning(go.TUNE_MERGE, 0)
    assert merged(S) == (False, False)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_pick_does_not_depend_on_who_asked_first(make, precision):
    """A solver taken apart by hand and then autotuned leaves the same pick for
    later ones as one that was not touched: on these two grids of about 6000
    cells (shapes no other test tunes) the merged launches are far ahead."""
    n = (20, 18, 16 + precision)
    A = make(precision, n)
    for p in (go.TUNE_CHUNK, go.TUNE_EMF_CHUNK):
        A.set_tuning(p, 4)
    A.autotune(2)
    B = make(precision, n)
    assert B.autotune(0) > 0
    for S in (A, B):
        assert S.get_tuning(go.TUNE_MERGE) == 3 and merged(S) == (True, True)
    assert [A.get_tuning(p) for p in PARAMS] == [B.get_tuning(p) for p in PARAMS]
    C = make(precision, n)
    C.set_tuning(go.TUNE_MERGE, 0)
    assert C.autotune(0) > 0 and merged(C) == (True, True)


@pytest.mark.gpu
def test_pick_is_for_the_kernels_it_was_timed_on(make):
    """A background field per point runs other kernels on the same shape."""
    n = (22, 18, 14)
    A = make(0, n)
    assert A.autotune(1) > 0
    B = make(0, n, go.VARYING_B0_BOX)
    before = [B.get_tuning(p) for p in PARAMS]
    assert B.autotune(0) == 0 and [B.get_tuning(p) for p in PARAMS] == before
    C = make(0, n)
    assert C.autotune(0) == A.get_tuning(go.TUNE_CHUNK)


@pytest.mark.gpu
@pytest.mark.parametrize("merge", [3, 0])
def test_every_stage_can_be_timed_by_name(make, merge):
    """Stages that run inside another's launch answer to their own names too."""
    S = make(0, (12, 10, 16))
    S.set_tuning(go.TUNE_MERGE, merge)
    for name in ("k_begin", "k_sweep_i", "k_sweep_j", "k_vstrip_j", "k_sweep_k", "k_emf_i", "k_emf_j",
                 "k_emf_k", "k_ct", "k_cell", "k_ghost", "k_mags"):
        S.time_stage(name)
        S.step(2)
        assert {k for k, v in S.kernel_times().items() if v > 0.0} == {name}, name
    S.time_stage("no such stage")
    S.step(1)
    assert not any(S.kernel_times().values())

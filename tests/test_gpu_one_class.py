"""FP32-bulk grids whose classes differ only below FP32 resolution.

Such a grid is given one class, and with it the uniform-table kernels.  The same
grid is handed over a second time with one table row changed that no cell reads
(axis 0, face 0, the last class pair), which keeps all its classes: both must step bitwise
alike.
"""
import numpy as np
import pytest

import gamera_op as go

STRIDE, B0_FIELDS = 18, 24


def descriptor(P):
    """The descriptor blob, the byte offset of the reconstruction rows in it and
    the class pairs of each axis (header words 19 to 21 are the allocated
    extents, 22 to 27 the classes, 18 the B0 mode; the rows end where the class maps begin)."""
    blob = P.desc_blob()
    head = np.frombuffer(blob, np.int32, 28)
    N = [int(x) for x in head[19:22]]
    pairs = [int(head[22 + 2 * a] * head[23 + 2 * a]) for a in range(3)]
    end = len(blob) - 8 * sum(N)
    if head[18] == 2:  # a per-point background field follows
        end -= 8 * B0_FIELDS * N[0] * N[1] * N[2]
    return blob, end - 8 * STRIDE * sum(n * c for n, c in zip(N, pairs)), N, pairs


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n", [
    (go.SINUSOID_SPHERE, (6, 7, 5)), (go.WALL_BOX, (9, 8, 70)),
    (go.SINUSOID_BLAST, (61, 43, 37)), (go.SINUSOID_BLAST, (70, 11, 100))])
def test_one_class_steps_like_all_classes(kind, n):
    print("one class", kind, n, flush=True)
    P = go.Problem(kind, 63, *n)
    try:
        blob, at, N, pairs = descriptor(P)
        assert pairs[0] > 1, "this grid has one class already"
        off = at
        for n_a, c in zip(N, pairs):
            rows = np.frombuffer(blob, np.float64, n_a * c * STRIDE, off)
            rows = rows.reshape(n_a, c, STRIDE).astype(np.float32)
            assert (rows == rows[:, :1]).all()
            off += rows.size * 8
        prim = [np.array(P.gas(f)) for f in range(6)]
        bface = [np.array(P.gem(f)) for f in range(3)]
    finally:
        P.close()
    apart = bytearray(blob)
    row = np.frombuffer(apart, np.float64, STRIDE, at + 8 * STRIDE * (pairs[0] - 1))
    row[0] += 1.0
    S = [go.Solver.from_parts(b, prim, bface, 1) for b in (blob, bytes(apart))]
    try:
        for s in S:
            s.step(5)
        (p0, b0), (p1, b1) = (s.state() for s in S)
        assert all(np.array_equal(x, y) for x, y in zip(p0 + b0, p1 + b1))
        assert S[0].scalars()["time"] == S[1].scalars()["time"]
    finally:
        for s in S:
            s.close()

"""Which grids keep their table classes.

test_gpu_one_class.py compares a grid that is given one class with the same grid
that keeps all of them; that it does keep them shows in the tables' size (18 values
per face and class pair, in FP64 and FP32).
"""
import numpy as np
import pytest

import gamera_op as go
from test_gpu_one_class import STRIDE, descriptor


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(6, 7, 5), (61, 43, 37)])
def test_a_row_apart_keeps_all_classes(n):
    P = go.Problem(go.SINUSOID_BLAST, 64, *n)
    try:
        blob, at, N, pairs = descriptor(P)
        prim = [np.array(P.gas(f)) for f in range(6)]
        bface = [np.array(P.gem(f)) for f in range(3)]
    finally:
        P.close()
    extra = STRIDE * sum(f * (c - 1) for f, c in zip(N, pairs))
    assert extra > 0
    apart = bytearray(blob)
    np.frombuffer(apart, np.float64, STRIDE, at + 8 * STRIDE * (pairs[0] - 1))[0] += 1.0
    size = {}
    for name, b, precision in [("one", blob, 1), ("apart", bytes(apart), 1),
                               ("FP64", blob, 0), ("FP64 apart", bytes(apart), 0)]:
        S = go.Solver.from_parts(b, prim, bface, precision)
        size[name] = S.device_bytes()
        S.close()
    print(n, pairs, size, flush=True)
    assert size["apart"] - size["one"] == extra * 12  # 8 and 4 bytes a value
    assert size["FP64 apart"] == size["FP64"]  # FP64 keeps its classes in any case

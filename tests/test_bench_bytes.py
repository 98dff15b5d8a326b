"""The benchmark's compulsory bytes of a stage follow what its launch holds."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def test_merged_launches_count_all_their_stages():
    n = 60  # 61 faces along k: no leftover columns
    apart = {d: bench.kernel_alg_bytes("k_sweep_" + d, n) for d in "ijk"}
    assert bench.kernel_alg_bytes("k_sweep_i", n, 1) == sum(apart.values())
    assert bench.kernel_alg_bytes("k_emf_i", n, 2) == sum(
        bench.kernel_alg_bytes("k_emf_" + d, n) for d in "ijk")
    for merged in (0, 2):
        assert bench.kernel_alg_bytes("k_sweep_i", n, merged) == apart["i"]
    for merged in (0, 1):
        assert bench.kernel_alg_bytes("k_emf_i", n, merged) == bench.kernel_alg_bytes("k_emf_j", n)
    assert bench.kernel_alg_bytes("k_cell", n, 3) == bench.kernel_alg_bytes("k_cell", n)

"""The kernels that bench.py looks up in the committed counter summary are in it under the names that they have."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


@pytest.mark.parametrize("workload,kernel,K,V", [
    ("train", "fwd.fused_fwd", 64, 64), ("train", "fwd.fixup", 64, 64), ("train", "bwd.fused_ckpt", 64, 64), ("train", "bwd.fused_rev", 64, 64),
    ("train", "bwd.chunk_grad", 64, 64), ("fwd", "fwd.fused_fwd", 64, 64), ("varlen", "fwd.prep", 128, 128), ("varlen", "fwd.scan_fwd", 128, 128),
    ("varlen", "bwd.prep", 128, 128), ("varlen", "bwd.scan_pair", 128, 128), ("varlen", "bwd.chunk_grad", 128, 128), ("decode", "recurrent", 128, 128)])
def test_kernels_of_the_operators(bench, workload, kernel, K, V):
    assert bench.measured_traffic(workload, kernel, K, V) > 1e6


@pytest.mark.parametrize("rows", [8192, 262144])
def test_the_norm(bench, rows):
    # x, gate, do once and dx, dgate once, 1024 channels of 2 bytes; beside them only the weight gradient's partial rows; of the small shape some
    # stays in the last-level cache
    least = 5 * 2 * 1024 * rows
    assert 0.9 * least < bench.norm_traffic(rows) < 1.2 * least

"""The kernels that bench.py looks up in the committed counter summary are in it under the names that they have."""
import importlib.util
import json
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


def test_launches_of_other_kinds_are_not_taken(bench, tmp_path, monkeypatch):
    """Scans that leave something for a backward pass, and those of the HDLA parameterisation, whatever their place in the summary."""
    names = {"scan_out_kernel<128, 128, 2, 1, false>": 1, "scan_out_kernel<128, 128, 2, 2, false>": 2, "scan_out_kernel<128, 128, 2, 0, true>": 3, "scan_out_share_kernel<128, 128, 2, false>": 4,
             "scan_out_share_kernel<128, 128, 0, true>": 5, "scan_grad_kernel<128, 128, 2, true>": 6, "scan_grad_share_kernel<128, 128, true>": 7, "scan_rev_share_kernel<128, 128>": 8}
    (tmp_path / "profiles").mkdir()
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    for more, want in (({}, (None, None)), ({"scan_out_share_kernel<128, 128, 0, false>": 10, "scan_grad_share_kernel<128, 128, false>": 11}, (10, 11)),
                       ({"scan_out_kernel<128, 128, 4, 0, false>": 12, "scan_grad_kernel<128, 128, 4, false>": 13}, (12, 13))):
        table = {"varlen": {n: {"hbm_bytes_per_launch": b} for n, b in {**names, **more}.items()}}
        (tmp_path / "profiles" / "hbm_traffic.json").write_text(json.dumps(table))
        assert tuple(bench.measured_traffic("varlen", k, 128, 128) for k in ("fwd.scan_fwd", "bwd.scan_pair")) == want

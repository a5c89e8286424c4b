"""What the host hands to the graded live-row product (``gemm.rows_graded``): the workspace that its parts are chosen by."""

import os
import subprocess
import sys

import pytest
import torch

from speculators_amd import gemm


@pytest.fixture
def calls(monkeypatch):
    """``rows_graded`` of ``(M, N, K)`` on the host with the launch replaced: the parts and the workspace's bytes."""
    seen = {}
    monkeypatch.setattr(gemm._lib, "call", lambda name, *a: seen.update({name: a}))
    monkeypatch.setattr(gemm._lib, "stream_ptr", lambda device: 0)
    monkeypatch.setattr(gemm, "_workspaces", gemm._Workspaces())
    count, rows = torch.zeros(1, dtype=torch.int32), torch.zeros(40000, dtype=torch.int32)

    def run(m, n, k):
        a = torch.empty(m, 1, dtype=torch.bfloat16).expand(m, k)
        b = torch.empty(k, dtype=torch.bfloat16).expand(n, k)
        gemm.rows_graded(a, b, count, rows, torch.zeros(m), torch.ones(()), 1.0)
        *_, parts, ws, nbytes, _stream = seen["spx_gemm_bf16_rows_graded"]
        assert ws is None or ws.numel() * 4 >= nbytes
        return parts, nbytes

    return run


@pytest.mark.parametrize("m,n,k", [(4096, 1024, 8192), (888, 2048, 32000), (5000, 512, 56)])
def test_workspace_is_the_one_asked_for(calls, m, n, k):
    alone = calls(m, n, k)
    gemm._split_workspace(torch.device("cpu"), 2 * alone[1] // 4 + 65536)  # left behind by a larger product
    assert calls(m, n, k) == alone



@pytest.mark.parametrize("split,parts", [(None, 8), (1, 1), (2, 2), (3, 3), (4, 4), (8, 8)])
def test_parts_are_bounded_by_the_variable(split, parts):
    env = {k: v for k, v in os.environ.items() if k != "SPX_GEMM_SPLIT_PARTS"}
    if split is not None:
        env["SPX_GEMM_SPLIT_PARTS"] = str(split)
    run = [sys.executable, "-c", "from speculators_amd import gemm; print(gemm.LIVE_TAIL_PARTS if gemm.SPLIT_PARTS > 1 else 1)"]
    assert int(subprocess.run(run, env=env, check=True, capture_output=True, text=True).stdout) == parts

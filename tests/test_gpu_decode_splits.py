"""Small decode calls cut finer than ``split`` (fewer workgroups than the chip
holds): against the oracle at the edges of the splits, with gates around 1/2
(every later split stands) and near 0 (every split is recomputed), and with a
workspace that only has room for the caller's own split."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from cacheslide_amd import _hip
from cacheslide_amd.ccpe import ccpe_decode_paged, decode_workspace, decode_workspace_bytes
from oracle import ccpe as orc
from tests._helpers import acc_np, assert_close_bf16, fill_paged, paged_layout, seeded
from tests.test_gpu_ccpe import cope_on

pytestmark = pytest.mark.gpu


def setup(device, lens, hq, hkv, npos, low_gates=0.0):
    blocks, table, rows = paged_layout(lens, hkv, 16, 128, seed=sum(lens))
    cache = torch.zeros((blocks, hkv, 16, 256), dtype=torch.bfloat16)
    keys = [seeded((n, hkv, 128), 7 + i, dtype=torch.bfloat16) for i, n in enumerate(lens)]
    vals = [seeded((n, hkv, 128), 17 + i, dtype=torch.bfloat16) for i, n in enumerate(lens)]
    q = seeded((len(lens), hq, 128), 3, dtype=torch.bfloat16)
    if low_gates:                       # q.k / sqrt(128) around -7.2 low_gates: gates of 0.007 at 0.7
        q = q.abs()
        keys = [-(k.abs() * low_gates) for k in keys]
    fill_paged(cache, rows, keys, vals)
    e = seeded((128, npos), 5, scale=0.1)
    want = np.concatenate([orc.cope_attention(acc_np(q[i:i + 1]), acc_np(k), acc_np(v), e.numpy(),
                                              np.array([n - 1]))
                           for i, (n, k, v) in enumerate(zip(lens, keys, vals))])
    args = (q.to(device), cache.to(device), table.to(device), torch.tensor(lens, dtype=torch.int32, device=device),
            cope_on(device, 128, npos, table=e))
    return args, want


@pytest.mark.parametrize("npos", [64, 128])
@pytest.mark.parametrize("lens", [[1], [255], [256, 257], [384, 385, 511, 513], [1500], [4200, 37]])
def test_small_calls_match_the_oracle(device, lens, npos):
    args, want = setup(device, lens, 8, 2, npos)
    assert_close_bf16(ccpe_decode_paged(*args, max_context=max(lens)), want)


@pytest.mark.parametrize("lens", [[700], [1500, 129]])
def test_small_calls_with_low_gates(device, lens):
    args, want = setup(device, lens, 8, 1, 64, low_gates=0.7)
    assert_close_bf16(ccpe_decode_paged(*args, max_context=max(lens)), want)


def test_a_workspace_for_the_plain_split_is_taken(device):
    lens = [1500]
    args, want = setup(device, lens, 8, 2, 64)
    small = torch.empty(decode_workspace_bytes(1, 8, 1500, 1024), dtype=torch.uint8, device=device)
    assert decode_workspace(1, 8, 1500, 1024, device).numel() > small.numel()
    guard = torch.full((4096,), 77, dtype=torch.uint8, device=device)
    both = torch.cat([small, guard])
    flags = _hip.new_flags(device)
    out = ccpe_decode_paged(*args, max_context=1500, workspace=both[:small.numel()], flags=flags)
    assert_close_bf16(out, want)
    assert bool((both[small.numel():] == 77).all())


@pytest.mark.parametrize("hq,hkv,npos", [(8, 1, 64), (32, 8, 64), (6, 2, 128), (3, 3, 16)])
@pytest.mark.parametrize("lens", [[257], [1500], [900, 1500, 333], [4200]])
@pytest.mark.parametrize("low_gates", [0.2, 0.35, 0.7])
def test_splits_recomputed_side_by_side(device, lens, hq, hkv, npos, low_gates):
    """Gates of 0.2 to 0.007: some or all of the later splits are recomputed,
    each by a workgroup of its own, and the last to end merges: in the same
    order whichever that is."""
    args, want = setup(device, lens, hq, hkv, npos, low_gates=low_gates)
    workspace = decode_workspace(len(lens), hq, max(lens), 1024, device)
    first = ccpe_decode_paged(*args, max_context=max(lens), workspace=workspace)
    assert_close_bf16(first, want)
    for _ in range(20):
        workspace.fill_(0xFF)
        assert torch.equal(ccpe_decode_paged(*args, max_context=max(lens), workspace=workspace), first)


def test_recomputed_splits_under_graph_replay(device):
    """The count of recomputed splits is cleared by every replay of a call,
    also between eager calls of the same workspace."""
    lens = [1500, 300]
    args, want = setup(device, lens, 8, 2, 64, low_gates=0.35)
    workspace = decode_workspace(2, 8, 1500, 1024, device)
    flags, out = _hip.new_flags(device), torch.empty((2, 8, 128), dtype=torch.bfloat16, device=device)
    run = lambda: ccpe_decode_paged(*args, max_context=1500, workspace=workspace, flags=flags, out=out,  # noqa: E731
                                    check=False)
    run()
    torch.cuda.synchronize()
    eager = out.clone()
    assert_close_bf16(eager, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        out.zero_()
        run()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
    assert _hip.read_flags(flags)[0] == 0

"""The workspace of a decode call is large enough for the finest splits the
call can take, whatever its position count and KV heads (no GPU: 256 compute
units are assumed)."""

from __future__ import annotations

import pytest

from cacheslide_amd import _hip

SPLIT_BYTES = 8 + 8 + 4 * 128 + 4 + 4     # of one (request, head, split)


def splits(batch, hkv, keys, split, npos):
    """Splits of a call: halved while it has fewer workgroups than two per unit."""
    best, s = -(-keys // split), split
    while s >= 256 and s % 128 == 0 and batch * hkv * best < 512:
        s //= 2
        first = min(max(256, -(-4 * npos // 64) * 64, s), split)
        count = 1 if keys <= first else 1 + -(-(keys - first) // s)
        if count > 32:
            break
        best = count
    return best


@pytest.mark.parametrize("split", [128, 256, 512, 1024])
@pytest.mark.parametrize("batch,hq", [(1, 32), (1, 8), (3, 16), (8, 32), (64, 32)])
def test_workspace_holds_every_plan(batch, hq, split):
    lib = _hip.load()
    for keys in [*range(1, 9000, 61), 4225, 4480, 8300, 32769]:
        room = lib.cs_ccpe_decode_workspace_best_bytes(batch, hq, keys, split)
        assert room >= lib.cs_ccpe_decode_workspace_bytes(batch, hq, keys, split)
        most = max(splits(batch, hkv, keys, split, npos) for hkv in (max(1, hq // 8), hq // 4, hq)
                   for npos in (2, 64, 65, 96, 128, 200, 256))
        assert room >= batch * hq * most * SPLIT_BYTES

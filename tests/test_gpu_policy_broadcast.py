"""A profile that is one canonical table for all heads (a broadcast view): the
checker walks it once, and decides as it does on the same table stored per
head, wherever the faulty cell lies and also where the fault shows only
against the contextual position of a recomputed key, which differs by head."""

from __future__ import annotations

import dataclasses

import pytest
import torch

from cacheslide_amd import CanonicalPositionPolicy, CCPEPositionError, CoPE, SelectedAssociationPolicy, cope_attention
from tests._helpers import seeded
from tests.test_gpu_policies import HQ, P, make_plan, profile_for

pytestmark = pytest.mark.gpu

HKV = 2


def outcome(device, plan, profile, q, k, v, e, selected):
    cope = CoPE(128, P, device=device)
    with torch.no_grad():
        cope.position_embeddings.copy_(e)
    rows = torch.arange(q.shape[0], device=device)
    visible = SelectedAssociationPolicy(plan.fixed_indices, rows[list(plan.fixed_indices)]) if selected else None
    try:
        out = cope_attention(q, k, v, cope, rows, positions_transform=CanonicalPositionPolicy(plan, profile, "ckpt"),
                             visibility_transform=visible, query_chunk_size=64)
    except CCPEPositionError as error:
        return str(error)
    return out


@pytest.mark.parametrize("selected", [False, True])
@pytest.mark.parametrize("a,dyn,b", [(300, 0, 0), (256, 7, 512), (700, 300, 90), (40, 5, 30)])
def test_broadcast_profile_decides_as_a_stored_one(device, a, dyn, b, selected):
    n, fixed = a + dyn + b, a + b
    plan = make_plan(a, dyn, b) if dyn else None
    if plan is None:
        plan = make_plan(a - 20, 20, 20)
        n = a + 20
    q, k, v = (seeded((n, heads, 128), 9 + i, dtype=torch.bfloat16).to(device)
               for i, heads in enumerate((HQ, HKV, HKV)))
    e = seeded((128, P), 12, scale=0.1)
    ords = torch.arange(fixed)
    # half a position per key, saturated where the query lies past a chunk edge
    path = ((ords[:, None] - ords[None, :] + 1).clamp(min=0) * 0.5).clamp(max=P - 1)
    cells = [None, (fixed - 1, 0, float("nan")), (fixed // 2, fixed // 3, -0.5), (fixed - 1, fixed - 1, 1.5),
             (fixed - 1, fixed // 2, P - 0.5), (3, fixed - 1, 99.0), (fixed - 1, max(a - 21, 0), 0.0)]
    results = []
    for cell in cells:
        table = path.clone()
        if cell is not None:
            table[cell[0], cell[1]] = cell[2]
        stored = profile_for(plan, table.expand(HQ, fixed, fixed).numpy(), list(range(fixed)))
        shared = dataclasses.replace(stored, canonical_positions=table.to(device).expand(HQ, fixed, fixed))
        assert shared.canonical_positions.stride(0) == 0
        want = outcome(device, plan, stored, q, k, v, e, selected)
        got = outcome(device, plan, shared, q, k, v, e, selected)
        results.append(want)
        if isinstance(want, str):
            assert got == want
        else:
            assert torch.equal(got, want)
    assert any(isinstance(r, str) for r in results)

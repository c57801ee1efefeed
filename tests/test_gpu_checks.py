"""The input checks and policy lowerings that one launch each makes for a call:
every tensor and list is still scanned to its ends, in every layout."""

from __future__ import annotations

import pytest
import torch

from cacheslide_amd import CoPE, SelectedAssociationPolicy, cope_attention
from cacheslide_amd.attention import lower_policies
from tests._helpers import seeded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32, torch.float64])
@pytest.mark.parametrize("strided", [False, True])
def test_nonfinite_inputs_are_found_at_both_ends(device, dtype, strided):
    n = 70
    cope = CoPE(64, 16, device=device)
    rows = torch.arange(n, device=device)
    for which, name in enumerate(("query", "key", "value")):
        for at in (0, -1):
            x = [seeded((n, 2, 64 + 8 * strided), i, dtype=dtype).to(device)[..., :64] for i in range(3)]
            x[which][at, at, at] = float("nan") if at else float("-inf")
            with pytest.raises(ValueError, match=f"{name} must be finite"):
                cope_attention(*x, cope, rows)


@pytest.mark.parametrize("n", [2, 257, 700, 33_000])
def test_position_lists(device, n):
    q = torch.zeros((n, 1, 64), device=device)
    k = torch.zeros((3, 1, 64), device=device)
    cope = CoPE(64, 16, device=device)
    rows = torch.randperm(n, generator=torch.Generator().manual_seed(n))
    assert cope_attention(q, k, k, cope, rows.to(device)).shape == q.shape
    twice = rows.clone()
    twice[-1] = twice[0]
    with pytest.raises(ValueError, match="distinct"):
        cope_attention(q, k, k, cope, twice.to(device))
    below = rows.clone()
    below[-1] = -1
    with pytest.raises(ValueError, match="nonnegative"):
        cope_attention(q, k, k, cope, below.to(device))
    keys = torch.tensor([5, 4, 9], device=device)
    with pytest.raises(ValueError, match="strictly increasing"):
        cope_attention(q, k, k, cope, rows.to(device), keys)


@pytest.mark.parametrize("m", [0, 1, 255, 257, 5000])
@pytest.mark.parametrize("ordered", [False, True])
def test_selected_rows_and_fixed_keys(device, m, ordered):
    gen = torch.Generator().manual_seed(m)
    selected = torch.randperm(9000, generator=gen)[:m]
    selected = selected.sort().values if ordered else selected
    fixed = tuple(torch.randperm(900, generator=gen)[:300].tolist())
    rows = torch.randperm(9000, generator=gen)[:1000]
    for keys in (None, torch.arange(3, 1003)):
        want_keys = torch.arange(1000) if keys is None else keys
        _, sel, fix = lower_policies(None, SelectedAssociationPolicy(fixed, selected.to(device)), device,
                                     rows.to(device), None if keys is None else keys.to(device), 1000)
        assert torch.equal(sel.cpu().bool(), torch.isin(rows, selected))
        assert torch.equal(fix.cpu().bool(), torch.isin(want_keys, torch.tensor(fixed)))


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 128), (torch.float16, 64), (torch.float64, 64)])
@pytest.mark.parametrize("with_keys", [False, True])
def test_strided_position_lists(device, dtype, d, with_keys):
    n = 60
    cope = CoPE(d, 16, device=device)
    with torch.no_grad():
        cope.position_embeddings.copy_(seeded((d, 16), 5, scale=0.1))
    q, k, v = (seeded((n, 2, d), i, dtype=dtype).to(device) for i in range(3))
    rows = torch.arange(n, device=device).flip(0).contiguous()
    keys = 2 * torch.arange(n, device=device) if with_keys else None
    spread = lambda x: None if x is None else torch.stack([x, x + 7], 1)[:, 0]  # noqa: E731
    assert spread(rows).stride(0) == 2
    want = cope_attention(q, k, v, cope, rows, keys)
    assert torch.equal(cope_attention(q, k, v, cope, spread(rows), spread(keys)), want)
    logits = cope(q, k, rows, keys)
    assert torch.equal(cope(q, k, spread(rows), spread(keys)), logits)

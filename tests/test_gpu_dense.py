"""cope_attention on cs_ccpe_attention_dense (f16 and f32 at head size 64 and
128, bf16 at 64) against the fp64 oracle.

Tolerance, 2-norm relative: the rounding of the output (half a unit in the
last place: 2^-11 f16, 2^-8 bf16) plus 1e-5 for fp32 scores and sums; every
element also within that share of the result's largest value.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import cacheslide_amd.position as position_module
from cacheslide_amd import CoPE, cope_attention
from oracle import ccpe as orc
from tests._helpers import seeded

pytestmark = pytest.mark.gpu

REL = {torch.float32: 1e-5, torch.float16: 2.0**-11 + 1e-5, torch.bfloat16: 2.0**-8 + 1e-5}


@pytest.fixture
def called(monkeypatch):
    names = []
    real = position_module.call
    monkeypatch.setattr(position_module, "call", lambda name, *a: (names.append(name), real(name, *a))[1])
    return names


def cope_of(device, table):
    cope = CoPE(*table.shape, device=device)
    with torch.no_grad():
        cope.position_embeddings.copy_(table)
    return cope


def check(device, dtype, d, hq, hkv, n, rows, npos, strided=False, seed=0, positions=None):
    width = d + (16 // torch.empty((), dtype=dtype).element_size() if strided else 0)
    q, k, v = (seeded((n, heads, width), seed + i, dtype=dtype) for i, heads in enumerate((hq, hkv, hkv)))
    e = seeded((d, npos), seed + 3, scale=0.1)
    cope = cope_of(device, e)
    qd, kd, vd = (x.to(device)[..., :d] for x in (q[rows], k, v))
    positions = rows if positions is None else positions
    out = cope_attention(qd, kd, vd, cope, torch.from_numpy(positions).to(device)).cpu().double().numpy()
    wide = [x.double().numpy()[..., :d] for x in (q[rows], k, v)]
    expected = orc.cope_attention(*wide, e.double().numpy(), positions)
    diff = out - expected
    assert np.linalg.norm(diff) <= REL[dtype] * np.linalg.norm(expected)
    assert np.abs(diff).max() <= REL[dtype] * np.abs(expected).max()


@pytest.mark.parametrize("dtype,d", [(torch.float16, 128), (torch.float16, 64), (torch.float32, 128),
                                     (torch.float32, 64), (torch.bfloat16, 64)])
@pytest.mark.parametrize("n,hq,hkv", [(1, 4, 1), (31, 2, 2), (33, 8, 1), (65, 4, 2), (290, 8, 2)])
def test_dense_matches_fp64(device, called, dtype, d, n, hq, hkv):
    check(device, dtype, d, hq, hkv, n, np.arange(n), 64, seed=n)
    assert "cs_ccpe_attention_dense" in called and "cs_ccpe_attention" not in called


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("npos", [2, 37, 128])
def test_dense_tables_strides_and_sparse_rows(device, called, dtype, npos):
    """Odd, tiny and the largest table; rows in no order over padded K/V rows."""
    rows = np.random.default_rng(npos).permutation(300)[:77]
    check(device, dtype, 128, 8, 2, 300, rows, npos, strided=True, seed=npos)
    assert "cs_ccpe_attention" not in called


def test_dense_many_workgroups(device, called):
    """More row blocks than compute units, the same rows alone in a few."""
    check(device, torch.float16, 64, 32, 32, 2100, np.arange(2000, 2100), 64, seed=5)
    rng = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn((2100, 32, 64), generator=rng).half().to(device) for _ in range(3))
    cope = cope_of(device, seeded((64, 64), 4, scale=0.1))
    rows = torch.arange(2100, device=device)
    wide = cope_attention(q, k, v, cope, rows)                  # 544 workgroups
    few = torch.arange(1000, 1130, device=device)
    torch.testing.assert_close(wide[few], cope_attention(q[few], k, v, cope, few), rtol=0, atol=2.0**-9)
    assert "cs_ccpe_attention" not in called


@pytest.mark.parametrize("dtype,d", [(torch.float16, 128), (torch.float16, 64), (torch.float32, 128),
                                     (torch.float32, 64), (torch.bfloat16, 64)])
@pytest.mark.parametrize("hq,hkv", [(4, 1), (2, 2)])
def test_dense_largest_table(device, called, dtype, d, hq, hkv):
    """128 positions (one workgroup per CU) and rows past a workgroup's last."""
    check(device, dtype, d, hq, hkv, 421, np.arange(421), 128, seed=hq)
    assert "cs_ccpe_attention_dense" in called and "cs_ccpe_attention" not in called


def test_dense_values_past_the_range_take_the_generic_kernel(device, called):
    """A table product beyond fp32 is the reference's error, a large one that
    stays finite its result; a logit beyond fp32 is the reference's error."""
    q, k, v = (seeded((40, 2, 64), i).to(device) for i in range(3))
    rows = torch.arange(40, device=device)
    with pytest.raises(ValueError, match="logits are not finite"):
        cope_attention(q, k, v, cope_of(device, torch.full((64, 8), 3e38)), rows)
    with pytest.raises(ValueError, match="overflowed"):
        cope_attention(q * 1e19, k * 1e20, v, cope_of(device, torch.zeros((64, 8))), rows)
    large = v * 1e37
    out = cope_attention(q, k, large, cope_of(device, torch.zeros((64, 8))), rows)
    expected = orc.cope_attention(*(x.cpu().double().numpy() for x in (q, k, large)), np.zeros((64, 8)), np.arange(40))
    assert np.abs(out.cpu().double().numpy() - expected).max() <= 1e-5 * np.abs(expected).max()
    assert called.count("cs_ccpe_attention") == 3


@pytest.mark.parametrize("dtype,d", [(torch.float16, 128), (torch.float32, 64)])
def test_dense_largest_query_position(device, called, dtype, d):
    """A row past every key, up to the largest int64, sees all of them."""
    rows = np.arange(40, 70)
    positions = rows.copy()
    positions[[3, 29]] = 2**63 - 1, 2**31 + 5
    check(device, dtype, d, 4, 2, 70, rows, 64, seed=2, positions=positions)
    assert "cs_ccpe_attention" not in called


@pytest.mark.parametrize("dtype,d", [(torch.float16, 128), (torch.float16, 64), (torch.bfloat16, 64)])
@pytest.mark.parametrize("at", [0, 20_000, -1])
def test_dense_tail_of_small_probabilities(device, called, dtype, d, at):
    """One key 2^25.5 above a tail that alone carries V: the output is the
    tail's share of the sum, to the output's rounding and fp32 sums."""
    n, share = 40_000, 2.0**-25.5
    q, k = (torch.zeros((rows, 1, d), dtype=dtype) for rows in (1, n))
    v = torch.ones((n, 1, d), dtype=dtype)
    # exact in 16 bits: q.k is 64 x the dominant key's value
    q[..., 0] = 64.0
    k[at, :, 0] = -np.log(share) * d**0.5 / 64.0
    v[at] = 0.0
    logit = 64.0 * float(k[at, 0, 0]) / d**0.5
    expected = (n - 1) / (n - 1 + np.exp(logit))
    out = cope_attention(q.to(device), k.to(device), v.to(device), cope_of(device, torch.zeros((d, 64))),
                         torch.tensor([n - 1], device=device)).cpu().double().numpy()
    assert "cs_ccpe_attention" not in called
    np.testing.assert_allclose(out, expected, rtol=REL[dtype] + n * 2.0**-24 / 32)

"""A decoder step on the fused layer kernels against the same step on library
GEMMs and torch's elementwise operations, both from the same state: bf16
rounding at the same places, fp32 sums in another order."""

from __future__ import annotations

import pytest
import torch

import cacheslide_amd.decode_model as dm
from cacheslide_amd import _hip
from cacheslide_amd.ccpe import decode_workspace, raise_flags
from cacheslide_amd.decode_model import DecoderShape, PagedDecoder

pytestmark = pytest.mark.gpu


def run(device, shape, b, bs, fused, monkeypatch, positions=None, cols=6, max_context=None):
    monkeypatch.setattr(dm, "FUSED_BATCH", 32 if fused else 0)
    model = PagedDecoder(shape, device, seed=3, std=0.05)
    # the weights of every norm, as built all ones, distinct
    scales = torch.Generator(device=device).manual_seed(5)
    for norm in [model.norm, *(w for layer in model.layers for w in (layer.in_norm, layer.post_norm))]:
        norm.normal_(1.0, 0.5, generator=scales)
    gen = torch.Generator(device=device).manual_seed(4)
    wide = [torch.empty((b * cols + 1, shape.kv_heads, bs, 256), dtype=torch.bfloat16, device=device).normal_(
        generator=gen) for _ in range(shape.layers)]
    table = torch.randperm(b * cols, generator=torch.Generator().manual_seed(b)).to(torch.int32).view(b, cols)
    table = table.to(device)
    ids = (torch.arange(b, device=device) * 7) % shape.vocab
    if positions is None:
        positions = (torch.arange(b, device=device) * 13) % (cols * bs)
    before = [cache.clone() for cache in wide]
    flags = _hip.new_flags(device)
    max_context = cols * bs if max_context is None else max_context
    logits = model.step(ids, positions, wide, table, max_context=max_context, flags=flags,
                        workspace=decode_workspace(b, shape.heads, max_context, 1024, device))
    # only the records of new tokens inside the table may differ
    for cache, old in zip(wide, before):
        for i, pos in enumerate(positions.tolist()):
            if pos < cols * bs:
                old[table[i, pos // bs], :, pos % bs] = cache[table[i, pos // bs], :, pos % bs]
        assert torch.equal(cache, old)
    return logits, wide, flags


@pytest.mark.parametrize("b", [1, 16, 17, 32])
@pytest.mark.parametrize("heads,kv,ffn,vocab,bs", [(2, 1, 96, 33, 16), (9, 3, 416, 1000, 8), (16, 4, 1408, 517, 32)])
def test_fused_step_matches_library_step(device, monkeypatch, b, heads, kv, ffn, vocab, bs):
    shape = DecoderShape(layers=2, hidden=128 * heads, heads=heads, kv_heads=kv, ffn=ffn, vocab=vocab, npos=16)
    called = []
    real = dm.call
    monkeypatch.setattr(dm, "call", lambda name, *a: (called.append(name), real(name, *a))[1])
    got, got_cache, flags = run(device, shape, b, bs, True, monkeypatch)
    raise_flags(flags)
    assert called.count("cs_decoder_qkv") == called.count("cs_decoder_mlp") == 2
    want, want_cache, _ = run(device, shape, b, bs, False, monkeypatch)
    assert called.count("cs_decoder_qkv") == 2
    # a step rounds each activation to bf16 (2^-9) some ten times a layer
    def close(x, y):
        return (x.double() - y.double()).norm() <= 2e-2 * y.double().norm()
    assert got.shape == want.shape and close(got, want)
    for x, y in zip(got_cache, want_cache):
        same = (x == y).all(-1)
        assert int((~same).sum()) <= b * kv and close(x, y)


def test_a_position_past_the_table_is_flagged_and_skipped(device, monkeypatch):
    shape = DecoderShape(layers=1, hidden=256, heads=2, kv_heads=1, ffn=64, vocab=64, npos=16)
    positions = torch.tensor([3, 96], device=device)       # six blocks of 16: keys 0..95
    # a context of 97 keys is allowed, so that only the missing block is reported
    _, _, flags = run(device, shape, 2, 16, True, monkeypatch, positions=positions, max_context=112)
    assert _hip.read_flags(flags)[0] & _hip.FLAG_BLOCK_INVALID
    assert not _hip.read_flags(flags)[0] & _hip.FLAG_CONTEXT_RANGE
    with pytest.raises(ValueError):
        raise_flags(flags)

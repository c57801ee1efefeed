"""A Mistral-shaped CoPE decoder stepping one token per request over paged KV
caches: the caller of the fused decode in end-to-end runs.

Each layer follows the order of the reference's decoder layer
(src/cacheslide_vllm/reference.py:177-193, vLLM's Llama layer with a learned
CoPE table in place of rotary embeddings): RMSNorm with a fused residual, one
q/k/v projection, the new token's K/V written to its paged slot
(``cs_slot_scatter``, the paged.py:205-240 write), CCPE attention of the new
row over every key of its request (``cs_ccpe_decode_bf16``, the decode call of
runtime.py:489-508), the output projection, RMSNorm and a SiLU-gated MLP.  A
final norm and the LM head give the next-token logits.  Greedy decoding takes
their argmax on the device, so a generation loop never waits for the host;
error flags of every attention call collect in one tensor that is checked
once at the end.

All layers share one block table (one paged cache tensor per layer, the vLLM
layout [blocks, KV heads, block_size, 2 x 128]).  Weights are bf16 from
``torch.Generator`` seeds; the projections are plain library GEMMs, or for a
few requests kernels that stream the weights once with the rest of the layer
fused into them (``cs_decoder_*``).
"""

from __future__ import annotations

from dataclasses import dataclass

import torch
import torch.nn.functional as F
from torch import Tensor

from . import _hip
from ._hip import call, ptr
from .ccpe import (SharedRuns, ccpe_decode_paged, ccpe_decode_shared, decode_shared_workspace, decode_workspace,
                   raise_flags)
from .position import CoPE

HEAD_DIM = 128
# Requests up to which a step's projections are cs_decoder_* launches: 16 heads
# over 4, FFN 5632, 4 layers, 1000 keys a request, per step 305 us (library
# calls 773) at 1 request, 493 (761) at 32, the most those kernels take.
FUSED_BATCH = 32


@dataclass(frozen=True)
class DecoderShape:
    layers: int = 32
    hidden: int = 4096
    heads: int = 32
    kv_heads: int = 8
    ffn: int = 14336
    vocab: int = 32000
    npos: int = 64
    eps: float = 1e-5

    def __post_init__(self):
        if self.hidden != self.heads * HEAD_DIM:
            raise ValueError("hidden must be heads x 128")
        if self.heads % self.kv_heads or self.heads // self.kv_heads > 8:
            raise ValueError("GQA groups of at most 8 query heads per KV head")

    @property
    def parameters(self) -> int:
        qkv = (self.heads + 2 * self.kv_heads) * HEAD_DIM * self.hidden
        per_layer = qkv + self.hidden * self.hidden + 3 * self.ffn * self.hidden + 2 * self.hidden
        return self.layers * per_layer + 2 * self.vocab * self.hidden + self.hidden


MISTRAL_7B = DecoderShape()


@dataclass
class _Layer:
    qkv: Tensor       # [(Hq + 2 Hkv) x 128, hidden]
    o: Tensor         # [hidden, hidden]
    gate_up: Tensor   # [2 ffn, hidden]: gate rows, then up rows
    down: Tensor      # [hidden, ffn]
    in_norm: Tensor
    post_norm: Tensor
    cope: CoPE


class PagedDecoder:
    """Random-init decoder of ``shape``: weights N(0, std) in ``dtype``, norm
    weights 1, CoPE tables N(0, std) in fp32."""

    def __init__(self, shape: DecoderShape, device, *, seed: int = 0, std: float = 0.02,
                 dtype: torch.dtype = torch.bfloat16):
        self.shape, self.device, self.dtype = shape, torch.device(device), dtype
        gen = torch.Generator(device=self.device).manual_seed(seed)

        def normal(*dims, dt=dtype):
            t = torch.empty(dims, dtype=dt, device=self.device)
            return t.normal_(0.0, std, generator=gen)

        s = shape
        self.embed = normal(s.vocab, s.hidden)
        self.layers: list[_Layer] = []
        for _ in range(s.layers):
            cope = CoPE(HEAD_DIM, s.npos, device=self.device)
            with torch.no_grad():
                cope.position_embeddings.copy_(normal(HEAD_DIM, s.npos, dt=torch.float32))
            self.layers.append(_Layer(
                qkv=normal((s.heads + 2 * s.kv_heads) * HEAD_DIM, s.hidden),
                o=normal(s.hidden, s.hidden),
                gate_up=normal(2 * s.ffn, s.hidden),
                down=normal(s.hidden, s.ffn),
                in_norm=torch.ones(s.hidden, dtype=dtype, device=self.device),
                post_norm=torch.ones(s.hidden, dtype=dtype, device=self.device),
                cope=cope,
            ))
        self.norm = torch.ones(s.hidden, dtype=dtype, device=self.device)
        self.lm_head = normal(s.vocab, s.hidden)

    def new_caches(self, num_blocks: int, block_size: int) -> list[Tensor]:
        """One paged cache per layer, [blocks, KV heads, block_size, 2 x 128]."""
        return [torch.empty((num_blocks, self.shape.kv_heads, block_size, 2 * HEAD_DIM), dtype=self.dtype,
                            device=self.device) for _ in range(self.shape.layers)]

    def _rms(self, x: Tensor, weight: Tensor) -> Tensor:
        return F.rms_norm(x, (self.shape.hidden,), weight, self.shape.eps)

    def step(self, ids: Tensor, positions: Tensor, caches: list[Tensor], block_table: Tensor, *,
             max_context: int, workspace: Tensor, flags: Tensor, split: int = 1024,
             attn_out: Tensor | None = None, shared: SharedRuns | None = None) -> Tensor:
        """One token per request: ``ids`` [B] at ``positions`` [B] (int64, the
        request's key count before this token) -> logits [B, vocab].  Writes the
        token's K/V to slot ``block_table[b, p // bs] * bs + p % bs`` of every
        layer's cache; ``max_context`` bounds positions + 1.  With ``shared``
        (runs of blocks the requests share, built on ``block_table``) the
        attention reads each run once for the batch (``ccpe_decode_shared``,
        whose ``workspace`` this then is)."""
        s = self.shape
        b = ids.shape[0]
        bs = caches[0].shape[2]
        if 1 <= b <= FUSED_BATCH and self._fused_ok(ids, positions, caches, block_table, flags, attn_out):
            return self._step_fused(ids, positions, caches, block_table, max_context, workspace, flags, split,
                                    attn_out, shared)
        slots = block_table.gather(1, (positions // bs).unsqueeze(1)).squeeze(1).long() * bs + positions % bs
        context = (positions + 1).to(torch.int32)
        if attn_out is None:
            attn_out = torch.empty((b, s.heads, HEAD_DIM), dtype=self.dtype, device=self.device)
        stream = _hip.stream_of(self.device)
        lib = _hip.load()
        tail = shared.tail_lens(context) if shared is not None else None
        q_end, k_end = s.heads * HEAD_DIM, (s.heads + s.kv_heads) * HEAD_DIM
        x, residual = self.embed[ids], None
        for layer, cache in zip(self.layers, caches):
            if residual is None:
                residual = x
            else:
                residual = x + residual
            h = self._rms(residual, layer.in_norm)
            qkv = h @ layer.qkv.T
            q = qkv[:, :q_end].view(b, s.heads, HEAD_DIM)
            k = qkv[:, q_end:k_end].view(b, s.kv_heads, HEAD_DIM)
            v = qkv[:, k_end:].view(b, s.kv_heads, HEAD_DIM)
            status = lib.cs_slot_scatter(_hip.vref(cache), _hip.vref(None), _hip.vref(None), _hip.ptr(slots),
                                         _hip.ptr(None), b, _hip.vref(k), _hip.vref(v), stream)
            if status:
                _hip.check(status, "cs_slot_scatter")
            if shared is not None:
                ccpe_decode_shared(q, cache, block_table, context, layer.cope, shared, max_context=max_context,
                                   split=split, tail=tail, workspace=workspace, out=attn_out, flags=flags,
                                   check=False)
            else:
                ccpe_decode_paged(q, cache, block_table, context, layer.cope, max_context=max_context,
                                  split=split, workspace=workspace, out=attn_out, flags=flags, check=False)
            residual = attn_out.view(b, s.hidden) @ layer.o.T + residual
            h = self._rms(residual, layer.post_norm)
            gate, up = (h @ layer.gate_up.T).split(s.ffn, dim=-1)
            x = (F.silu(gate) * up) @ layer.down.T
        return self._rms(x + residual, self.norm) @ self.lm_head.T

    def _fused_ok(self, ids, positions, caches, block_table, flags, attn_out) -> bool:
        """Whether the layout is the one cs_decoder_* reads: bf16 weights as
        built, contiguous int64 ids and positions, bf16 caches with whole
        contiguous records."""
        s = self.shape

        def plain(t, dtype, *dims):
            return (t.dtype == dtype and t.shape == dims and t.is_contiguous() and t.device == caches[0].device
                    and t.data_ptr() % 16 == 0)

        wide = (s.heads + 2 * s.kv_heads) * HEAD_DIM
        bf16, b = torch.bfloat16, ids.shape[0]
        return (
            s.ffn % 32 == 0 and len(caches) == len(self.layers)
            and positions.dtype == torch.long and positions.shape == (b,) and positions.is_contiguous()
            and positions.device == caches[0].device
            and ids.dtype == torch.long and ids.ndim == 1
            and block_table.dtype == torch.int32 and block_table.ndim == 2 and block_table.stride(1) == 1
            and block_table.shape[0] == b and block_table.shape[1] > 0 and block_table.device == caches[0].device
            and flags.dtype == torch.int32 and flags.numel() >= 1 and flags.device == caches[0].device
            and (attn_out is None or plain(attn_out, bf16, b, s.heads, HEAD_DIM))
            and plain(self.embed, bf16, s.vocab, s.hidden) and plain(self.lm_head, bf16, s.vocab, s.hidden)
            and plain(self.norm, bf16, s.hidden)
            and all(c.dtype == bf16 and c.ndim == 4 and c.shape[1:] == caches[0].shape[1:]
                    and c.shape[1] == s.kv_heads and c.shape[3] == 2 * HEAD_DIM and c.stride(3) == 1
                    and c.data_ptr() % 16 == 0 for c in caches)
            and all(plain(layer.qkv, bf16, wide, s.hidden) and plain(layer.o, bf16, s.hidden, s.hidden)
                    and plain(layer.gate_up, bf16, 2 * s.ffn, s.hidden) and plain(layer.down, bf16, s.hidden, s.ffn)
                    and plain(layer.in_norm, bf16, s.hidden) and plain(layer.post_norm, bf16, s.hidden)
                    for layer in self.layers))

    def _step_fused(self, ids, positions, caches, block_table, max_context, workspace, flags, split, attn_out,
                    shared) -> Tensor:
        """``step`` with each layer's launches fused around its attention call
        (cs_decoder_qkv, cs_decoder_mlp)."""
        s, b = self.shape, ids.shape[0]
        stream = _hip.stream_of(self.device)
        residual = self.embed[ids]
        context = torch.empty(b, dtype=torch.int32, device=residual.device)
        call("cs_decoder_context", ptr(positions), b, ptr(context), stream)
        rows = torch.empty((2, b, s.heads, HEAD_DIM), dtype=self.dtype, device=residual.device)
        q = rows[0]
        if attn_out is None:
            attn_out = rows[1]
        act = torch.empty((b, s.ffn), dtype=self.dtype, device=residual.device)
        tail = shared.tail_lens(context) if shared is not None else None
        args = _hip.CsDecoderLayerArgs()
        args.batch, args.hidden, args.heads, args.kv_heads, args.ffn = b, s.hidden, s.heads, s.kv_heads, s.ffn
        args.eps = s.eps
        args.residual, args.q, args.attn, args.act = (t.data_ptr() for t in (residual, q, attn_out, act))
        args.table, args.table_stride, args.table_cols = block_table.data_ptr(), block_table.stride(0), block_table.shape[1]
        args.positions, args.flags = positions.data_ptr(), flags.data_ptr()
        for layer, cache in zip(self.layers, caches):
            args.qkv, args.o = layer.qkv.data_ptr(), layer.o.data_ptr()
            args.gate_up, args.down = layer.gate_up.data_ptr(), layer.down.data_ptr()
            args.in_norm, args.post_norm = layer.in_norm.data_ptr(), layer.post_norm.data_ptr()
            args.cache, args.blocks, args.block_size = cache.data_ptr(), cache.shape[0], cache.shape[2]
            args.s_block, args.s_head, args.s_offset = cache.stride()[:3]
            call("cs_decoder_qkv", args, stream)
            if shared is not None:
                ccpe_decode_shared(q, cache, block_table, context, layer.cope, shared, max_context=max_context,
                                   split=split, tail=tail, workspace=workspace, out=attn_out, flags=flags,
                                   check=False)
            else:
                ccpe_decode_paged(q, cache, block_table, context, layer.cope, max_context=max_context,
                                  split=split, workspace=workspace, out=attn_out, flags=flags, check=False)
            call("cs_decoder_mlp", args, stream)
        logits = torch.empty((b, s.vocab), dtype=self.dtype, device=residual.device)
        call("cs_decoder_head", ptr(residual), ptr(self.norm), ptr(self.lm_head), ptr(logits), b, s.hidden, s.vocab,
             s.eps, stream)
        return logits

    def generate(self, first_ids: Tensor, lengths: Tensor, caches: list[Tensor], block_table: Tensor,
                 steps: int, *, max_context: int, split: int = 1024, check: bool = True,
                 shared: SharedRuns | None = None) -> Tensor:
        """Greedy decoding of ``steps`` tokens per request after contexts of
        ``lengths`` keys -> token ids [steps, B] (on the device); ``shared`` as
        in ``step``."""
        b = first_ids.shape[0]
        if shared is not None:
            workspace = decode_shared_workspace(b, self.shape.heads, shared, max_context, split, self.device)
        else:
            workspace = decode_workspace(b, self.shape.heads, max_context, split, self.device)
        flags = _hip.new_flags(self.device)
        attn_out = torch.empty((b, self.shape.heads, HEAD_DIM), dtype=self.dtype, device=self.device)
        out = torch.empty((steps, b), dtype=torch.long, device=self.device)
        ids, positions = first_ids, lengths.to(torch.long).clone()
        for t in range(steps):
            logits = self.step(ids, positions, caches, block_table, max_context=max_context,
                               workspace=workspace, flags=flags, split=split, attn_out=attn_out, shared=shared)
            ids = logits.argmax(dim=-1)
            out[t] = ids
            positions += 1
        if check:
            raise_flags(flags)
        return out

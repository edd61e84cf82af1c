"""Fused LM head + cross-entropy on MI355X (no (M, V) logits).

Drop-ins for ``fused_lmhead_xent`` / ``FusedLMHeadXent`` / ``FusedLMHeadXentModule``
(r2/dhammic-ai/src/kernels/lmhead_xent.py:256-431) and ``ChunkedLMHeadXent``
(r2/dhammic-ai/src/runtime/chunked_lmhead.py:288-431): same arguments, scalar fp32 mean loss
over the non-ignored targets, gradients for hidden and the (tied) weight.

Device work (include/ssd_lmhead.h): the forward kernel multiplies hidden and weight tiles on bf16
MFMA and keeps only each row's running max / sum of exp and its target logit; the backward kernel
recomputes the tiles and writes the logits gradient (softmax - onehot) * dloss / n_valid for one
chunk of rows in bf16, from which d_hidden = G^T W and d_weight += G hidden are library GEMMs
(hipBLASLt through torch). The scale dloss / n_valid stays on the device (the reference reads it
back to the host, lmhead_xent.py:330). bf16 hidden and weight only (the block's dtype); other
dtypes raise NotImplementedError. Any d up to the reference's 4096 (lmhead_xent.py:284): the
kernels read 16-byte rows, so a d that is not a multiple of 8 is zero-padded (the padded columns
add nothing to any product).
"""
from __future__ import annotations

import math
from typing import Iterable, Union

import torch
import torch.nn as nn
from torch import Tensor

from . import _capi as C_
from .ssd_scan import _on, _p, _stream

__all__ = ["fused_lmhead_xent", "FusedLMHeadXent", "FusedLMHeadXentModule", "ChunkedLMHeadXent"]

# bytes of the backward's bf16 logits-gradient buffer (V x rows); at config 4's head (V = 50 304)
# 2 GiB holds all 16 384 rows, so one pair of GEMMs produces d_weight without a running sum
_BWD_BYTES = 2 << 30


_DTYPES = (torch.bfloat16, torch.float16, torch.float32)


def check_supported(hidden_dtype: torch.dtype, weight_dtype: torch.dtype) -> None:
    """The dtypes the head takes: hidden and weight of one dtype, bf16, fp16 or fp32 (NotImplementedError
    otherwise). bf16 runs the kernels on the operands as given; fp16 and fp32 run them on split bf16
    operands (``_split_operand``) with the gradient GEMMs in fp32."""
    if hidden_dtype != weight_dtype or hidden_dtype not in _DTYPES:
        raise NotImplementedError(f"fused_lmhead_xent: hidden and weight of one dtype among bf16, fp16 and fp32 "
                                  f"(got {hidden_dtype}, {weight_dtype})")


def _split_operand(t: Tensor, order: str) -> Tensor:
    """An fp32 operand t (rows, d) as bf16 parts side by side along d: ``order`` "hhl" gives
    [hi | hi | lo], "hlh" gives [hi | lo | hi], with hi = bf16(t) and lo = bf16(t - hi). The products of an
    "hhl" and an "hlh" operand sum hi hi' + hi lo' + lo hi', t t' to about 2^-16 relative (the lo lo'
    term is below it): the bf16 kernels then multiply fp32 operands."""
    hi = t.to(torch.bfloat16)
    lo = (t - hi.float()).to(torch.bfloat16)
    parts = [hi, hi, lo] if order == "hhl" else [hi, lo, hi]
    return torch.cat(parts, dim=1).contiguous()


def _pad8(t: Tensor) -> Tensor:
    """t (rows, d) with its last dimension zero-padded to a multiple of 8 (16-byte bf16 rows)."""
    pad = (-t.shape[-1]) % 8
    return torch.nn.functional.pad(t, (0, pad)) if pad else t


class FusedLMHeadXent(torch.autograd.Function):
    @staticmethod
    def forward(ctx, hidden: Tensor, weight: Tensor, targets: Tensor, ignore_index: int = -100,
                bwd_rows: int | None = None) -> Tensor:
        assert hidden.is_cuda and weight.is_cuda and targets.is_cuda, "FusedLMHeadXent requires CUDA tensors"
        assert weight.dim() == 2, f"weight must be 2-D (V, d), got {tuple(weight.shape)}"
        assert hidden.shape[-1] == weight.shape[-1], (
            f"hidden last dim {hidden.shape[-1]} != weight last dim {weight.shape[-1]}")
        assert targets.dtype == torch.long, f"targets must be int64, got {targets.dtype}"
        check_supported(hidden.dtype, weight.dtype)
        D0, V = hidden.shape[-1], weight.shape[0]
        split = hidden.dtype != torch.bfloat16
        h = _pad8(hidden.contiguous().view(-1, D0))
        w = _pad8(weight.contiguous())
        if split:  # fp16 / fp32: the kernels multiply split bf16 operands of width 3 d
            h, w = h.float(), w.float()
            hk, wk = _split_operand(h, "hhl"), _split_operand(w, "hlh")
        else:
            hk, wk = h, w
        D = hk.shape[-1]
        t = targets.contiguous().view(-1)
        M = h.shape[0]
        assert t.shape[0] == M, f"targets length {t.shape[0]} != hidden rows {M}"
        dev = h.device
        logZ = torch.empty(M, dtype=torch.float32, device=dev)
        tl = torch.empty(M, dtype=torch.float32, device=dev)
        mask = torch.empty(M, dtype=torch.int32, device=dev)
        lib = C_.load()
        ws = torch.empty(lib.ssd_lmhead_xent_workspace(M, V), dtype=torch.uint8, device=dev)
        with _on(dev):
            st = lib.ssd_lmhead_xent_fwd(M, V, D, _p(hk), _p(wk), _p(t), int(ignore_index), _p(logZ), _p(tl),
                                         _p(mask), _p(ws), ws.numel(), _stream(dev))
        C_.check(st, "ssd_lmhead_xent_fwd")
        maskf = mask.to(torch.float32)
        n_valid = maskf.sum().clamp_min(1.0)
        loss = ((logZ - tl) * maskf).sum() / n_valid
        ctx.save_for_backward(h, w, t, logZ, n_valid)
        ctx.ignore_index = int(ignore_index)
        ctx.shape = hidden.shape
        ctx.d = D0
        ctx.dtypes = (hidden.dtype, weight.dtype)
        ctx.split = split
        # the split backward holds two bf16 parts and their fp32 sum per element of a chunk
        per = 8 if split else 2
        ctx.bwd_rows = int(bwd_rows) if bwd_rows else max(128, _BWD_BYTES // (per * V) // 128 * 128)
        return loss

    @staticmethod
    def backward(ctx, dloss: Tensor):
        h, w, t, logZ, n_valid = ctx.saved_tensors
        M, D = h.shape
        V = w.shape[0]
        dev = h.device
        scale = (dloss.detach().to(torch.float32) / n_valid).reshape(1).contiguous()
        rows = min(M, ctx.bwd_rows)
        ldg = (rows + 7) // 8 * 8
        if ctx.split:
            return FusedLMHeadXent._backward_split(ctx, h, w, t, logZ, scale, rows, ldg)
        G = torch.empty(V, ldg, dtype=torch.bfloat16, device=dev)
        dh = torch.empty_like(h)
        dw32 = None
        dw = None
        lib = C_.load()
        for r0 in range(0, M, rows):
            n = min(rows, M - r0)
            with _on(dev):
                st = lib.ssd_lmhead_xent_dlogits(M, V, D, r0, n, _p(h), _p(w), _p(t), ctx.ignore_index, _p(logZ),
                                                 _p(scale), _p(G), ldg, _stream(dev))
            C_.check(st, "ssd_lmhead_xent_dlogits")
            g = G[:, :n]
            torch.mm(g.t(), w, out=dh[r0:r0 + n])  # a row slice of dh is contiguous: no copy
            part = torch.mm(g, h[r0:r0 + n])
            if r0 == 0 and n == M:
                dw = part
            else:
                dw32 = part.float() if dw32 is None else dw32.add_(part.float())
        if dw is None:
            dw = dw32.to(w.dtype)
        if D != ctx.d:  # drop the zero padding
            dh, dw = dh[:, :ctx.d], dw[:, :ctx.d].contiguous()
        return dh.reshape(ctx.shape), dw, None, None, None


    @staticmethod
    def _backward_split(ctx, h, w, t, logZ, scale, rows, ldg):
        """fp16 / fp32 backward: per chunk of rows the kernels write the logits gradient as two bf16 parts
        (from the split operands' fp32-accurate logits); their fp32 sum enters fp32 GEMMs."""
        M, D = h.shape
        V = w.shape[0]
        dev = h.device
        hk, wk = _split_operand(h, "hhl"), _split_operand(w, "hlh")
        G = torch.empty(V, ldg, dtype=torch.bfloat16, device=dev)
        G_lo = torch.empty(V, ldg, dtype=torch.bfloat16, device=dev)
        dh = torch.empty(M, D, dtype=torch.float32, device=dev)
        dw = torch.zeros(V, D, dtype=torch.float32, device=dev)
        lib = C_.load()
        for r0 in range(0, M, rows):
            n = min(rows, M - r0)
            with _on(dev):
                st = lib.ssd_lmhead_xent_dlogits_split(M, V, hk.shape[1], r0, n, _p(hk), _p(wk), _p(t),
                                                       ctx.ignore_index, _p(logZ), _p(scale), _p(G), _p(G_lo), ldg,
                                                       _stream(dev))
            C_.check(st, "ssd_lmhead_xent_dlogits_split")
            g = G[:, :n].float() + G_lo[:, :n].float()
            torch.mm(g.t(), w, out=dh[r0:r0 + n])
            dw.addmm_(g, h[r0:r0 + n])
        dh, dw = dh[:, :ctx.d].to(ctx.dtypes[0]), dw[:, :ctx.d].to(ctx.dtypes[1]).contiguous()
        return dh.reshape(ctx.shape), dw, None, None, None


def fused_lmhead_xent(hidden: Tensor, weight: Tensor, targets: Tensor, ignore_index: int = -100) -> Tensor:
    """Mean cross-entropy of (hidden @ weight.T) against targets, without the (M, V) logits."""
    return FusedLMHeadXent.apply(hidden, weight, targets, ignore_index)


class FusedLMHeadXentModule(nn.Module):
    """Drop-in fused LM-head + cross-entropy module; a given ``weight`` is shared (weight tying)."""

    def __init__(self, d_model: int, vocab_size: int, weight: nn.Parameter | None = None, ignore_index: int = -100):
        super().__init__()
        self.d_model = d_model
        self.vocab_size = vocab_size
        self.ignore_index = ignore_index
        if weight is None:
            self.weight = nn.Parameter(torch.empty(vocab_size, d_model).normal_(mean=0.0, std=1.0 / math.sqrt(d_model)))
        else:
            assert weight.shape == (vocab_size, d_model), (
                f"tied weight shape {tuple(weight.shape)} != ({vocab_size}, {d_model})")
            self.weight = weight

    def forward(self, hidden: Tensor, targets: Tensor) -> Tensor:
        return fused_lmhead_xent(hidden, self.weight, targets, self.ignore_index)

    def extra_repr(self) -> str:
        return f"d_model={self.d_model}, vocab_size={self.vocab_size}, ignore_index={self.ignore_index}"


class ChunkedLMHeadXent(nn.Module):
    """Sequence-chunked LM head (chunked_lmhead.py:288-431): the token-weighted mean loss over all
    non-ignored positions of a (B, T, D) tensor, or of an iterable of (B, chunk, D) chunks with
    matching target chunks. With a tensor, the backward's logits gradient is built for
    ``chunk_size * B`` rows at a time."""

    def __init__(self, d_model: int, vocab_size: int, weight: nn.Parameter | None = None, chunk_size: int = 256,
                 ignore_index: int = -100) -> None:
        super().__init__()
        if chunk_size <= 0:
            raise ValueError(f"chunk_size must be positive, got {chunk_size}")
        self.d_model = d_model
        self.vocab_size = vocab_size
        self.chunk_size = chunk_size
        self.ignore_index = ignore_index
        if weight is None:
            self.weight = nn.Parameter(torch.empty(vocab_size, d_model).normal_(mean=0.0, std=1.0 / math.sqrt(d_model)))
        else:
            if tuple(weight.shape) != (vocab_size, d_model):
                raise ValueError(f"tied weight shape {tuple(weight.shape)} != ({vocab_size}, {d_model})")
            self.weight = weight

    def forward(self, hidden: Union[Tensor, Iterable[Tensor]], targets: Union[Tensor, Iterable[Tensor]],
                total_tokens: int | None = None) -> Tensor:
        weight = self.weight
        if not weight.is_cuda:
            raise RuntimeError(f"ChunkedLMHeadXent requires a CUDA weight; got {weight.device}.")
        if isinstance(hidden, Tensor) != isinstance(targets, Tensor):
            raise TypeError("hidden and targets must both be tensors or both be iterables, got "
                            f"{type(hidden).__name__} and {type(targets).__name__}")
        if isinstance(hidden, Tensor):
            B = hidden.shape[0] if hidden.dim() == 3 else 1
            return FusedLMHeadXent.apply(hidden.to(weight.device), weight, targets.to(weight.device),
                                         self.ignore_index, max(1, self.chunk_size * B))
        pairs = [(h.to(weight.device), t.to(weight.device)) for h, t in zip(hidden, targets)]
        if not pairs:
            return weight.sum() * 0.0
        counts = [(t != self.ignore_index).sum() for _, t in pairs]
        total = torch.stack(counts).sum().clamp_min(1).to(torch.float32)
        loss = None
        for (h, t), n in zip(pairs, counts):
            part = fused_lmhead_xent(h, weight, t, self.ignore_index) * n.to(torch.float32)
            loss = part if loss is None else loss + part
        return loss / total

    def extra_repr(self) -> str:
        return (f"d_model={self.d_model}, vocab_size={self.vocab_size}, chunk_size={self.chunk_size}, "
                f"ignore_index={self.ignore_index}")

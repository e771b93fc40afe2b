"""Softmax cross-entropy for LM heads (HIP kernels).

``cross_entropy(logits, target)`` -- standard autograd op (fwd saves lse; bwd writes grads).
``fused_linear_cross_entropy(h, W, target)`` -- LM head + loss in one autograd node: the logits
buffer is overwritten in place with d(loss)/d(logits) during the forward (loss is the graph's
terminal node, so the gradient is known up to the scalar upstream factor), the backward is just two
GEMMs. Peak memory is one bf16 [T, V] buffer instead of logits + fp32 softmax + grad, and
``chunk_tokens`` bounds even that (ALST's TiledLoss, reference
runtime/sequence_parallel/ulysses_sp.py:915, plays the same role). On bf16 GPU training steps whose
shapes fit its tile, the gradient is instead written in the backward by ``xent_grad_dual``
(token-major over the logits + vocab-major copy for the TN weight-gradient GEMM, upstream scalar
folded in).
"""
import os

import torch
import torch.nn.functional as F

from . import native
from .linear import keep_local, local_grad_target, product


class _XEnt(torch.autograd.Function):
    @staticmethod
    def forward(ctx, logits, target, ignore_index):
        logits2 = logits.contiguous().view(-1, logits.shape[-1])
        loss, lse = torch.ops.sxe.xent_fwd(logits2, target.reshape(-1).contiguous(), int(ignore_index), False, None, 1.0)
        ctx.save_for_backward(logits2, target.reshape(-1).contiguous(), lse)
        ctx.ignore_index = ignore_index
        ctx.shape = logits.shape
        return loss.view(logits.shape[:-1])

    @staticmethod
    def backward(ctx, dloss):
        logits2, target, lse = ctx.saved_tensors
        g = torch.ops.sxe.xent_bwd(logits2, target, lse, dloss.reshape(-1).float().contiguous(), int(ctx.ignore_index),
                                   False)
        return g.view(ctx.shape), None, None


def cross_entropy(logits, target, ignore_index=-100, reduction="mean"):
    if native.use_hip(logits):
        per_tok = _XEnt.apply(logits, target, ignore_index)
    else:
        per_tok = F.cross_entropy(logits.float().reshape(-1, logits.shape[-1]), target.reshape(-1),
                                  ignore_index=ignore_index, reduction="none").view(target.shape)
    if reduction == "none":
        return per_tok
    if reduction == "sum":
        return per_tok.sum()
    n = (target != ignore_index).sum().clamp_min(1)
    return per_tok.sum() / n


def _column_states(h):
    """[tokens, K] of the hidden states, rounded up to 64 tokens by zeros, whole 16-byte vectors."""
    h2 = h.reshape(-1, h.shape[-1])
    if h2.shape[0] % 64:
        h2 = F.pad(h2, (0, 0, 0, -h2.shape[0] % 64))
    h2 = h2.contiguous()
    return h2.clone() if h2.data_ptr() % 16 else h2  # a view that starts inside a vector


class _ColumnHeadXEnt(torch.autograd.Function):
    """LM head and loss over logits with a token per column (``xent_cols_fwd``): the logits, the data gradient and the weight gradient
    are products of whole 16-byte vectors although a row of logits is not."""

    @staticmethod
    def forward(ctx, h, weight, target, ignore_index):
        tgt = target.reshape(-1).contiguous()
        h2 = _column_states(h)
        logits = torch.ops.sxe.gemm_tn(weight, h2, None, False)
        loss, lse = torch.ops.sxe.xent_cols_fwd(logits, tgt, int(ignore_index))
        # the rows that were rounded up are kept beside h: making them again costs 2368 x 768 a fill and a copy, 8 us
        ctx.save_for_backward(logits, lse, tgt, h, h2 if h2.data_ptr() != h.data_ptr() else None, weight)
        ctx.ignore_index = int(ignore_index)
        ctx.weight = keep_local(weight)
        return loss.view(target.shape)

    @staticmethod
    def backward(ctx, dloss):
        logits, lse, tgt, h, h2, weight = ctx.saved_tensors
        g = torch.ops.sxe.xent_cols_bwd(logits, tgt, lse, dloss.detach().reshape(-1).float().contiguous(), ctx.ignore_index)
        del logits
        dh = dw = None
        if torch.is_grad_enabled():  # derivatives of these products may be asked for, which the kernels below do not have
            g = g[:, :tgt.numel()]
            if ctx.needs_input_grad[0]:
                dh = (g.t() @ weight).view(h.shape)
            if ctx.needs_input_grad[1]:
                dw = g @ h.reshape(-1, h.shape[-1])
            return dh, dw, None, None
        h2 = _column_states(h) if h2 is None else h2
        if ctx.needs_input_grad[0]:  # contracts the vocabulary: the form of a weight gradient, in fp32 parts
            dh = torch.empty(h2.shape, device=h2.device, dtype=torch.float32)
            torch.ops.sxe.wgrad_gemm_(g, weight, dh, 1.0, False)
            dh = dh[:tgt.numel()].to(h2.dtype).view(h.shape)
        if ctx.needs_input_grad[1]:
            into = local_grad_target(ctx.weight, ctx) if native.plain(dloss) else None
            # in fp32 into the optimizer's buffer: no gradient of the table is written, read and added up besides
            if into is not None and into[0].shape == weight.shape and into[0].data_ptr() % 16 == 0:
                torch.ops.sxe.gemm_tn_into(g, torch.ops.sxe.transpose16(h2), *into)
                ctx.weight._sxe_grad_done(ctx.weight)
            else:
                dw = torch.ops.sxe.gemm_tn(g, torch.ops.sxe.transpose16(h2), None, False)
        return dh, dw, None, None


def head_cross_entropy(h, weight, target, ignore_index=-100):
    """``cross_entropy(F.linear(h, weight), target)``, the mean over the targets that count.

    A vocabulary that is no multiple of 8 puts the rows of its logits off 16 bytes, and the library's products then take 0.7 (logits,
    weight gradient) and 0.45 PFLOP/s (data gradient). 50257 x 768, the three of them, us, so / with a token per column: 64 tokens
    244 / 121, 512 330 / 184, 2048 723 / 498, 8192 1940 / 1751."""
    if _columns_ok(h, weight, target):
        native.require_hip()
        loss = _ColumnHeadXEnt.apply(h, weight, target, ignore_index)
        return loss.sum() / (target != ignore_index).sum().clamp_min(1)
    return cross_entropy(F.linear(h, weight), target, ignore_index)


def _columns_ok(h, weight, target):
    if not (h.is_cuda and weight.dim() == 2 and weight.shape[0] % 8 and h.dim() > 1 and h.shape[-1] == weight.shape[1]
            and h.shape[:-1] == target.shape and target.dtype == torch.long and target.device == h.device and native.use_hip(h)
            and native.plain(h, weight, target) and not torch.is_autocast_enabled("cuda")):
        return False
    tokens, K = target.numel(), h.shape[-1]
    return (0 < tokens < 1 << 23 and (tokens + 63) * K < 1 << 31 and weight.shape[0] >= 64 and K % 64 == 0 and weight.device == h.device
            and h.dtype == weight.dtype == torch.bfloat16 and weight.is_contiguous() and weight.data_ptr() % 16 == 0)


DUAL = os.environ.get("SXE_XENT_DUAL", "1") == "1"


def _dual_ok(h2, weight):
    """The dual-layout gradient path applies: bf16 GPU operands, tokens % 64, vocab % 256, hidden % 64
    (the kernel's tile and the transpose kernel's)."""
    return (DUAL and h2.is_cuda and h2.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16
            and weight.dim() == 2 and h2.shape[0] % 64 == 0 and h2.shape[0] > 0 and weight.shape[0] % 256 == 0
            and h2.shape[1] % 64 == 0 and h2.is_contiguous() and native.use_hip(h2))


class _FusedLinearXEnt(torch.autograd.Function):
    @staticmethod
    def forward(ctx, h, weight, target, ignore_index, chunk_tokens, reduction="mean"):
        H = h.shape[-1]
        h2 = h.reshape(-1, H)
        tgt = target.reshape(-1).contiguous()
        T = h2.shape[0]
        if reduction == "sum":
            n_valid = torch.ones((), device=h.device, dtype=torch.float32)
        else:
            n_valid = (tgt != ignore_index).sum().clamp_min(1).float()
        inv_n = (1.0 / n_valid).reshape(1)
        need_grad = torch.is_grad_enabled() or h.requires_grad or weight.requires_grad
        chunk = T if not chunk_tokens else min(int(chunk_tokens), T)
        if chunk == T and need_grad and _dual_ok(h2, weight):
            # dual layout: the forward computes only loss + lse; the backward writes the scaled
            # gradient over the logits AND its vocab-major transpose in one pass (xent_grad_dual),
            # so the LM-head weight gradient is a TN GEMM with no transpose of the 4 GB gradient
            logits = product(h2, weight)
            loss, lse = torch.ops.sxe.xent_fwd(logits, tgt, int(ignore_index), False, None, 1.0)
            ctx.save_for_backward(logits, lse, tgt, inv_n, h2, weight)
            ctx.mode = "dual"
            ctx.ignore_index = int(ignore_index)
            ctx.hshape = h.shape
            return loss.sum() / n_valid
        if chunk == T:
            # unchunked: keep d(loss)/d(logits) (written over the logits) and do both GEMMs in
            # backward, where the weight-grad GEMM can land directly in the optimizer's buffer
            logits = product(h2, weight)
            loss, _ = torch.ops.sxe.xent_fwd(logits, tgt, int(ignore_index), need_grad, inv_n, 1.0)
            ctx.save_for_backward(logits if need_grad else None, h2, weight)
            ctx.mode = "dlogits"
            ctx.hshape = h.shape
            return loss.sum() / n_valid
        ctx.mode = "chunked"
        loss_sum = torch.zeros((), device=h.device, dtype=torch.float32)
        dh = torch.empty_like(h2) if need_grad else None
        dW = None
        for s in range(0, T, chunk):
            e = min(T, s + chunk)
            logits = torch.matmul(h2[s:e], weight.t())
            loss, _ = torch.ops.sxe.xent_fwd(logits, tgt[s:e], int(ignore_index), need_grad, inv_n, 1.0)
            loss_sum = loss_sum + loss.sum()
            if need_grad:
                torch.matmul(logits, weight, out=dh[s:e])
                part = torch.matmul(logits.t(), h2[s:e])
                if dW is None:
                    dW = part if chunk == T else part.float()
                else:
                    dW.add_(part.float())
            del logits
        ctx.save_for_backward(dh, dW)
        ctx.wdtype = weight.dtype
        ctx.hshape = h.shape
        return loss_sum / n_valid

    @staticmethod
    def backward(ctx, gout):
        if ctx.mode == "dual":
            logits, lse, tgt, inv_n, h2, weight = ctx.saved_tensors
            gT = torch.ops.sxe.xent_grad_dual(logits, tgt, lse, ctx.ignore_index, inv_n,
                                              gout.detach().float().reshape(1).contiguous())
            from .linear import data_grad
            from .mlp import weight_grad_tn
            dh = data_grad(logits, weight).view(ctx.hshape)  # logits now hold the gradient
            del logits
            dW = None
            if ctx.needs_input_grad[1]:
                dW = weight_grad_tn(weight, gT, torch.ops.sxe.transpose16(h2))
            return dh, dW, None, None, None, None
        if ctx.mode == "dlogits":
            dl, h2, weight = ctx.saved_tensors
            dl.mul_(gout.to(dl.dtype))  # upstream scalar (1/GAS, loss scale, ...), in place
            from .linear import data_grad, write_weight_grad
            dh = data_grad(dl, weight).view(ctx.hshape)
            dW = None
            if ctx.needs_input_grad[1]:
                if not write_weight_grad(weight, dl, h2):
                    dW = dl.t() @ h2
            return dh, dW, None, None, None, None
        dh, dW = ctx.saved_tensors
        g = gout.to(torch.float32)
        dh = (dh * g.to(dh.dtype)).view(ctx.hshape)
        dW = (dW * g.to(dW.dtype)).to(ctx.wdtype)
        return dh, dW, None, None, None, None


def fused_linear_cross_entropy(h, weight, target, ignore_index=-100, chunk_tokens=None, reduction="mean"):
    """CE of ``h @ weight.T`` against ``target`` (ignore_index excluded); mean or sum."""
    if native.use_hip(h):
        return _FusedLinearXEnt.apply(h, weight, target, ignore_index, chunk_tokens, reduction)
    logits = torch.matmul(h, weight.t()).float()
    return F.cross_entropy(logits.reshape(-1, logits.shape[-1]), target.reshape(-1), ignore_index=ignore_index,
                           reduction=reduction)

"""Linear layer whose weight gradient is written straight into the ZeRO gradient buffer.

If a weight carries ``_sxe_grad_target`` (installed by the ZeRO optimizers), the backward weight-grad
GEMM writes its result directly where the optimizer wants it:
  * fp32 accumulator (single-rank / persistent units): ONE hipBLASLt GEMM with fp32 output and
    beta = 1 (``aten::addmm.dtype_out``) -- no bf16 ``p.grad`` tensor, no separate fp32 add pass,
    and micro-batch accumulation happens at fp32 precision inside the GEMM epilogue;
  * bf16 reduce-scatter staging slot (multi-rank units): the GEMM output IS the send buffer.
then calls ``_sxe_grad_done`` so the optimizer can launch the unit's reduce-scatter. Without a
target it behaves exactly like ``torch.nn.functional.linear``. (The reference's analogue is
Megatron-style ``gradient_accumulation_fusion``; DeepSpeed's ZeRO copies each ``p.grad`` into an
IPG bucket instead, stage_1_and_2.py:1137-1139.)
"""
import math
import os
import weakref

import torch
import torch.nn.functional as F

from . import native

# Large weight gradients that gemm_wgrad.hip does not take (bf16 reduce-scatter slots, few tokens of the largest weights, SXE_WGRAD=0) run
# faster as two HBM-speed transposes + a forward-layout ("TN") GEMM than in the token-major "NT" layout: hipBLASLt reaches
# 1.47-1.61 PF in TN vs 1.06-1.19 PF in NT on MI355X (tools/wgrad_layout_exp.py, tools/wgrad_tn_exp.py: -0.13 ms per 28672x4096 /
# 4096x14336 call, -0.47 ms for the 128256x4096 LM head, at K = 8192 tokens).
TN_MIN_ELEMS = int(os.environ.get("SXE_WGRAD_TN_MIN_ELEMS", 32 * 2**20))
# TN weight gradient into an fp32 accumulator: one fp32-output GEMM with beta = 1 (hipBLASLt "BSS"
# kernels), or (SXE_WGRAD_TN_FP32OUT=0) the bf16-output TN GEMM -- the faster kernel family -- plus
# an fp32 accumulate pass (what ops/mlp.py's weight_grad_tn does for the MLP weights)
TN_FP32_OUT = os.environ.get("SXE_WGRAD_TN_FP32OUT", "1") == "1"

# Decode-shaped products (<= 4 rows, no autograd) stream the weight through the MFMA skinny-GEMM
# kernel (csrc/kernels/skinny_gemm.hip) instead of hipBLASLt's general tiles. Measured on MI355X
# (tools/skinny_bench.py, profiles/skinny_bench.log), Llama-3-8B shapes, M = 1: o_proj 7.3 vs
# 11.8 us, gate_up 42 vs 56 us, down 24.8 vs 25.7 us, LM head 169 vs 180 us, QKV 12.4 vs 10.6 us. From 5 rows on
# stream_gemm.hip is the faster kernel (below); this one supports M <= 16.
SKINNY_MAX_M = int(os.environ.get("SXE_SKINNY_MAX_M", 4))


def _bias_ok(bias, weight):
    return bias is None or (bias.dtype == torch.bfloat16 and bias.shape == weight.shape[:1] and bias.is_contiguous())


def _skinny(x, weight, bias):
    K = x.shape[-1]
    if not (x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and weight.dim() == 2
            and weight.is_contiguous() and K % 8 == 0 and weight.data_ptr() % 16 == 0):
        return None
    if not _bias_ok(bias, weight):
        return None
    x2 = x.reshape(-1, K)
    if not (0 < x2.shape[0] <= SKINNY_MAX_M and x2.stride(1) == 1 and x2.stride(0) % 8 == 0
            and x2.data_ptr() % 16 == 0):
        return None
    native.require_hip()
    return torch.ops.sxe.skinny_gemm(x2, weight, bias).view(*x.shape[:-1], weight.shape[0])


# Batched decode: up to 32 rows take the weight-streaming kernel (csrc/kernels/stream_gemm.hip) where it is the faster one. A workgroup
# takes 16 columns, so the last round of them over the CUs decides, and long rows of the weight are where the library is good. us,
# library / streaming, 16 rows: 3072 x 2048 11.2 / 6.0, 4096 x 4096 14.9 / 9.6, 6144 x 4096 14.0 / 14.6, 28672 x 4096 60 / 47,
# 4096 x 14336 25.5 / 25.3, 15360 x 5120 33.5 / 34.2, 8192 x 8192 28.5 / 28.9; but 5120 x 5120 15.2 / 17.2, 5120 x 13824 31.9 / 39.1,
# 10240 x 8192 34.1 / 38.4, 2048 x 8192 12.7 / 13.0, 50264 x 768 18.3 / 20.6. 24 rows: 2048 x 2048 8.4 / 5.9, 4096 x 4096
# 12.8 / 11.6; but 5120 x 3072 11.6 / 13.5, 6144 x 4096 14.4 / 16.1, 1024 x 8192 11.6 / 15.1, 11264 x 2048 14.6 / 15.7. Wide weights, 32
# columns a workgroup, in a captured sequence of weights that are each read once, 24 rows: 32000 x 4096 60.6 / 52.2, 32000 x 2048 32.5 /
# 27.6, 128256 x 4096 191 / 186, 65536 x 4096 121 / 99, 16384 x 4096 31.8 / 29.8, 8192 x 3072 18.4 / 13.9 (32 rows: 64000 x 2560 60.7 /
# 62.4, 32000 x 3072 37.2 / 38.3); but 12288 x 4096 23.6 / 26.9, 9216 x 3072 17.1 / 19.5, 8192 x 4096 16.7 / 18.3. Long rows, a workgroup
# for every CU, weights that are each read once, 17 / 32 rows: the library is slow where rows are no whole pieces of 1 KB, 4096 x 11008 30.3 / 23.4,
# 29.8 / 24.9, 4096 x 14080 35.5 / 27.2, 34.7 / 29.4, or longer than 32 KB, 4096 x 18432 119 / 35, 121 / 37, 4096 x 28672 173 / 51, 177 / 55, else
# level with it, 4096 x 12288 23.5 / 24.5, 26.3 / 26.1, 4096 x 14336 27.6 / 28.0, 30.6 / 30.1, 4096 x 15360 28.4 / 29.9, 31.4 / 31.8 (in a
# decode step with four such layers, us a step, 17 rows 695 / 694, 20 701 / 695, 24 706 / 702, 28 714 / 712, 32 723 / 723); with
# 32 columns a workgroup 8192 x 5632 20.0 / 19.4, 20.9 / 20.3, 8192 x 12288 41.6 / 37.9, 42.6 / 40.4, 8192 x 28672 90.4 / 83.9, 103 / 90, 7936 x
# 11008 51.4 / 38.2, 52.8 / 39.5, but 8192 x 5120 18.8 / 19.0, 19.4 / 19.8. Not rows whose starts fall on the same channels, 24 rows, 4096 x 8192
# 17.9 / 18.7, 4096 x 16384 33.4 / 35.9, 8192 x 8192 29.9 / 33.2, nor 3840 x 15360 30.1 / 31.5, 12288 x 12288 64.2 / 66.6.
STREAM_ROWS, STREAM_ROWS_SMALL = 16, 32


def _full_rounds(workgroups):
    """Share of the CUs that are busy over the rounds that one workgroup a CU makes."""
    rounds = workgroups / 256
    return rounds / max(1, math.ceil(rounds))


def _stream_faster(rows, N, K):
    if rows > STREAM_ROWS:
        if K > 4096:
            if rows > STREAM_ROWS_SMALL or not 4096 <= N <= 8192 or N * K < 1 << 25 or (K <= 16384 and K % 8192 == 0):
                return False
            if N >= 6144:
                return K > 5120 and _full_rounds(N / 32) > 0.95
            return (K > 16384 or K % 512 != 0 or rows >= 20) and _full_rounds(N / 16) > 0.95
        return rows <= STREAM_ROWS_SMALL and K <= 4096 and (N <= 4096 or N * K <= 1 << 23 or ((N >= 16384 or K <= 3072)
                                                                                              and _full_rounds(N / 32) > 0.93))
    return not (K >= 5120 and N * K >= 1 << 24 and _full_rounds(N / 16) < 0.9) and not (K < 1024 and N > 16384)


def glu_faster(rows, weight):
    """Whether ``glu_linear`` beats the product and the activation's launch. e4m3: always (8 rows of 28672 x 4096 34 / 26 us with the
    product of skinny_gemm.hip). bf16, us, with the library's product / here: 8 rows 28672 x 4096 63 / 40; 16 rows 16384 x 2048 20.5 / 14.5, 28672 x
    4096 68 / 42, 36864 x 5120 90 / 70; 24 rows 10240 x 2560 19.7 / 18.7, 16384 x 3072 24.9 / 21.9, 28672 x 4096 55 / 46; 32 rows 28672 x 4096 58 / 48;
    but 24 rows 27648 x 5120 56 / 58. The line lies where four tiles a workgroup had it, and layers that chain their products do not ask; two
    tiles are ahead behind it as well: 16 rows 57344 x 8192 194 / 154, 24 rows 17920 x 2560 26.6 / 24.3, 7168 x 4096 18.6 / 16.6, 32 rows 22016 x 4096
    46 / 38."""
    if not isinstance(weight, torch.Tensor):
        return True
    N, K = weight.shape
    if rows > STREAM_ROWS and K <= 3072 and N <= 16384:
        return True
    return N * K <= 1 << 28 and (rows <= STREAM_ROWS or _full_rounds(N / 64) > 0.85)


def _streamable(x2, weight, bias, unit=8):
    return (x2.dtype == torch.bfloat16 and x2.stride(1) == 1 and x2.stride(0) % 8 == 0 and x2.data_ptr() % 16 == 0
            and weight.dim() == 2 and weight.stride(1) == 1 and weight.stride(0) % unit == 0 and weight.data_ptr() % 16 == 0
            and weight.shape[1] == x2.shape[1] and x2.shape[1] % unit == 0 and weight.shape[0] % 4 == 0 and weight.shape[0] > 0
            and x2.shape[1] > 0 and _bias_ok(bias, weight))


def _stream(x, weight, bias):
    if weight.dtype != torch.bfloat16 or not weight.is_cuda:
        return None
    rows = x.numel() // max(1, x.shape[-1])
    if rows <= SKINNY_MAX_M or weight.dim() != 2 or not _stream_faster(rows, *weight.shape):
        return None
    x2 = x.reshape(-1, x.shape[-1])
    if not _streamable(x2, weight, bias):
        return None
    native.require_hip()
    return torch.ops.sxe.stream_gemm(x2, weight, None, bias, False).view(*x.shape[:-1], weight.shape[0])


def glu_linear(x, weight):
    """silu(gate) * up of ``linear(x, weight)`` with weight = [gate | up], in ONE launch (stream_gemm.hip): up to 32 rows (16 of an
    FP8Weight), no autograd; None when not covered (``glu_faster``: where it pays). One rounding, of the result."""
    wk = _pro_weight(weight)
    if wk is None or SKINNY_MAX_M <= 0 or not x.is_cuda or x.requires_grad or x.dim() != 2 or not native.plain(x):
        return None
    w, sc = wk
    if not 0 < x.shape[0] <= (STREAM_ROWS_SMALL if sc is None else STREAM_ROWS) or w.shape[0] % 32:
        return None
    if not _streamable(x, w, None, 8 if sc is None else 16):
        return None
    return torch.ops.sxe.stream_gemm(x, w, sc, None, True)


def stream_weight(weight, rows, columns=16):
    """(w, scale) for the products of a decoder's layer that are chained without launches for its norms (``stream_res``, ``stream_glu``,
    ``stream_rope``, ``stream_head``), or None: a bf16 weight, up to 32 rows, or an FP8Weight, up to 16; its rows a multiple of ``columns``."""
    wk = _pro_weight(weight)
    if wk is None or SKINNY_MAX_M <= 0:
        return None
    w, sc = wk
    N, K = w.shape
    if not 0 < rows <= (STREAM_ROWS_SMALL if sc is None else STREAM_ROWS) or N % columns or N == 0 or K == 0 or K % (8 if sc is None else 16):
        return None
    return (w, sc) if w.is_cuda and w.data_ptr() % 16 == 0 and native.plain(w) else None


def chain_faster(rows, weights):
    """Whether a layer's products (qkv, o, gate | up, down; of MoE layers the first) gain by having its norms, residual sums and RoPE in their
    epilogues, three launches of ~4.7 us a layer, also where the library has the faster product. us a decode step of three layers (two from
    5120 on) and the head, launches of their own (up to 4 rows the norms in prologues of skinny_gemm.hip) / so, 1, 8, 16 and 32 rows: hidden 2048,
    ff 8192 184 / 168, 202 / 177, 208 / 188, 249 / 216; 3072, 8192 247 / 229, 265 / 234, 280 / 249, 324 / 297; 3584, 18944 386 / 345, 456 / 352,
    472 / 374, 729 / 458; 4096, 11008 350 / 332, 374 / 341, 409 / 377, 540 / 509; 4096, 14336 362 / 340, 382 / 355, 402 / 379, 470 / 455; 6144,
    16384, 16 and 32 rows 619 / 604, 688 / 659; 8192, 28672, 4 rows 868 / 756; e4m3 4096, 14336 265 / 252, 297 / 257, 339 / 301; 3072, 8192 187 / 178,
    219 / 183, 245 / 212; 2048, 8192 138 / 128, 172 / 143; 5120, 13824, 1 and 8 rows 263 / 226, 275 / 254. From 17 rows on not 5120, 13824 with 40 kv
    heads (8 rows 382 / 347, 32 rows 483 / 513), whose last round of the gate's workgroups is short. One row again, behind 900 keys, on another card:
    2048 177 / 154, 3072 241 / 217, 4096, 14336 356 / 322, e4m3 133 / 119, 172 / 161, 243 / 232; behind 64 keys 171 / 151, 234 / 205, 346 / 311, e4m3 124 /
    114, 167 / 149, 234 / 220."""
    if rows <= STREAM_ROWS or len(weights) == 1:
        return True
    N, K = weights[2][0].shape
    return K <= 4096 or N * K > 1 << 28 or _full_rounds(N / 64) > 0.85


def stream_res(x, wk, res, norm_weight):
    """h = res + x . w^T and what the next product takes of rms_norm(h) * norm_weight, in ONE launch (stream_gemm.hip):
    (bf16(h * norm_weight), h, sums of h^2 by tiles of 16 columns, of 8 for up to 8 rows of up to 2048 columns)."""
    return torch.ops.sxe.stream_gemm_res(x, wk[0], wk[1], None, res, norm_weight)


# Rows and columns of a weight that stream_gemm.hip merges the splits for in its own launch, however many there are: one sequence, three layers of
# hidden 2048, us a step with a launch for the merge / so: 4 kv heads 900 keys (8 splits) 163 / 157, 8000 (32) 180 / 172, 16000 (64) 204 / 197, 60000
# (128, 1 MB of partials) 282 / 279, e4m3 126 / 119, 152 / 146, 173 / 169, 247 / 247; 16 kv heads 16000 257 / 249; hidden 1024, 2 kv heads, 60000 (256)
# 248 / 240.
MERGE_COLUMNS = 2048


def stream_res_splits(parts, wk, res, norm_weight):
    """``stream_res`` of one row that ``paged_attention_parts`` has left in splits, weights of up to MERGE_COLUMNS each way."""
    return torch.ops.sxe.stream_gemm_res_splits(parts[0], parts[1], wk[0], wk[1], res, norm_weight)


def stream_glu(x, wk, sums, eps):
    """silu(gate) * up of the product of a normed input, x and ``sums`` of ``stream_res`` (None: x is normed)."""
    return torch.ops.sxe.stream_gemm_normed(x, wk[0], wk[1], sums, float(eps), True)


def stream_head(x, wk, sums, eps):
    """The product of a normed input in fp32."""
    return torch.ops.sxe.stream_gemm_normed(x, wk[0], wk[1], sums, float(eps), False)


def stream_rope(x, wk, sums, eps, rope, positions, cache, slots, nq, nkv):
    """q, k, v of a normed input [T, (nq + 2 nkv) * 128], q and k rotated, k and v in the paged cache as well."""
    return torch.ops.sxe.stream_gemm_rope(x, wk[0], wk[1], sums, float(eps), rope.cos, rope.sin, positions.reshape(-1).contiguous().long(),
                                          slots, cache, int(nq), int(nkv))


# Many rows: csrc/kernels/gemm_tn.hip, us, library / here. The library's kernels fit whole tiles of 256 rows (8192 rows, 28672 x 4096
# 1255 / 1285, 4096 x 4096 174 / 184) and many other counts, but by far not all: 6695 rows, 5120 x 5120 1.59 times as long, 7584, 4096 x 14336
# 1.68, 2716, 6144 x 4096 1.69, 8810, 4096 x 4096 1.57, 2588, 16384 x 3072 1.52; where it fits it is up to 10 % ahead (3072 x 3072, 1630 rows
# 39 / 44; 32000 x 4096, 4000 rows 0.94). From 1500 to 13000 rows the library takes 1.085 times as long on average (17 weights of 2048 x
# 2048 to 32000 x 4096, 14 counts each); further on 1.03 at equal weights, 1.01 to 1.02 in all, and more than 2 % less for every third count
# (3072 x 8192, 19089 rows 666 / 736).
# Fewer rows, long rows of the weight, whose products are split along them: 1.5 times on average, 40 rows, 8192 x 28672 127 / 88, 4096 x 14336
# 33 / 32, 200 rows 55 / 40, 1100 rows, 3072 x 8192 70 / 64; but up to 128 rows (few workgroups, or rows 32 KB apart) 64 rows, 8192 x 8192 33 / 39,
# 128 rows, 2048 x 8192 21 / 25, 33 rows, 2048 x 16384 0.74; others do not: 600 rows, 5120 x 3072 26 / 29, 4096 x 4096 28 / 31.
# From 1025 rows to 1500, wide weights: 1.07 times on average (20 of them, 11 counts each), 1040 rows, 6144 x 4096 55 / 49, 1208, 50304 x
# 2048 1.27, 1351, 7680 x 2560 1.14, 1237, 28672 x 8192 0.94; but 4608 x 4096 0.96, 4096 x 4096 0.89, 3072 x 3072 0.92; up to 1024 rows 0.96.
TILED_ROWS, TILED_ROWS_MOST = 1500, 13000
TILED_ROWS_WIDE, TILED_WIDE, TILED_WIDE_WORK = 1024, 6144, 18 * 10 ** 6
# SwiGLU of the products in one launch, us, product and activation / here: 16384 x 2048, 330 rows 35 / 29, 2100 rows 144 / 112;
# 28672 x 4096, 330 rows 85 / 73, 1040 rows 226 / 200, 7588 rows 1390 / 1250; but 240 rows of 16384 x 3072 38 / 43, 72 of 28672 x 4096
# 59 / 67, and of weights beyond 2^28 elements 493 rows, 57344 x 8192 0.90, 1423 rows 1.02, 3000 rows 1.12
TILED_GLU_ROWS, TILED_GLU_ROWS_LARGE = 300, 1024


def _tiled_faster(rows, N, K):
    if N < 2048 or K < 2048:
        return False
    if rows >= TILED_ROWS or (rows > TILED_ROWS_WIDE and N >= TILED_WIDE and N * K >= TILED_WIDE_WORK):
        return rows < TILED_ROWS_MOST and rows % 256 != 0
    if rows <= 128 and (N >= K or K % 16384 == 0 or (rows > 64 and N < 3072)):
        return False
    return STREAM_ROWS_SMALL < rows and K >= 8192 and N <= K


def _tileable(x2, weight, bias=None):
    """The operands that gemm_tn.hip reads: rows of whole 128-byte pieces that start on 16 bytes, offsets in 32 bits."""
    N, K = weight.shape
    return (x2.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and weight.is_cuda and x2.stride(1) == 1 and weight.stride(1) == 1
            and x2.stride(0) % 8 == 0 and weight.stride(0) % 8 == 0 and x2.stride(0) >= K and weight.stride(0) >= K and x2.data_ptr() % 16 == 0
            and weight.data_ptr() % 16 == 0 and x2.shape[1] == K and K % 64 == 0 and N % 16 == 0 and x2.shape[0] < 1 << 30
            and x2.stride(0) < 1 << 23 and N * weight.stride(0) < 1 << 31
            and (bias is None or (_bias_ok(bias, weight) and bias.data_ptr() % 16 == 0)))


def _tiled(x, weight, bias, faster=False):
    """gemm_tn.hip, where it covers the operands and is the faster one (``faster``: as the caller has found), else None."""
    if weight.dim() != 2 or not (faster or _tiled_faster(x.numel() // max(1, x.shape[-1]), *weight.shape)):
        return None
    x2 = x.reshape(-1, x.shape[-1])
    if not _tileable(x2, weight, bias):
        return None
    native.require_hip()
    if x.dim() == 2 or x.is_contiguous():  # the result is no view: autograd functions return it, and their callers write to it
        return torch.ops.sxe.gemm_tn(x, weight, bias, False)
    return torch.ops.sxe.gemm_tn(x2, weight, bias, False).view(*x.shape[:-1], weight.shape[0])


def _own_products(x, weight, bias=None):
    """Whether ``product`` may run own kernels: no graph is recorded, nobody follows the call by its operators."""
    return (SKINNY_MAX_M > 0 and x.is_cuda and not torch.is_grad_enabled() and native.plain(x, weight, bias) and (x.dim() == 2 or x.is_contiguous())
            and (not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") == torch.bfloat16))


# Products of training with narrow weights, up to this many multiplications. A call of the library costs the host 19.5 us whatever its size, one
# of gemm_tn.hip 6, which is what steps of this size wait for: GPT-2, four layers, ZeRO-1, us a step with the library / here, 64 tokens 4790 /
# 4095, 1024 4288 / 3728, 2100 5035 / 4629, 4096 4446 / 3908, 7000 5943 / 5958. On the device most of them take longer, the step's kernels 1720 /
# 1810, 2280 / 2410, 3360 / 3360, 3840 / 3890, 5940 / 6040 together; single ones, 2048 rows, 2304 x 768 16.6 / 13.8, 3072 x 768 15.6 / 14.8,
# 768 x 768 9.3 / 11.9, 768 x 3072 19 / 25, 512 x 2048 12 / 24, 300 rows 7.7 / 11.5, 7.9 / 11.6, 7.0 / 11.2, 9.1 / 15.2, 8.4 / 12.6. So not where
# a graph is captured, whose replays cost the host nothing, nor behind this limit: 8192 rows, 768 x 3072 39 / 36, 4096 x 1024 57 / 60,
# 8192 x 1536 158 / 168.
NARROW_WORK = 10 ** 10


def _narrow(rows, N, K):
    """A weight that ``_tiled_faster`` leaves to the library for its width, and a product whose call costs more than its work."""
    return (N < 2048 or K < 2048) and N >= 512 and K >= 512 and rows > STREAM_ROWS_SMALL and rows * N * K <= NARROW_WORK


_capturing = torch.cuda.is_current_stream_capturing


def _eager_own(rows, N, K):
    """Products of eager serving passes of 33 to 768 rows: these wait for the host, whom a call of the library costs 14 us more; on the device own ones
    take (us, library / here) at 2048 x 2048, 64 to 512 rows 12 / 14 - 13 / 24, 3072 x 2048 12 / 15 - 15 / 24, 4096 x 4096 15 / 19 - 29 / 31, 6144 x
    4096 18 / 21 - 37 / 40, 16384 x 3072 26 / 32 - 53 / 51, beside 40 us and more of a layer's other kernels. So not where a graph is captured,
    nor beyond NARROW_WORK, where the device is what a pass waits for. us a pass of two layers: prompts of 26 - 30 tokens, 1b 677 / 484, 136 and 140,
    3b 652 / 568, 51 of 31 - 56, 8b 804 / 716; 256 tokens at a time beside 7 sequences, 8b 1550 / 1203."""
    return STREAM_ROWS_SMALL < rows <= 768 and N >= 512 and K >= 512 and rows * N * K <= NARROW_WORK and not _capturing()


def product(x, weight, bias=None):
    """``F.linear`` for the inside of autograd functions: no graph is built where it runs own kernels (``_tiled``)."""
    rows = x.numel() // max(1, x.shape[-1])
    if weight.dim() == 2:
        faster = _tiled_faster(rows, *weight.shape)
        if (faster or _narrow(rows, *weight.shape)) and _own_products(x, weight, bias) and (faster or not _capturing()):
            y = _tiled(x, weight, bias, True)
            if y is not None:
                return y
    return F.linear(x, weight, bias)


def glu_tiled(x, weight):
    """silu(gate) * up of ``linear(x, weight)`` with weight = [gate | up], bf16, in ONE launch (gemm_tn.hip): many rows, no autograd; None
    where the product and the activation's launch are the better or only form. One rounding, of the result."""
    if (not isinstance(weight, torch.Tensor) or weight.dim() != 2 or x.dim() != 2 or not x.is_cuda or x.requires_grad or not native.plain(x, weight)
            or x.shape[0] <= TILED_GLU_ROWS or weight.shape[0] < 8192 or weight.shape[1] < 2048 or not _tileable(x, weight)
            or (weight.numel() > 1 << 28 and x.shape[0] <= TILED_GLU_ROWS_LARGE) or SKINNY_MAX_M <= 0 or torch.is_autocast_enabled("cuda")):
        return None
    native.require_hip()
    return torch.ops.sxe.gemm_tn(x, weight, None, True)


def _pro_weight(weight):
    """(w, scale) for the fused-prologue skinny kernels: a bf16 [N, K] tensor or an FP8Weight."""
    if isinstance(weight, torch.Tensor):
        if weight.dtype == torch.bfloat16 and weight.dim() == 2 and weight.is_contiguous() and weight.data_ptr() % 16 == 0:
            return weight, None
        return None
    from .fp_quantizer import FP8Weight
    if not isinstance(weight, FP8Weight):  # other quantized formats (MX, FP6/FP4 planes, int) run unfused
        return None
    q, sc = weight.q, weight.scale
    if q.element_size() == 1 and q.dim() == 2 and q.is_contiguous():
        return q.view(torch.uint8), sc
    return None


def _pro_ok(x, rows_max=4):
    return (x.is_cuda and x.dtype == torch.bfloat16 and x.dim() == 2 and 0 < x.shape[0] <= rows_max
            and x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0 and not x.requires_grad)


def fused_rms_linear(x, residual, norm_weight, eps, weight, bias=None):
    """Decode (<= 4 rows): ``linear(rms_norm(x + residual), weight)`` in ONE launch
    (skinny_gemm.hip PRO_RMS). Returns (y, h = x + residual) -- h is x itself without a residual --
    or None when the fused kernel does not cover the operands (the caller runs the unfused ops)."""
    wk = _pro_weight(weight)
    if wk is None or not _pro_ok(x) or norm_weight.dtype != torch.bfloat16 or not norm_weight.is_contiguous():
        return None
    if residual is not None and (residual.shape != x.shape or residual.stride() != x.stride()
                                 or residual.dtype != x.dtype):
        return None
    w, sc = wk
    if x.shape[1] != w.shape[1]:
        return None
    y, h = torch.ops.sxe.skinny_gemm_pro(x, residual, norm_weight, float(eps), w, sc, bias, 1)
    return y, (h if residual is not None else x)


# Rows x K up to which the GEMM builds its normed input itself; every workgroup does. us, one launch / norm and streaming kernel:
# bf16, 1 x 4096 47.0 / 55.0, 2 x 4096 51.1 / 54.3, 4 x 2048 20.1 / 21.8, 3 x 3072 27.8 / 27.0, 4 x 4096 59.0 / 54.8;
# e4m3, 1 x 4096 31.4 / 34.2, 1 x 3072 16.2 / 18.3, 2 x 4096 34.5 / 34.1, 4 x 2048 16.8 / 14.1
RMS_GLU_BF16, RMS_GLU_FP8 = 8192, 4096


def fused_rms_glu(x, residual, norm_weight, eps, weight):
    """Decode (<= 4 rows): ``silu(gate) * up`` of ``linear(rms_norm(x + residual), [gate | up])`` in ONE launch (skinny_gemm.hip
    PRO_RMS with the SwiGLU epilogue; one rounding, of the result). Returns (y, h) like ``fused_rms_linear``, or None."""
    wk = _pro_weight(weight)
    if (wk is None or not _pro_ok(x) or norm_weight.dtype != torch.bfloat16 or not norm_weight.is_contiguous()
            or x.shape[1] != wk[0].shape[1] or wk[0].shape[0] % 16
            or x.numel() > (RMS_GLU_BF16 if wk[1] is None else RMS_GLU_FP8)):
        return None
    if residual is not None and (residual.shape != x.shape or residual.stride() != x.stride()
                                 or residual.dtype != x.dtype):
        return None
    y, h = torch.ops.sxe.skinny_gemm_pro(x, residual, norm_weight, float(eps), wk[0], wk[1], None, 3)
    return y, (h if residual is not None else x)


def fused_rms_rope_linear(x, residual, norm_weight, eps, weight, rope, positions, cache, slots, nq, nkv):
    """Decode (<= 4 rows) QKV projection in ONE launch: residual + RMSNorm prologue, GEMM, and the
    RoPE + paged-KV-append epilogue (skinny_gemm.hip ``skinny_gemm_pro_rope``; head dim 128).
    Returns (qkv with q / k rotated, h) -- the rotated k and v are already in ``cache`` -- or None
    when not covered (the caller runs fused_rms_linear + rope_kv_cache_append)."""
    wk = _pro_weight(weight)
    if (wk is None or not _pro_ok(x) or norm_weight.dtype != torch.bfloat16 or not norm_weight.is_contiguous()
            or rope.cos.shape[-1] != 64 or not cache.is_contiguous() or cache.dim() != 5 or cache.shape[-1] != 128):
        return None
    if residual is not None and (residual.shape != x.shape or residual.stride() != x.stride()
                                 or residual.dtype != x.dtype):
        return None
    w, sc = wk
    if x.shape[1] != w.shape[1] or w.shape[0] != (nq + 2 * nkv) * 128:
        return None
    y, h = torch.ops.sxe.skinny_gemm_pro_rope(x, residual, norm_weight, float(eps), w, sc, rope.cos, rope.sin,
                                              positions.reshape(-1).contiguous().long(), slots, cache, int(nq), int(nkv))
    return y, (h if residual is not None else x)


def fused_swiglu_linear(gu, weight, bias=None):
    """Decode (<= 4 rows): ``linear(silu(gu[:, :I]) * gu[:, I:], weight)`` in ONE launch
    (skinny_gemm.hip PRO_SWIGLU); None when not covered."""
    wk = _pro_weight(weight)
    if wk is None or not _pro_ok(gu):
        return None
    w, sc = wk
    if gu.shape[1] != 2 * w.shape[1]:
        return None
    return torch.ops.sxe.skinny_gemm_pro(gu, None, None, 0.0, w, sc, bias, 2)[0]


def fused_merge_linear(part_o, part_ml, weight, bias=None):
    """Decode (<= 4 rows): ``linear(merge(part_o, part_ml), weight)`` in ONE launch -- the
    flash-decoding merge of paged attention's KV-split partials runs as the o_proj skinny GEMM's
    prologue (skinny_gemm.hip PRO_MERGE). None when the weight is not covered (bf16 / FP8 only)."""
    wk = _pro_weight(weight)
    if wk is None or not part_o.is_cuda or part_o.shape[1] > 4:
        return None
    w, sc = wk
    if w.shape[1] != part_o.shape[2] * part_o.shape[3]:
        return None
    return torch.ops.sxe.skinny_gemm_merge(part_o, part_ml, w, sc, bias)


def fused_addnorm_linear(y, res, norm_weight, alpha, eps, offset, weight):
    """Decode (<= 4 rows), norm after a scaled 32-bit residual sum, in ONE launch (skinny_gemm.hip
    PRO_ADDNORM): v = alpha r + y, returns ``(linear(rms(v) (offset + norm_weight), weight), state)``. ``res`` is
    either r itself (fp32 tensor) or the ``state`` (v, 1 / rms(v), norm_weight) of an earlier call, whose
    normalised sum is r. None when not covered."""
    wk = _pro_weight(weight)
    if (wk is None or wk[1] is not None or not _pro_ok(y) or not y.is_contiguous() or y.shape[1] != wk[0].shape[1]
            or y.shape[1] % 8 or norm_weight.dtype != torch.bfloat16 or norm_weight.data_ptr() % 16
            or y.numel() * 2 > 144 * 1024):
        return None
    h, rinv, rw = res if isinstance(res, tuple) else (res, None, None)
    out, v, ri = torch.ops.sxe.skinny_gemm_addnorm(y, h, rinv, rw, norm_weight, float(alpha), float(eps), float(offset), wk[0])
    return out, (v, ri, norm_weight)


def fused_gatesum_linear(part, gate, weight):
    """Decode (<= 4 rows): ``linear(sigmoid(gate) * part.sum(0), weight)`` in ONE launch (skinny_gemm.hip
    PRO_GATESUM); part fp32 [splits, M, K]. None when not covered."""
    wk = _pro_weight(weight)
    if (wk is None or wk[1] is not None or part.shape[1] > 4 or part.shape[2] % 8 or gate.stride(0) % 8
            or gate.data_ptr() % 16 or part.shape[1] * part.shape[2] * 2 > 144 * 1024):
        return None
    return torch.ops.sxe.skinny_gemm_gatesum(part, gate, wk[0])


# wider products run more workgroups than fit at once, each building the input again
SANDWICH_MAX_N = int(os.environ.get("SXE_SANDWICH_MAX_N", 8192))


def sandwich_fusable(x, y, *weights):
    """Whether the decode kernels with the sandwich-norm prologue (csrc/include/sxe_sandwich.h) take these rows:
    up to 4, M K <= 8192."""
    M, K = x.shape
    return (0 < M <= 4 and K % 8 == 0 and M * K <= 8192 and x.is_contiguous() and y.is_contiguous()
            and all(t.dtype == torch.bfloat16 and t.is_contiguous() and t.data_ptr() % 16 == 0 for t in (y, *weights)))


def fused_sandwich_linear(x, y, post_weight, next_weight, eps, slots, add, weight):
    """Decode (<= 4 rows): ``sandwich_norm`` (ops/residual_norm.py) and the projection that reads its result in
    ONE launch (skinny_gemm.hip PRO_SANDWICH): (linear(h, weight), x'). None when not covered."""
    wk = _pro_weight(weight)
    if (wk is None or wk[1] is not None or wk[0].shape[0] > SANDWICH_MAX_N or x.shape[1] != wk[0].shape[1]
            or not sandwich_fusable(x, y, post_weight, next_weight)):
        return None
    return torch.ops.sxe.skinny_gemm_sandwich(x, y, post_weight, next_weight, slots, add, float(eps), wk[0])


def fused_gatenorm_linear(x, norm_weight, gate, eps, weight):
    """Decode (<= 4 rows): ``linear(gated_rms_norm(x, norm_weight, gate), weight)`` in ONE launch (skinny_gemm.hip
    PRO_GATENORM). None when not covered."""
    wk = _pro_weight(weight)
    if (wk is None or wk[1] is not None or not _pro_ok(x) or not x.is_contiguous() or x.shape[1] != wk[0].shape[1]
            or x.shape[1] % 8 or gate.stride(0) % 8 or gate.data_ptr() % 16 or norm_weight.data_ptr() % 16
            or x.numel() * 2 > 144 * 1024):
        return None
    return torch.ops.sxe.skinny_gemm_gatenorm(x, norm_weight, gate, float(eps), wk[0])


# Hand-written weight-gradient GEMM (csrc/kernels/gemm_wgrad.hip: both operands read transposed through LDS, fp32 C): no transposed
# copies of dY / X, any number of tokens. Beside the library's fp32-output product, with transposed copies or without, it is the faster one
# from 768 x 768 to 128256 x 4096 at 128 - 16384 tokens (figures there), but for 1024 and 2048 tokens of 2048 x 2048 (24 us for 22, 34 for
# 31) and what ``_wgrad_faster`` leaves out.
SXE_WGRAD = os.environ.get("SXE_WGRAD", "1") == "1"


def _sxe_wgrad_ok(gy2, x2, buf):
    """gy2 [.., T, M], x2 [.., T, N], buf [.., M, N]: one product, or one for every expert."""
    if not (SXE_WGRAD and gy2.is_cuda and buf.dtype == torch.float32 and gy2.dtype == torch.bfloat16
            and x2.dtype == torch.bfloat16 and buf.is_contiguous() and gy2.stride(-1) == 1 and x2.stride(-1) == 1):
        return False
    K, M, N = gy2.shape[-2], gy2.shape[-1], x2.shape[-1]
    if M % 8 or N % 8 or M < 64 or N < 64 or K == 0 or gy2.stride(-2) % 8 or x2.stride(-2) % 8:
        return False
    if not native.plain(gy2, x2):  # traced: no memory to look at, sizes whose operands start on 16 bytes
        return K % 128 == 0 and M % 256 == 0 and N % 256 == 0
    return (gy2.data_ptr() % 16 == 0 and x2.data_ptr() % 16 == 0 and buf.data_ptr() % 16 == 0 and max(gy2.stride(-2), x2.stride(-2)) < 1 << 24
            and min(gy2.stride(-2), x2.stride(-2)) > 0 and max(M, N, K) < 1 << 30)


def _wgrad_faster(T, M, N):
    """us, the library with transposed copies or without / own, each call on another dW: 28672 x 4096, 128 tokens 200 / 196, 512 262 / 241;
    128256 x 4096, 128 845 / 773, 2048 2298 / 2096, 8192 7361 / 6912; 57344 x 8192, 512 947 / 920, 2048 1898 / 1894; but few tokens of
    large weights of rows 32 KB apart, 57344 x 8192, 128 754 / 832, 256 800 / 841, 16384 x 8192 224 / 240, 242 / 251."""
    return T >= 512 or M * N < 1 << 27 or N % 8192 != 0


def _tn_ok(gy2, x2):
    return (gy2.is_cuda and gy2.dtype == torch.bfloat16 and x2.dtype == torch.bfloat16 and TN_MIN_ELEMS > 0
            and gy2.shape[1] * x2.shape[1] >= TN_MIN_ELEMS and gy2.shape[0] % 64 == 0 and gy2.shape[1] % 64 == 0
            and x2.shape[1] % 64 == 0 and gy2.is_contiguous() and x2.is_contiguous())


# Data-gradient GEMMs dX = dY W run in hipBLASLt's "NN" layout at 1.03-1.35 PF on MI355X; with W^T
# materialised by the HBM-speed transpose they run in the forward layout at 1.25-1.56 PF
# (tools/gemm_layout_bench.py, profiles/gemm_layout.log: net -0.03..-0.06 ms per Llama-3-8B layer
# GEMM, -0.48 ms for the LM head, at 8192 tokens). The transpose reads/writes only the weight.
DGRAD_WT_MIN_ELEMS = int(os.environ.get("SXE_DGRAD_WT_MIN_ELEMS", 16 * 2**20))


# The transposed weights are constant between optimizer steps: with gradient accumulation each
# micro-step's backward (and each chunk of a chunked LM-head loss) would transpose the same weight
# again (the transpose kernel was 1.7 % of the Llama-3-8B ZeRO-3 step at 2 micro-steps). The engine
# enables this cache for gradient_accumulation_steps > 1 and clears it after every optimizer step
# and checkpoint load; it holds at most SXE_WT_CACHE_GB of transposes (ZeRO-3 models whose
# gathered weights do not stay resident simply stop caching at the cap).
WT_CACHE = False
WT_CACHE_MAX_BYTES = int(float(os.environ.get("SXE_WT_CACHE_GB", "20")) * 2**30)
_wt_cache = {}
_wt_cache_bytes = 0


def invalidate_transposed_weights():
    global _wt_cache_bytes
    _wt_cache.clear()
    _wt_cache_bytes = 0


def _transpose16(t):
    native.require_hip()
    return torch.ops.sxe.transpose16(t)


def _transposed_weight(w):
    global _wt_cache_bytes
    if not WT_CACHE or not isinstance(w, torch.nn.Parameter):
        return _transpose16(w)
    hit = _wt_cache.get(id(w))
    # a weight rebound to other storage (ZeRO-3 gather into a new buffer) or bumped by an in-place
    # write through the Parameter itself misses instead of returning a stale transpose; writers that
    # go through other views of a flat buffer call invalidate_transposed_weights()
    if (hit is not None and hit[0]() is w and hit[1].shape == w.shape[::-1] and hit[2] == w.data_ptr()
            and hit[3] == w._version):
        return hit[1]
    if hit is not None:
        _wt_cache.pop(id(w))
        _wt_cache_bytes -= hit[1].numel() * hit[1].element_size()
    wt = _transpose16(w)
    nbytes = wt.numel() * wt.element_size()
    if _wt_cache_bytes + nbytes <= WT_CACHE_MAX_BYTES:
        _wt_cache[id(w)] = (weakref.ref(w), wt, w.data_ptr(), w._version)
        _wt_cache_bytes += nbytes
    return wt


def transposed_weight_cache_bytes():
    return _wt_cache_bytes


def configure_transposed_weight_cache(enabled, free_bytes=None):
    """Turn the cache on / off; with ``free_bytes`` (free HBM after the engine is built) the cap is
    at most a quarter of it, so the cache never takes memory a configuration needs to fit."""
    global WT_CACHE, WT_CACHE_MAX_BYTES
    WT_CACHE = bool(enabled)
    cap = int(float(os.environ.get("SXE_WT_CACHE_GB", "20")) * 2**30)
    if free_bytes is not None:
        cap = min(cap, int(free_bytes) // 4)
    WT_CACHE_MAX_BYTES = cap
    invalidate_transposed_weights()
    return cap


def _wt_few_faster(rows, N, K):
    """Whether fewer than 2048 rows pay for the transpose of w [N, K], too: where the product sums over many columns and gemm_tn.hip takes
    it. us, NN / transpose and own product: 256 rows, 28672 x 4096 206 / 171, 16384 x 2048 81 / 60, 1000 rows 350 / 268, 141 / 95, 32000 x
    3072 314 / 261; 1819 rows, 16384 x 2048 1.18, 1808, 32000 x 3072 1.49; but 1962 rows, 28672 x 3072 0.82; 1371 rows, 28672 x 4096
    308 / 338; 512 rows, 16384 x 4096 0.94, 57344 x 4096, 640 rows 0.74, 16384 x 8192 0.70, 400 rows, 128256 x 4096 829 / 1022."""
    if not 256 <= rows <= 1900 or not 16384 <= N <= 49152 or not _tiled_faster(rows, K, N):
        return False
    return K <= 3072 or (K <= 5120 and N >= 20480 and rows <= 1280)


def _narrow_data_grad(gy, w):
    """gy @ w of ``_narrow`` weights: up to 1280 rows of the weight by the product that reads them as they lie (experts_kn_tile.hip, one
    expert), else with the transpose, which the splits of gemm_tn.hip make up for. us on the device, library / as they lie / transposed,
    2048 rows: 768 x 3072 18 / 17 / 21, 768 x 768 12 / 14 / 15, 1280 x 5120 36 / 32 / 35, 2304 x 768 24 / 28 / 27, 3072 x 768 30 / 35 / 28,
    300 rows 8.7 / 13.7 / 17, 7.3 / 13 / 14, 14 / 19 / 27, 11.5 / 27 / 19, 14 / 33 / 20; on the host 19 / 8 / 13, which decides, as above.
    None where they do not cover the operands and where a graph is captured."""
    N, K = w.shape
    if not (_narrow(gy.numel() // max(1, gy.shape[-1]), N, K) and gy.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and N % 64 == 0
            and K % 64 == 0 and gy.is_contiguous() and w.is_cuda and w.is_contiguous() and _own_products(gy, w)
            and gy.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0 and not _capturing()):  # last: compilation has no memory to look at
        return None
    native.require_hip()
    if N <= 1280:
        return torch.ops.sxe.expert_mm_kn(gy.view(1, -1, N), w.unsqueeze(0)).view(*gy.shape[:-1], K)
    return torch.ops.sxe.gemm_tn(gy, _transposed_weight(w), None, False)


def data_grad(gy, w):
    """dX = gy @ w for w [N, K] (gy [..., N])."""
    if (DGRAD_WT_MIN_ELEMS > 0 and gy.is_cuda and gy.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
            and w.dim() == 2 and w.is_contiguous() and w.numel() >= DGRAD_WT_MIN_ELEMS and w.shape[0] % 64 == 0
            and w.shape[1] % 64 == 0):
        rows = gy.numel() // gy.shape[-1]
        if rows >= 2048 or (_wt_few_faster(rows, *w.shape) and gy.is_contiguous() and _own_products(gy, w) and gy.data_ptr() % 16 == 0):
            return product(gy, _transposed_weight(w))
    if gy.is_cuda and w.dim() == 2:
        dx = _narrow_data_grad(gy, w)
        if dx is not None:
            return dx
    return torch.matmul(gy, w)


def grad_target(w):
    """The optimizer's direct weight-grad target of ``w`` (``_sxe_grad_target``), or None when the
    gradient must take autograd's ``.grad`` path instead: a partial gradient of a tiled / recomputed
    sub-graph (``_sxe_grad_partial``, set by sequence/tiled.py for every tile but the last -- the
    reference's ``ds_grad_is_ready = False``, runtime/sequence_parallel/ulysses_sp.py:720-724), or a
    ``.grad`` that already holds such partial sums (the last tile adds into it, and the ZeRO hook
    then delivers the total once)."""
    tgt = getattr(w, "_sxe_grad_target", None)
    if tgt is None or getattr(w, "_sxe_grad_partial", False) or w.grad is not None:
        return None
    return tgt


def drop_grad_target(p):
    """Give the gradient of ``p`` back to autograd: nothing of the optimizer's direct target stays on the parameter."""
    for a in ("_sxe_grad_target", "_sxe_grad_done", "_sxe_grad_local"):
        p.__dict__.pop(a, None)


def _accumulates(ctx, p):
    """Whether the backward that runs ``ctx`` adds the gradient of ``p`` up: not ``torch.autograd.grad``, which returns it, nor a backward
    of other ``inputs``. 1 us."""
    for node, _ in ctx.next_functions:
        if node is not None and getattr(node, "variable", None) is p:
            try:
                return torch._C._will_engine_execute_node(node)
            except RuntimeError:  # the gradient of p itself is asked for
                return False
    return False


def local_grad_target(p, ctx):
    """``grad_target`` of a parameter whose gradient only this rank ever adds up, in fp32 (``_sxe_grad_local``), in the backward of
    ``ctx``, whose gradient the caller has found ``native.plain``: (buffer, whether it holds a sum), for gradients that may come in several
    pieces or besides autograd's. None elsewhere, where hooks of the parameter's gradient want to see it, and where the caller of
    autograd does."""
    if (p is None or not getattr(p, "_sxe_grad_local", False) or p._backward_hooks
            or len(getattr(p, "_post_accumulate_grad_hooks", None) or ()) > 1 or not _accumulates(ctx, p)):
        return None
    tgt = grad_target(p)
    if tgt is None:
        return None
    buf, accumulate = tgt(p)
    return (buf, bool(accumulate)) if buf.dtype == torch.float32 and buf.is_contiguous() else None


def keep_local(p):
    """``p`` for an autograd function to ask for its target in the backward, if it may have one (not a saved tensor: its values are not
    read, and may change until then)."""
    return p if getattr(p, "_sxe_grad_local", False) else None


# Elements up to which column sums go into the optimizer's buffer by colsum.hip whether it is the faster reduction or not: what follows a
# general one (autograd's accumulation and the conversion, two launches and 20 us of the host) costs more than it gains. us, general /
# kernel: 128 x 768 6.6 / 3.6, 64 x 50257 5.6 / 10.1, 33 x 65544 4.9 / 8.3, 2048 x 1001 13 / 22; behind it 2048 x 3001 23 / 28, 1000 x 50257
# 32 / 72, 2048 x 50257 60 / 134, 16 x 1048576 6 / 83.
BIAS_GRAD_ELEMS = 1 << 22


def write_bias_grad(b, gy2, ctx):
    """The column sums of gy2 into the optimizer's buffer of ``b`` (``keep_local``), in fp32: one launch instead of the sum, autograd's
    accumulation and a conversion. True if written."""
    if b is None or not (gy2.is_cuda and gy2.dtype in (torch.bfloat16, torch.float16, torch.float32) and gy2.stride(1) == 1
                         and native.plain(gy2)) or torch.is_grad_enabled() or not (gy2.numel() <= BIAS_GRAD_ELEMS or _colsum_faster(gy2)):
        return False
    tgt = local_grad_target(b, ctx)
    if tgt is None:
        return False
    native.require_hip()
    torch.ops.sxe.column_sum_(gy2, tgt[0].view(-1), tgt[1])
    b._sxe_grad_done(b)
    return True


def write_weight_grad(w, gy2, x2):
    """dW = gy2^T @ x2 into the optimizer-provided target of `w`; returns True if handled."""
    tgt = grad_target(w)
    if tgt is None:
        return False
    buf, accumulate = tgt(w)
    if _sxe_wgrad_ok(gy2, x2, buf) and _wgrad_faster(gy2.shape[0], gy2.shape[1], x2.shape[1]):
        torch.ops.sxe.wgrad_gemm_(gy2, x2, buf, 1.0, bool(accumulate))
    elif _tn_ok(gy2, x2) and buf.is_contiguous():
        a, b = torch.ops.sxe.transpose16(gy2), torch.ops.sxe.transpose16(x2).t()
        if buf.dtype == gy2.dtype and not accumulate:
            torch.mm(a, b, out=buf)  # the reduce-scatter staging slot of a multi-rank unit
        elif buf.dtype == torch.float32 and TN_FP32_OUT:
            # fp32-out TN GEMM accumulating in its epilogue (beta = 1): no bf16 dW round trip and no
            # separate fp32 add pass (28672x4096 at 8192 tokens: 1.62 vs 1.74 ms, wgrad_tn_fp32_exp)
            torch.ops.aten.addmm.dtype_out(buf, a, b, torch.float32, beta=1 if accumulate else 0, alpha=1, out=buf)
        else:
            dw = torch.mm(a, b).view_as(buf)
            buf.add_(dw) if accumulate else buf.copy_(dw)
    elif buf.dtype == torch.float32 and gy2.dtype != torch.float32:
        if gy2.is_cuda:
            torch.ops.aten.addmm.dtype_out(buf, gy2.t(), x2, torch.float32, beta=1 if accumulate else 0, alpha=1,
                                           out=buf)
        else:  # CPU processes (gloo plumbing runs): no fp32-out GEMM for 16-bit inputs there
            dw = (gy2.t() @ x2).float()
            buf.add_(dw) if accumulate else buf.copy_(dw)
    elif accumulate:
        buf.addmm_(gy2.t(), x2)
    else:
        torch.mm(gy2.t(), x2, out=buf)
    w._sxe_grad_done(w)
    return True


def _autocast_dtype(x):
    """The torch.autocast compute dtype active for ``x``'s device, or None."""
    dev = x.device.type
    if dev in ("cuda", "cpu") and torch.is_autocast_enabled(dev):
        return torch.get_autocast_dtype(dev)
    return None


COLSUM_ROWS = 256


def _colsum_faster(x):
    """Whether csrc/kernels/colsum.hip beats the general reduction, us, general / kernel: bf16 256 x 768 8.6 / 3.5, 2048 x 3072
    17.0 / 5.4, 2048 x 14336 99 / 12, 16384 x 8192 49 / 46; but 16 x 1048576 5.9 / 79, 8192 x 28672 80 / 93, and where rows do not
    start on 16 bytes 2048 x 1001 12.9 / 21.8, 2048 x 50257 60 / 133, from 4096 rows on 22 / 16 at 1001, 48 / 23 at 3001 columns.
    Steps of fewer rows are bound by the host, where the kernel costs 3 us more: 128 x 768 5.8 / 3.3 on the device, 5.5 / 8.3 there."""
    R, N = x.shape
    if N % 8 or x.stride(0) * x.element_size() % 16 or x.data_ptr() % 16:
        return R >= 4096 and 64 <= N <= 8192
    return R >= COLSUM_ROWS and N <= 65536 and (N <= 8192 or R < 8192)


def column_sum(x, dtype):
    """``x.sum(0)`` of [R, N] in ``dtype``, accumulated in fp32 (csrc/kernels/colsum.hip; fp64, recorded sums and sizes where it is
    not the faster one: torch)."""
    if (x.is_cuda and x.shape[0] >= COLSUM_ROWS and x.dtype in (torch.bfloat16, torch.float16, torch.float32) and x.stride(1) == 1
            and dtype in (x.dtype, torch.float32)
            and not (torch.is_grad_enabled() and x.requires_grad) and native.plain(x) and _colsum_faster(x)):
        native.require_hip()
        return torch.ops.sxe.column_sum(x, dtype)
    return x.sum(0) if dtype == x.dtype else x.float().sum(0).to(dtype)


class _Linear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias):
        ctx.param = None
        ac = _autocast_dtype(x)
        if ac is not None and weight.dtype != ac:
            # torch_autocast training (runtime/torch_autocast.py): fp32 master-precision parameters,
            # GEMMs in the autocast dtype. The fp32 Parameter keeps receiving its gradient through
            # the optimizer's direct weight-grad target; the bf16 copies are what backward reads.
            ctx.param = weight
            x, weight = x.to(ac), weight.to(ac)
            bias = bias.to(ac) if bias is not None else None
        ctx.save_for_backward(x, weight)
        ctx.has_bias = bias is not None
        ctx.bias = keep_local(bias)
        return product(x, weight, bias)

    @staticmethod
    def backward(ctx, gy):
        x, w = ctx.saved_tensors
        wp = ctx.param if ctx.param is not None else w
        if gy.dtype != x.dtype:
            gy = gy.to(x.dtype)
        gy2 = gy.reshape(-1, gy.shape[-1])
        dx = dw = db = None
        if ctx.needs_input_grad[0]:
            dx = data_grad(gy, w)
        if ctx.needs_input_grad[1]:
            x2 = x.reshape(-1, x.shape[-1])
            if not write_weight_grad(wp, gy2, x2):
                dw = gy2.t() @ x2
        if ctx.has_bias and ctx.needs_input_grad[2] and not write_bias_grad(ctx.bias, gy2, ctx):
            db = column_sum(gy2, gy2.dtype)
        return dx, dw, db


def linear(x, weight, bias=None, host_bound=False):
    """``host_bound``: the calls around this one wait for the host, so short ones may take longer on the device (``_eager_own``)."""
    if not isinstance(weight, torch.Tensor):  # quantized inference weight (ops/fp_quantizer.FP8Weight)
        return weight.linear(x, bias)
    grad = torch.is_grad_enabled() and (weight.requires_grad or x.requires_grad or (bias is not None and bias.requires_grad))
    if grad and weight.requires_grad and hasattr(weight, "_sxe_grad_target"):
        return _Linear.apply(x, weight, bias)
    if not grad and SKINNY_MAX_M > 0 and x.is_cuda:
        n, K = x.numel(), x.shape[-1]
        few = n <= max(SKINNY_MAX_M, STREAM_ROWS_SMALL) * K
        # the sizes first: a call that stays with the library is host-bound at a few hundred rows, and what follows is 2 us
        if ((few or (weight.dim() == 2 and (_tiled_faster(n // K, *weight.shape) or (host_bound and _eager_own(n // K, *weight.shape)))))
                and (not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") == torch.bfloat16)
                and native.plain(x, weight, bias)):
            if few:
                y = _skinny(x, weight, bias)
                if y is None:
                    y = _stream(x, weight, bias)
            else:
                y = _tiled(x, weight, bias, True)
            if y is not None:
                return y
    return F.linear(x, weight, bias)


def is_own_forward(mod, *types):
    """``mod(x)`` runs the forward of one of ``types`` and nothing else, so a caller may read its weight and run another kernel: not a
    subclass (low-rank, fake-quantized or partitioned layers), no patched forward, no hooks."""
    every = torch.nn.modules.module
    return (type(mod) in types and "forward" not in mod.__dict__ and not mod._forward_hooks and not mod._forward_pre_hooks
            and not every._global_forward_hooks and not every._global_forward_pre_hooks)


def is_own_call(mod, *types):
    """A caller may choose the arguments of ``mod(...)``: it runs the forward of one of ``types``, and nobody looks at what goes in, comes
    out or flows back (the optimizer's hooks that wait for parameters do not)."""
    every = torch.nn.modules.module
    return (type(mod) in types and "forward" not in mod.__dict__ and not mod._forward_hooks and not mod._backward_hooks
            and not mod._backward_pre_hooks and all(getattr(h, "_sxe_wait", False) for h in mod._forward_pre_hooks.values())
            and not every._global_forward_hooks and not every._global_forward_pre_hooks and not every._global_backward_hooks
            and not every._global_backward_pre_hooks)


class Linear(torch.nn.Linear):
    """``nn.Linear`` whose GEMMs go through ``linear`` (fused weight-grad into ZeRO buffers).
    AutoTP swaps it for a column/row-parallel layer with the same call signature.

    ``init_std``: initialise the weight N(0, init_std) (bias zero) inside the constructor, i.e.
    on the whole tensor before a partitioning ``zero.Init`` cuts it -- the initial model then
    depends only on the seed, not on the number of ranks."""

    _sxe_lower_precision_safe = True  # torch_autocast: GEMM weights may communicate in bf16 / fp16

    def __init__(self, in_features, out_features, bias=True, device=None, dtype=None, init_std=None):
        super().__init__(in_features, out_features, bias=bias, device=device, dtype=dtype)
        if init_std is not None:
            with torch.no_grad():
                self.weight.normal_(0.0, init_std)
                if self.bias is not None:
                    self.bias.zero_()
            self._sxe_inited = True

    def forward(self, x, skip_bias=False):
        return linear(x, self.weight, None if skip_bias else self.bias)


class _Embed(torch.autograd.Function):
    @staticmethod
    def forward(ctx, ids, weight):
        ctx.save_for_backward(ids)
        ctx.rows = weight.shape[0]
        ctx.weight = keep_local(weight)
        return F.embedding(ids, weight)

    @staticmethod
    def backward(ctx, gy):
        ids, = ctx.saved_tensors
        if (torch.is_grad_enabled() and gy.requires_grad) or not native.plain(gy, ids):  # a derivative of the gradient is asked for
            return None, torch.ops.aten.embedding_dense_backward(gy, ids, ctx.rows, -1, False)
        g2 = gy.reshape(-1, gy.shape[-1])
        if not g2.is_contiguous() or g2.data_ptr() % 16:
            g2 = g2.clone(memory_format=torch.contiguous_format)
        ids = ids.reshape(-1).contiguous()
        tgt = None if torch.is_grad_enabled() else local_grad_target(ctx.weight, ctx)
        if tgt is not None and tgt[0].data_ptr() % 16 == 0 and tgt[0].shape == (ctx.rows, g2.shape[1]):
            if not tgt[1]:
                tgt[0].zero_()
            torch.ops.sxe.embedding_grad_(g2, ids, tgt[0])  # only the rows that tokens took
            ctx.weight._sxe_grad_done(ctx.weight)
            return None, None
        return None, torch.ops.sxe.embedding_grad(g2, ids, ctx.rows)


EMBED_GRAD_IDS = 16384  # indices up to which ranking them by comparison is the faster way to their gradient (rows.hip)


class Embedding(torch.nn.Embedding):
    """``nn.Embedding`` with the constructor-time N(0, init_std) init of ``Linear`` and, on the GPU, a gradient of its own."""

    def __init__(self, num_embeddings, embedding_dim, init_std=None, **kw):
        super().__init__(num_embeddings, embedding_dim, **kw)
        if init_std is not None:
            with torch.no_grad():
                self.weight.normal_(0.0, init_std)
            self._sxe_inited = True

    def forward(self, input):
        w = self.weight
        if (w.is_cuda and torch.is_grad_enabled() and w.requires_grad and self.padding_idx is None and self.max_norm is None
                and not self.scale_grad_by_freq and not self.sparse and isinstance(input, torch.Tensor) and 0 < input.numel() <= EMBED_GRAD_IDS
                and w.dim() == 2 and w.shape[1] % 8 == 0 and w.dtype in (torch.bfloat16, torch.float16, torch.float32)
                and input.device == w.device and input.dtype in (torch.int64, torch.int32) and native.use_hip(w) and native.plain(w, input)):
            return _Embed.apply(input, w)
        return super().forward(input)

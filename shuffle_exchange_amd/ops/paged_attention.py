"""Paged-KV attention ops for the ragged inference engine (HIP kernels in csrc/kernels/paged_attn.hip).

Cache layout per layer: ``[num_blocks, 2, n_kv_heads, block_size, head_dim]`` (bf16 on GPU).
``kv_cache_append`` scatters the k/v rows of the new tokens into their slots
(``slot = block_id * block_size + offset``); ``paged_attention`` runs causal attention of the new
tokens of each sequence over all of its cached keys. Both have PyTorch reference implementations
(CPU processes / numerics oracles).
"""
import functools
import math
import os

import torch

from . import native


def rope_kv_cache_append(qkv, rope, positions, cache, slots, nq, nkv):
    """RoPE on the q and k heads of ``qkv`` [T, nq + 2 nkv, D] (in place, absolute ``positions``)
    and the rotated k + v appended to the paged ``cache`` -- one HIP launch
    (paged_attn.hip ``rope_kv_append_kernel``) instead of rope_ + kv_cache_append."""
    from .rope import apply_rope_tokens_
    if (native.use_hip(qkv) and qkv.dtype == torch.bfloat16 and qkv.shape[-1] in (64, 128, 256)
            and qkv.is_contiguous() and rope.cos.shape[-1] * 2 == qkv.shape[-1]):
        torch.ops.sxe.rope_kv_cache_append(qkv, rope.cos, rope.sin, positions.reshape(-1).contiguous().long(), cache,
                                           slots, int(nq), int(nkv))
        return qkv
    apply_rope_tokens_(qkv, rope, nq + nkv, positions)
    kv_cache_append(qkv, cache, slots, nq, nkv)
    return qkv


def kv_cache_append(qkv, cache, slots, nq, nkv):
    """qkv: [T, nq + 2 nkv, D]; cache: [blocks, 2, nkv, bs, D]; slots: int64 [T] (-1 = skip)."""
    if native.use_hip(qkv) and qkv.shape[-1] in (64, 128) and qkv.is_contiguous():
        torch.ops.sxe.kv_cache_append(qkv, cache, slots, int(nq), int(nkv))
        return
    bs = cache.shape[3]
    ok = slots >= 0
    if not bool(ok.any()):
        return
    s = slots[ok]
    blk, off = s // bs, s % bs
    k = qkv[ok, nq:nq + nkv]
    v = qkv[ok, nq + nkv:nq + 2 * nkv]
    cache[blk, 0, :, off] = k.to(cache.dtype)
    cache[blk, 1, :, off] = v.to(cache.dtype)


def _gather_kv(cache, block_row, kv_len):
    bs = cache.shape[3]
    nb = (kv_len + bs - 1) // bs
    blocks = block_row[:nb].long()
    kv = cache[blocks]  # [nb, 2, nkv, bs, D]
    k = kv[:, 0].permute(1, 0, 2, 3).reshape(kv.shape[2], nb * bs, -1)[:, :kv_len]
    v = kv[:, 1].permute(1, 0, 2, 3).reshape(kv.shape[2], nb * bs, -1)[:, :kv_len]
    return k, v  # [nkv, kv_len, D]


def paged_attention_reference(q, cache, block_table, q_start, q_len, kv_len, scale, window=None):
    T, nq, D = q.shape
    nkv = cache.shape[2]
    G = nq // nkv
    out = torch.zeros(T, nq, D, dtype=q.dtype, device=q.device)
    for s in range(block_table.shape[0]):
        qs, ql, kl = int(q_start[s]), int(q_len[s]), int(kv_len[s])
        if ql == 0:
            continue
        k, v = _gather_kv(cache, block_table[s], kl)
        k = k.float().repeat_interleave(G, dim=0)
        v = v.float().repeat_interleave(G, dim=0)
        qq = q[qs:qs + ql].float().transpose(0, 1)  # [nq, ql, D]
        sc = torch.matmul(qq, k.transpose(1, 2)) * scale  # [nq, ql, kl]
        pos = torch.arange(kl - ql, kl, device=q.device)[:, None]
        keys = torch.arange(kl, device=q.device)[None, :]
        mask = keys > pos
        if window:  # sliding-window attention (Mistral / Qwen2): only the last `window` keys
            mask = mask | (keys <= pos - window)
        sc = sc.masked_fill(mask, float("-inf"))
        o = torch.matmul(torch.softmax(sc, dim=-1), v)  # [nq, ql, D]
        out[qs:qs + ql] = o.transpose(0, 1).to(q.dtype)
    return out


# keys per split floor (see choose_splits and _short_splits): 256 = four 64-key wave chunks per split. Llama-3-8B decode,
# HIP graphs, fused merge: batch 1 ctx 1024 3.571 / 3.604 / 3.700 ms per token at 256 / 128 / 64,
# ctx 4096 3.745 / 3.927 / 3.926; batch 8 and 32 within 1 % (profiles/r06/decode_split_floor_ab.log)
PA_MIN_KEYS = int(os.environ.get("SXE_PA_MIN_KEYS", 256))


PA_TARGET_WGS = int(os.environ.get("SXE_PA_TARGET_WGS", 512))


def choose_splits(num_seqs, nkv, max_kv_len, target_wgs=None):
    """KV splits so (seqs x kv heads x splits) fills the 256 CUs, never below PA_MIN_KEYS keys per
    split: at batch 1 the kernel is a latency chain (block table -> K/V loads -> MFMA -> merge), so
    more, shorter splits shorten it; at large batch one split per (seq, kv head) streams best."""
    target_wgs = PA_TARGET_WGS if target_wgs is None else target_wgs
    base = max(1, num_seqs * nkv)
    want = max(1, math.ceil(target_wgs / base))
    return max(1, min(want, math.ceil(max(max_kv_len, 1) / PA_MIN_KEYS)))


# Keys of a split at most where sequences differ in length. One layer's attention of a decode step, heads 32 / 8 of 128, us with the
# splits of choose_splits / of at most 512 keys: sequences of 300 - 4000 keys, 16 of them 35 / 26, 32 61 / 44, 64 111 / 85, 128
# 167 / 152; but all of 4000 keys 44 / 51, 95 / 102, 177 / 195; all of 2000 - 4000 38 / 40, 77 / 79, 145 / 149; 64 of 1000 42 / 50.
# Half of them where the splits of 512 keys all run at once (so the launch has up to twice as many workgroups as do, of which those behind
# a sequence's end exit at once): a workgroup's few chunks one after the other are what the call takes. With the merge, 512 / 256 keys:
# 8 sequences of 256 - 3000 keys 23.0 / 20.7, 16 of 200 - 2500 (640, then 1280 workgroups) 26.3 / 22.7; 24 of 256 - 6000 (2304, not
# halved) a step of four layers 841 / 850, 40 of 100 - 3000 (1920) of two 432 / 438; heads of 64 13.9 / 13.1, 17.8 / 16.3, of 256, one
# workgroup a CU, 29.2 / 33.7.
PA_SPLIT_KEYS = 512
# Lengths are even where the longest is at most this many times the mean (a log-uniform spread over a factor of 2 has 1.4, of 10 2.6).
PA_EVEN = 1.5
# Workgroups that run at once, three a CU (other head dims: by registers). Even sequences finish together, so a last round that is nearly
# empty costs a whole one: 100 sequences (800 workgroups a split) of 2500 keys 221 / 194 us with 1 / 3 splits, but 160 (1280) of 1500
# 174 / 182; heads of 64, 128 sequences of 12 heads and 4000 keys 278 / 262 with 1 / 2.
PA_RESIDENT_WGS = 768
PA_RESIDENT = {64: 1024, 128: PA_RESIDENT_WGS, 256: 256}
# Bytes of fp32 partials that such short splits may take: 256 decoding sequences keep splits of 512 keys up to 32k keys (heads of
# 32 x 128), a call of many tokens has the splits of choose_splits, as its partials grow with tokens x splits.
PA_SPLIT_BYTES = 1 << 28


def even_lengths(lengths):
    """Whether sequences of these lengths keep a batch's workgroups busy alike."""
    return len(lengths) * max(lengths, default=0) <= PA_EVEN * sum(lengths)


def two_a_cu(workgroups, head_dim):
    """Whether one split runs better on the kernel's form of 64 keys a wave and two workgroups a CU: these make whole rounds of 512, of
    768 the last one would be nearly empty. Heads of 128, us, so / one split of the other form / the best number of its splits: 128
    sequences of 8 kv heads 1500 keys 136 / 156 / 147, 4000 keys 350 / 392 / 360; 32 of 32 kv heads 1000 keys 94 / 106 / 103; a remainder
    of 512 (64 of 32 kv heads, 2048 workgroups, 1000 to 3000 keys) 183 - 507 / 190 - 523, 256 of 8 379 / 367 at 2000."""
    return head_dim == 128 and workgroups > 768 and 0 < workgroups % 768 <= 256 and (-workgroups) % 512 < 64


def choose_balanced_splits(num_seqs, nkv, max_kv_len, split_bytes, even=False, head_dim=128):
    """``choose_splits``, and no split over PA_SPLIT_KEYS keys: where sequences of a batch differ in length, a workgroup that
    walks a long one alone outlasts the rest. Splits behind a sequence's end exit at once, the merge does not read them.
    ``even`` (``even_lengths``): as few splits as fill the chip, in rounds that are mostly full.
    ``split_bytes``: partials of one split (rows x heads x head dim, fp32)."""
    splits, most = choose_splits(num_seqs, nkv, max_kv_len), PA_SPLIT_BYTES // max(1, split_bytes)
    resident = PA_RESIDENT.get(head_dim, PA_RESIDENT_WGS)
    if not even:
        n = math.ceil(max_kv_len / PA_SPLIT_KEYS)
        if head_dim <= 128 and num_seqs * nkv * n <= resident:
            n = math.ceil(2 * max_kv_len / PA_SPLIT_KEYS)
        return max(splits, min(n, most))

    def full(s):  # share of the resident workgroups that the rounds keep busy
        rounds = num_seqs * nkv * s / resident
        return 1 if rounds <= 1 else rounds / math.ceil(rounds)
    if full(splits) > 0.8 or (splits == 1 and two_a_cu(num_seqs * nkv, head_dim)):
        return splits
    more = [s for s in range(splits, splits + 3) if s == splits or (s <= most and max_kv_len >= s * 320)]
    return max(more, key=full)


# Keys up to which few decoding sequences with heads of 128 have splits of half of PA_MIN_KEYS, as long as these are at most one workgroup a CU:
# its four waves take 128 keys at a time. The same splits of 256 keys have the kernel's form of eight waves. A step of three layers, us, 256
# keys in two rounds of four waves / in one of eight / splits of 128: hidden 2048, 1 sequence of 500 keys 175.0 / 172.1 / 168.0, 4 of 1000
# 187.6 / 182.8 / 180.0; 3072, 2 of 1500 246.0 / 242.1 / 239.8; 4096, 1 of 1000 357.2 / 353.3 / 348.8; but with two workgroups a CU, hidden
# 2048, 8 of 1500 191.9 / 189.3 / 191.7. 3000 keys, one sequence of hidden 2048 180.1 / 176.7 / 181.7, 4096 364.5 / 360.2 / 370.8.
# Up to 256 keys one split stays one, with nothing to merge. One sequence, 1 / 2 splits of 128 keys, merged in the next product's launch: hidden
# 2048, 64 keys 151 / 155, 250 keys 156 / 156, e4m3 113 / 118, 117 / 119; 4096 311 / 311, 316 / 316; o product of skinny_gemm.hip, 64 keys 171 / 174, e4m3
# 125 / 131, hidden 4096 348 / 354, 236 / 240 (from 400 to 2000 keys there, splits of 256 / 128 keys, 360 / 356, 246 / 242).
PA_SHORT_KEYS = 2048
PA_SHORT_WGS = 256


def _short_splits(splits, num_seqs, nkv, max_kv_len, split_bytes, head_dim):
    if head_dim != 128 or not PA_MIN_KEYS < max_kv_len <= PA_SHORT_KEYS:
        return splits
    want = min(PA_SHORT_WGS // max(1, num_seqs * nkv), math.ceil(max_kv_len / max(1, PA_MIN_KEYS // 2)))
    return max(splits, min(want, PA_SPLIT_BYTES // max(1, split_bytes)))


@functools.lru_cache(maxsize=4096)
def _decode_plan(num_seqs, nkv, max_kv_len, split_bytes, even, head_dim, tuned):
    """(splits, two workgroups a CU) of a launch: all layers of a step ask for the same, a microsecond of the host each. ``tuned``: the
    settings that the choice reads."""
    splits = _short_splits(choose_balanced_splits(num_seqs, nkv, max_kv_len, split_bytes, even, head_dim), num_seqs, nkv, max_kv_len,
                           split_bytes, head_dim)
    return splits, splits == 1 and two_a_cu(num_seqs * nkv, head_dim)


def decode_plan(num_seqs, nkv, max_kv_len, split_bytes, even, head_dim):
    """``_decode_plan`` by the settings as they are."""
    return _decode_plan(num_seqs, nkv, max_kv_len, split_bytes, even, head_dim, (PA_TARGET_WGS, PA_MIN_KEYS))


def paged_attention_parts(q, cache, block_table, q_start, q_len, kv_len, scale, max_kv_len, splits=None):
    """``paged_attention`` without the split-merge launch (HIP only): returns ``(out, None)`` when the
    kernel ran one split per (sequence, kv head), else ``(None, (part_o, part_ml))`` -- fp32
    partials [splits, T, nq, D] / [splits, T, nq, 2] for a consumer that merges them in its own
    prologue (``ops.linear.fused_merge_linear``: the o_proj skinny GEMM; ``stream_res_splits``)."""
    if splits is None:
        S, nkv = block_table.shape[0], cache.shape[2]
        splits = _short_splits(choose_splits(S, nkv, max_kv_len), S, nkv, int(max_kv_len), 4 * q.numel(), q.shape[-1])
    out, po, pml = torch.ops.sxe.paged_attention_parts(q, cache, block_table, q_start, q_len, kv_len, float(scale),
                                                       int(max_kv_len), int(splits), 0)
    return (out, None) if po.numel() == 0 else (None, (po, pml))


def merge_attention_parts(part_o, part_ml, dtype):
    """Flash-decoding merge of ``paged_attention_parts``' KV-split partials (the math of
    paged_attn.hip's merge kernel / skinny_gemm.hip PRO_MERGE): sum_s 2^(M_s - M) o_s /
    sum_s 2^(M_s - M) L_s over the splits, M the max of the split maxima (log2 domain).
    part_o [splits, T, nq, D], part_ml [splits, T, nq, 2] fp32 -> [T, nq, D] in ``dtype``."""
    m, l = part_ml[..., 0], part_ml[..., 1]
    mx = m.amax(0)
    f = torch.where(torch.isinf(m), torch.zeros_like(m), torch.exp2(m - torch.where(torch.isinf(mx), 0, mx)))
    den = (f * l).sum(0)
    num = (f.unsqueeze(-1) * part_o).sum(0)
    return torch.where(den.unsqueeze(-1) > 0, num / den.clamp_min(1e-30).unsqueeze(-1), 0.).to(dtype)


# SXE_PA_LAST_MERGE=1: with several KV splits the last split workgroup of each (sequence, kv head)
# merges the partials inside the attention launch (paged_attn.hip, arrival counters) instead of a
# second merge launch. Off: its device-scope fences write back / invalidate the L2 the K/V stream
# lives in -- Llama-3-8B ctx 1024 decode 4.50 vs 3.73 ms/token at batch 1, 6.60 vs 4.91 at batch 8
# (profiles/r06/decode_split_merge_ab.log)
PA_LAST_MERGE = os.environ.get("SXE_PA_LAST_MERGE", "0") == "1"
_COUNTERS = {}


def _split_counters(device, n):
    """Zeroed int32 split-arrival counters (self-resetting in the kernel), one buffer per device,
    grown outside any graph capture in the normal flow (the decode engine runs eagerly first)."""
    c = _COUNTERS.get(device)
    if c is None or c.numel() < n:
        c = _COUNTERS[device] = torch.zeros(max(n, 4096), dtype=torch.int32, device=device)
    return c


def paged_attention(q, cache, block_table, q_start, q_len, kv_len, scale, max_kv_len, splits=None, window=None, even=False):
    """q: [T, nq, D] (head stride D); metadata int32 [S]; returns [T, nq, D]. ``window``: sliding
    window length (keys older than ``window`` positions are masked, Mistral / Qwen2). The HIP kernel
    covers head dims 64 / 128 / 256, with or without a window (the window also skips the key chunks
    it masks entirely). ``even``: the sequences are about as long as one another (``even_lengths``)."""
    if window is not None and max_kv_len <= window:
        window = None
    if native.use_hip(q) and q.shape[-1] in (64, 128, 256):
        S, nkv = block_table.shape[0], cache.shape[2]
        if splits is None:
            splits, wide = decode_plan(S, nkv, int(max_kv_len), 4 * q.numel(), even, q.shape[-1])
        else:
            wide = splits == 1 and two_a_cu(S * nkv, q.shape[-1])
        cnt = (_split_counters(q.device, S * nkv)
               if PA_LAST_MERGE and splits > 1 and q.shape[0] <= 4 * S else None)
        return torch.ops.sxe.paged_attention(q, cache, block_table, q_start, q_len, kv_len, float(scale),
                                             int(max_kv_len), int(splits), int(window or 0), cnt, wide)
    if q.is_cuda:
        from ..utils.logging import warning_once
        warning_once(f"paged_attention: head_dim={q.shape[-1]} window={window} not covered by the HIP kernel; "
                     f"using the PyTorch reference")
    return paged_attention_reference(q, cache, block_table, q_start, q_len, kv_len, scale, window)


# A sequence takes the tile kernel from this many rows (new tokens x query heads of a kv head): up to 16 rows the decode
# kernel reads the keys once, beyond it once for every 16 rows. Heads 32 / 8 of 128, us in the decode / the tile kernel:
# 16 rows: 8 sequences behind 3000 keys 29 / 26, one behind 3000 15 / 19, 32 fresh 9.7 / 12; 20 rows: 44 / 25, 20 / 20,
# 13.5 / 12.6; 128 rows: 159 / 40, 73 / 24, 60 / 12.5.
TILE_MIN_ROWS = 17
TILE_ROWS = 128  # rows of a workgroup of the tile kernel


def choose_tile_splits(num_tiles, nkv, max_keys, target_wgs=None):
    """(splits, keys of a split) of the tile kernel: the fewest splits that give every CU two workgroups, none under
    512 keys (a split's partials cost as much traffic as ~64 keys of its tile)."""
    target_wgs = PA_TARGET_WGS if target_wgs is None else target_wgs
    want = math.ceil(target_wgs / max(1, num_tiles * nkv))
    splits = max(1, min(want, math.ceil(max_keys / 512)))
    keys = -(-math.ceil(max(max_keys, 1) / splits) // 64) * 64
    return -(-max(max_keys, 1) // keys), keys


# Heads that run all sequences of a batch in the tile kernel's launch, in pieces by ``paged_prefill_plan`` (csrc/kernels/paged_prefill.hip has the
# figures). Heads of 64 and 256 have another balance: so, and by ``choose_tile_splits`` with the decodes in a launch of their own, 1024
# tokens behind 2048 63 / 54 us, 128 decodes of 2000 keys beside 32 tokens 361 / 218.
TILE_DIM = 128


def _tileable(q, cache, scale):
    return (native.use_hip(q) and q.dtype == torch.bfloat16 and cache.dtype == torch.bfloat16 and q.shape[-1] in (64, 128, 256)
            and q.shape[1] % cache.shape[2] == 0 and q.shape[1] // cache.shape[2] <= TILE_ROWS and scale > 0
            and q.stride(2) == 1 and q.stride(1) == q.shape[2] and q.stride(0) % 8 == 0 and q.data_ptr() % 16 == 0)


def paged_batch_attention(q, cache, batch, scale, window=None):
    """``paged_attention`` of a whole ragged batch."""
    return paged_attention(q, cache, batch.block_table, batch.q_start, batch.q_len, batch.kv_len, scale, batch.max_kv_len,
                           window=window, even=batch.even_lengths)


# The longest prompts take the training forward (csrc/kernels/flash_attn.hip) on the new tokens' own keys up to their last multiple of
# 128 tokens, the tile kernel the tail. It is faster a tile, but starts with few of them and one prompt a launch; a tail costs a
# launch with its merge. us, training forward (and tail) / tile kernel, heads of 128: 32 / 8 heads: 3072 tokens 114 / 106, 4096
# 163 / 174, 5120 256 / 249, 6144 345 / 348, 6200 397 / 366, 8192 544 / 618, 8193 589 / 623, 16500 2200 / 2421, 32767 8850 / 9420;
# 24 / 8: 5120 181 / 199, 9000 554 / 580; 16 / 4: 6144 189 / 191, 8192 280 / 330, 9000 388 / 388, 12300 681 / 694; 8 / 2: 12300
# 388 / 378, 16384 538 / 640; 4 / 1: 12416 270 / 240, 65500 4440 / 4830.
# (new tokens, new tokens x query heads) from which, without a tail and with one
FLASH_WHOLE, FLASH_TAIL = (4096, 1 << 17), (8192, 3 << 16)


def _flash_prompts(q, kv, batch, window):
    """Pairs (sequence, first tokens) that the training forward takes."""
    if kv is None or window is not None or q.shape[-1] != 128 or not (kv.is_cuda and kv.dtype == q.dtype and kv.stride()[1:] == (128, 1)):
        return ()
    took = []
    for i, (n, seen) in enumerate(zip(batch.host_q_len, batch.host_seen)):
        tokens, work = FLASH_TAIL if n % 128 else FLASH_WHOLE
        if seen == 0 and n >= tokens and n * q.shape[1] >= work:
            took.append((i, n // 128 * 128))
    return tuple(took)


def _tile_plan(lists, nq, nkv, dim, window):
    """All layers of a pass ask for the same."""
    if window is not None or dim != TILE_DIM:
        return choose_tile_splits(lists.tiles.shape[0], nkv, lists.tile_keys)
    plan = lists.plans.get((nq, nkv, dim))
    if plan is None:
        most = lists.tile_keys
        plan = lists.plans[nq, nkv, dim] = ((1, -(-most // 64) * 64) if most <= 640 else  # no two pieces of 384 keys and more
                                            torch.ops.sxe.paged_prefill_plan(*lists.tile_sizes, nq, nkv, dim, PA_SPLIT_BYTES))
    return plan


def ragged_attention(q, cache, batch, scale, window=None, kv=None):
    """Causal attention of a ragged batch's new tokens q [T, nq, D] over their paged keys (the new ones among them).
    Sequences with many new tokens -- prompts, and chunks of prompts behind earlier tokens -- run the tile kernel, and the others with them
    (heads of 128; 16 sequences of 200 - 2500 keys beside 428 tokens behind 3072, us, in a launch of the decode kernel / so 78 / 56); other
    heads, under a window, and where no sequence has as many, they run the decode kernel. ``kv`` [T, 2 nkv, D]: the new tokens' keys and values as they are in the cache, for the longest
    prompts."""
    nkv = cache.shape[2]
    if window is not None and batch.max_kv_len <= window:
        window = None
    if not (hasattr(batch, "attention_lists") and _tileable(q, cache, scale)):
        return paged_batch_attention(q, cache, batch, scale, window)
    tile, least = TILE_ROWS // (q.shape[1] // nkv), -(-TILE_MIN_ROWS // (q.shape[1] // nkv))
    flash = _flash_prompts(q, kv, batch, window)
    if window is None and q.shape[2] == TILE_DIM:
        done = {i for i, _ in flash}
        if (max(batch.host_q_len, default=0) >= least if not done else any(n >= least and i not in done for i, n in enumerate(batch.host_q_len))):
            least = 1
    lists = batch.attention_lists(tile, least, flash)
    if lists is None and not flash:
        return paged_batch_attention(q, cache, batch, scale, window)
    out = None
    for i, n in flash:
        at = slice(batch.host_q_start[i], batch.host_q_start[i] + n)
        o = torch.ops.sxe.flash_attn_fwd(q[None, at], kv[None, at, :nkv], kv[None, at, nkv:], True, float(scale))[0][0]
        if n == q.shape[0]:
            return o
        out = torch.empty(q.shape, dtype=q.dtype, device=q.device) if out is None else out
        out[at] = o
    out = torch.empty(q.shape, dtype=q.dtype, device=q.device) if out is None else out
    meta = (q, cache, batch.block_table, batch.q_start, batch.q_len, batch.kv_len)
    for x in (batch.attention_lists(tile, least, flash, True) if flash else None, lists):
        if x is not None and x.tiles is not None:
            splits, keys = _tile_plan(x, q.shape[1], nkv, q.shape[2], window)
            rows = batch.tile_rows(x) if splits > 1 else None
            torch.ops.sxe.paged_prefill(*meta, x.tiles, rows, float(scale), int(window or 0), splits, keys, out)
    if lists is not None and lists.seqs is not None:
        n, D = lists.seqs.shape[0], q.shape[2]
        splits, wide = decode_plan(n, nkv, lists.seq_keys, 4 * lists.seq_rows.numel() * q.shape[1] * D, lists.seq_even, D)
        torch.ops.sxe.paged_attention_some(*meta, lists.seqs, lists.seq_rows, float(scale), int(lists.seq_keys), int(splits),
                                           int(window or 0), out, wide)
    return out

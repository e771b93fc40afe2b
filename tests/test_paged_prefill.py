"""Attention of ragged batches over the paged cache: the tile kernel (csrc/kernels/paged_prefill.hip) and the lists that
route sequences to it, against the fp32 reference."""
from types import SimpleNamespace

import pytest
import torch

from shuffle_exchange_amd.inference.v2.ragged.ragged import DSSequenceDescriptor, RaggedBatch
from shuffle_exchange_amd.ops import paged_attention as PA


def _batch(seqs, bs, device, seed=0):
    """A ragged batch of (earlier, new) token counts over shuffled cache blocks."""
    g = torch.Generator().manual_seed(seed)
    need = [(c + n + bs - 1) // bs for c, n in seqs]
    ids = torch.randperm(sum(need) + 2, generator=g).tolist()
    desc = []
    for i, ((c, n), k) in enumerate(zip(seqs, need)):
        d = DSSequenceDescriptor(i, 1 << 20)
        d.blocks, ids = ids[:k], ids[k:]
        d.seen_tokens = c
        desc.append(d)
    return RaggedBatch(desc, [torch.zeros(n, dtype=torch.int64) for _, n in seqs], bs, torch.device(device)), sum(need) + 2


def test_lists_hold_every_token_once():
    seqs = [(0, 70), (500, 1), (33, 200), (0, 8), (9, 9)]
    b, _ = _batch(seqs, 16, "cpu")
    x = b.attention_lists(32, 9)
    tiles = x.tiles.tolist()
    keys = [seqs[s][0] + (q - b.host_q_start[s]) + n for s, q, n, _ in tiles]
    assert keys == sorted(keys, reverse=True) and x.tile_keys == keys[0] and max(t[2] for t in tiles) <= 32
    got = sorted(t for _, q, n, _ in tiles for t in range(q, q + n))
    rows = b.tile_rows(x)
    assert got == sorted(rows.tolist()) and b.tile_rows(x) is rows and sorted(got + x.seq_rows.tolist()) == list(range(b.num_tokens))
    for _, q, n, at in tiles:
        assert rows[at:at + n].tolist() == list(range(q, q + n))
    for s, at in x.seqs.tolist():
        assert x.seq_rows[at:at + seqs[s][1]].tolist() == list(range(b.host_q_start[s], b.host_q_start[s] + seqs[s][1]))
    assert x.seq_keys == 501 and b.attention_lists(32, 201) is None


def test_tile_splits_cover_the_keys():
    for tiles in (1, 3, 40, 1000):
        for nkv in (1, 8):
            for keys in (1, 64, 500, 513, 4097, 100000):
                n, k = PA.choose_tile_splits(tiles, nkv, keys)
                assert k % 64 == 0 and n * k >= keys > (n - 1) * k


@pytest.mark.parametrize("sizes", [[(1, 1)], [(64, 32)], [(65, 1)], [(257, 32), (33, 32)], [(100000, 32)] * 3 + [(1, 1)] * 9, [(4096, 32)] * 1000,
                                   [(131072, 16)] * 2000])
@pytest.mark.parametrize("nq,nkv", [(32, 8), (7, 7)])
def test_tile_plan_covers_the_keys_and_bounds_its_partials(sizes, nq, nkv):
    from shuffle_exchange_amd.ops import native
    if not native.status()["hip"]:
        pytest.skip("the HIP library is not built")
    keys, tokens = zip(*sizes)
    n, k = torch.ops.sxe.paged_prefill_plan(keys, tokens, nq, nkv, 128, PA.PA_SPLIT_BYTES)
    assert k % 64 == 0 and n * k >= max(keys) > (n - 1) * k
    assert n == 1 or (k >= 384 and n * sum(tokens) * nq * 128 * 4 <= PA.PA_SPLIT_BYTES)


@pytest.mark.gpu
@pytest.mark.parametrize("seqs", [[(4000, 300), (700, 1), (31, 2), (5, 40)], [(0, 64), (63, 1), (64, 1), (300, 8)], [(0, 1), (0, 700)]])
@pytest.mark.parametrize("keys", [64, 320, 1024, 4352])
@pytest.mark.parametrize("nq,nkv,D,window", [(32, 8, 128, None), (12, 12, 128, None), (8, 4, 128, 100), (4, 4, 64, None), (8, 4, 256, 300)])
def test_pieces_of_tiles(seqs, keys, nq, nkv, D, window):
    """Tiles that lie in one piece, in several, in front of or behind the others' (windows): decodes and prompts in one launch."""
    from shuffle_exchange_amd.ops import native
    native.require_hip()
    b, blocks = _batch(seqs, 64, "cuda", seed=3)
    g = torch.Generator(device="cuda").manual_seed(4)
    cache = torch.randn(blocks, 2, nkv, 64, D, device="cuda", generator=g).to(torch.bfloat16)
    q = torch.randn(b.num_tokens, nq, D, device="cuda", generator=g).to(torch.bfloat16)
    x = b.attention_lists(128 // (nq // nkv), 1)
    splits = -(-x.tile_keys // keys)
    out = torch.full_like(q, float("nan"))
    torch.ops.sxe.paged_prefill(q, cache, b.block_table, b.q_start, b.q_len, b.kv_len, x.tiles, b.tile_rows(x) if splits > 1 else None,
                                D ** -0.5, window or 0, splits, keys, out)
    ref = PA.paged_attention_reference(q.float(), cache.float(), b.block_table, b.q_start, b.q_len, b.kv_len, D ** -0.5, window)
    for i in range(b.num_seqs):  # p and the output are rounded to 8 bits each, as in test_ragged_attention
        s, n = b.host_q_start[i], b.host_q_len[i]
        assert ((out[s:s + n].float() - ref[s:s + n]).norm() / ref[s:s + n].norm()).item() < 8e-3, seqs[i]


@pytest.mark.parametrize("rows,seqs,keys", [(8192, 1, 131072), (16984, 16, 16384), (32768, 64, 16384), (131072, 32, 4096), (256, 256, 131072),
                                            (64, 64, 8192), (1, 1, 131072), (0, 1, 1)])
@pytest.mark.parametrize("nq,nkv,D", [(32, 8, 128), (64, 8, 128), (16, 1, 256), (7, 7, 64)])
def test_decode_splits_bound_their_partials(rows, seqs, keys, nq, nkv, D):
    """The fp32 partials of a call do not grow with rows x keys: short splits only as far as they fit a fixed size."""
    row = nq * D * 4
    plain, n = PA.choose_splits(seqs, nkv, keys), PA.choose_balanced_splits(seqs, nkv, keys, rows * row)
    assert n >= plain and (n == plain or n * rows * row <= PA.PA_SPLIT_BYTES)
    if rows <= 64:  # decode-sized calls keep splits of at most 512 keys
        assert n >= -(-keys // 512)


@pytest.mark.gpu
@pytest.mark.parametrize("seqs", [[(0, 33)], [(0, 1), (63, 65), (64, 64), (0, 129)], [(4000, 300), (700, 1), (31, 2), (5, 40)],
                                  [(1, 127), (127, 1), (0, 700), (2500, 9)]])
@pytest.mark.parametrize("nq,nkv,D,bs,window", [(32, 8, 128, 64, None), (4, 4, 64, 16, None), (7, 1, 128, 128, 100),
                                                (6, 2, 64, 48, 1), (8, 4, 256, 32, 300), (16, 1, 128, 64, None)])
def test_ragged_attention(seqs, nq, nkv, D, bs, window):
    b, blocks = _batch(seqs, bs, "cuda", seed=1)
    g = torch.Generator(device="cuda").manual_seed(2)
    cache = torch.randn(blocks, 2, nkv, bs, D, device="cuda", generator=g).to(torch.bfloat16)
    # slots that no sequence has written hold anything
    used = torch.zeros(blocks * bs, dtype=torch.bool, device="cuda")
    for i, (c, n) in enumerate(seqs):
        p = torch.arange(c + n, device="cuda")
        used[b.block_table[i].long()[p // bs] * bs + p % bs] = True
    cache.view(blocks, 2, nkv, bs, D).permute(0, 3, 1, 2, 4)[~used.view(blocks, bs)] = float("nan")
    qkv = torch.randn(b.num_tokens, nq + 2 * nkv, D, device="cuda", generator=g).to(torch.bfloat16)
    q, scale = qkv[:, :nq], D ** -0.5
    ref = PA.paged_attention_reference(q.float(), cache.float(), b.block_table, b.q_start, b.q_len, b.kv_len, scale, window)
    got = PA.ragged_attention(q, cache, b, scale, window)
    # p and the output are rounded to 8 bits each, the rest is fp32: 2 x 2^-9 and slack for the rows' spread
    assert ((got.float() - ref).norm() / ref.norm()).item() < 6e-3
    for i in range(b.num_seqs):  # every sequence for itself: a short one cannot hide behind a long one
        s, n = b.host_q_start[i], b.host_q_len[i]
        assert ((got[s:s + n].float() - ref[s:s + n]).norm() / ref[s:s + n].norm()).item() < 8e-3, seqs[i]


@pytest.mark.gpu
@pytest.mark.parametrize("seqs", [[(0, 70)], [(300, 1)], [(0, 70), (300, 1)]])
def test_metadata_on_one_device(seqs):
    """Lists left in host memory are refused before any launch."""
    b, blocks = _batch(seqs, 64, "cuda")
    cache = torch.zeros(blocks, 2, 2, 64, 128, device="cuda", dtype=torch.bfloat16)
    q = torch.randn(b.num_tokens, 4, 128, device="cuda").to(torch.bfloat16)
    for name in ("block_table", "q_start", "q_len", "kv_len"):
        there = getattr(b, name)
        setattr(b, name, there.cpu())
        with pytest.raises(RuntimeError, match="operand is on cpu"):
            PA.ragged_attention(q, cache, b, 128 ** -0.5)
        setattr(b, name, there)
    with pytest.raises(RuntimeError, match="operand is on cpu"):
        PA.ragged_attention(q, cache.cpu(), b, 128 ** -0.5)
    PA.ragged_attention(q, cache, b, 128 ** -0.5)


def test_lists_without_long_prompts():
    """The sequences that another launch takes are in neither list, their last tokens in one of their own."""
    seqs = [(0, 300), (0, 70), (40, 1), (0, 256)]
    b, _ = _batch(seqs, 16, "cpu")
    done = ((0, 256), (3, 256))
    rest, tails = b.attention_lists(32, 9, done), b.attention_lists(32, 9, done, True)
    rows = lambda x: sorted(t for _, q, n, _ in x.tiles.tolist() for t in range(q, q + n))  # noqa: E731
    assert rows(rest) == list(range(300, 370)) and rest.seq_rows.tolist() == [370]
    assert rows(tails) == list(range(256, 300)) == b.tile_rows(tails).tolist() and tails.seqs is None and tails.tile_keys == 300
    for x in (rest, tails):
        for _, q, n, at in x.tiles.tolist():
            assert b.tile_rows(x)[at:at + n].tolist() == list(range(q, q + n))
    b, _ = _batch([(0, 256), (40, 1)], 16, "cpu")
    done = ((0, 256),)
    assert b.attention_lists(32, 9, done).tiles is None and b.attention_lists(32, 9, done).seq_rows.tolist() == [256]
    assert b.attention_lists(32, 9, done, True) is None
    b, _ = _batch([(0, 256)], 16, "cpu")
    assert b.attention_lists(32, 9, done) is None


@pytest.mark.gpu
@pytest.mark.parametrize("seqs", [[(0, 256)], [(0, 129)], [(0, 128), (40, 1)], [(0, 300), (0, 70), (200, 1), (0, 256), (130, 260)],
                                  [(0, 20), (0, 8319)]])
@pytest.mark.parametrize("nq,nkv", [(8, 2), (6, 2), (16, 16)])
def test_long_prompts(seqs, nq, nkv, monkeypatch):
    """The training forward for a prompt's first tokens beside the tile and decode kernels for the rest of the batch."""
    for name in ("FLASH_WHOLE", "FLASH_TAIL"):
        monkeypatch.setattr(PA, name, (128, 1))
    from shuffle_exchange_amd.ops import native
    native.require_hip()
    b, blocks = _batch(seqs, 64, "cuda", seed=3)
    g = torch.Generator(device="cuda").manual_seed(4)
    cache = torch.randn(blocks, 2, nkv, 64, 128, device="cuda", generator=g).to(torch.bfloat16)
    qkv = torch.randn(b.num_tokens, nq + 2 * nkv, 128, device="cuda", generator=g).to(torch.bfloat16)
    PA.kv_cache_append(qkv, cache, b.slots, nq, nkv)
    took = PA._flash_prompts(qkv[:, :nq], qkv[:, nq:], b, None)
    assert took == tuple((i, n // 128 * 128) for i, (c, n) in enumerate(seqs) if c == 0 and n >= 128)
    got = PA.ragged_attention(qkv[:, :nq], cache, b, 128 ** -0.5, kv=qkv[:, nq:])
    want = PA.ragged_attention(qkv[:, :nq], cache, b, 128 ** -0.5)  # checked against the reference above
    for i in range(b.num_seqs):
        s, n = b.host_q_start[i], b.host_q_len[i]
        # p and the output are rounded to 8 bits on either side: 2 x 2^-9 each
        assert ((got[s:s + n] - want[s:s + n]).float().norm() / want[s:s + n].float().norm()).item() < 8e-3, seqs[i]


def test_long_prompt_rule():
    """A prompt without history, long enough and with heads enough to fill the chip; never under a window."""
    class B:
        def __init__(self, *seqs):
            self.host_seen, self.host_q_len = [c for c, _ in seqs], [n for _, n in seqs]

    class T:
        is_cuda, dtype = True, torch.bfloat16

        def __init__(self, heads, D=128):
            self.shape, self.H = (1, heads, D), heads

        def stride(self):
            return (self.H * 128, 128, 1)
    b = B((0, 8192), (0, 8191), (64, 9000), (0, 9000), (0, 40), (0, 4096), (0, 3968))
    assert PA._flash_prompts(T(32), T(16), b, None) == ((0, 8192), (3, 8960), (5, 4096))
    assert PA._flash_prompts(T(16), T(8), b, None) == ((0, 8192),) and PA._flash_prompts(T(8), T(4), b, None) == ()
    assert PA._flash_prompts(T(32), T(16), b, 4096) == () == PA._flash_prompts(T(32), None, b, None) == PA._flash_prompts(T(32, 64), T(16), b, None)


def test_even_lengths():
    assert PA.even_lengths([]) and PA.even_lengths([7]) and PA.even_lengths([2000, 4000]) and PA.even_lengths([1000] * 30 + [1400])
    assert not PA.even_lengths([300, 4000]) and not PA.even_lengths([100] * 30 + [1000])
    b, _ = _batch([(100, 1), (3000, 1), (5, 60)], 16, "cpu")
    assert not b.even_lengths and not b.attention_lists(32, 9).seq_even
    b, _ = _batch([(2500, 1), (3000, 1), (5, 60)], 16, "cpu")
    assert not b.even_lengths and b.attention_lists(32, 9).seq_even


def test_short_splits_of_few_uneven_sequences():
    for seqs, nkv, keys, dim in ((8, 8, 3000, 128), (16, 8, 3072, 128), (2, 4, 512, 64), (3, 2, 10, 64)):  # splits of 512 keys would all run at once
        assert PA.choose_balanced_splits(seqs, nkv, keys, 1 << 10, False, dim) == max(PA.choose_splits(seqs, nkv, keys), -(-keys // 256))
    for seqs, nkv, keys, dim in ((16, 8, 3073, 128), (24, 8, 6000, 128), (4, 8, 3000, 256)):
        assert PA.choose_balanced_splits(seqs, nkv, keys, 1 << 10, False, dim) == max(PA.choose_splits(seqs, nkv, keys), -(-keys // 512))


@pytest.mark.parametrize("nkv", [1, 4, 8, 32])
def test_even_splits(nkv):
    """Even sequences: the fewest splits that fill the chip, or up to two more where the last round would be nearly empty."""
    for seqs in (1, 3, 16, 32, 50, 64, 96, 100, 128, 256):
        for keys in (1, 300, 512, 1024, 4096, 131072):
            plain, n = PA.choose_splits(seqs, nkv, keys), PA.choose_balanced_splits(seqs, nkv, keys, seqs * 16384, True)
            assert plain <= n <= plain + 2 and (n == plain or keys >= n * 320) and (n == plain or n * seqs * 16384 <= PA.PA_SPLIT_BYTES)
            if seqs * nkv * plain <= PA.PA_RESIDENT_WGS:
                assert n == plain


def test_two_workgroups_a_cu():
    """Whole rounds of 512 workgroups where the last of 768 is nearly empty, heads of 128 only, and then one split of even sequences."""
    took = [n for n in range(1, 4000) if PA.two_a_cu(n, 128)]
    assert {961, 1024, 2560}.issubset(took) and not {1, 512, 768, 960, 1025, 1280, 1536, 1792, 2048, 2304}.intersection(took)
    assert not PA.two_a_cu(1024, 64) and not PA.two_a_cu(1024, 256)
    assert PA.choose_balanced_splits(128, 8, 4000, 1 << 21, True) == 1 and PA.choose_balanced_splits(128, 8, 4000, 1 << 21) == 8
    assert PA.choose_balanced_splits(128, 8, 4000, 1 << 20, True, 64) == 1 and PA.choose_balanced_splits(128, 12, 4000, 1 << 20, True, 64) == 2
    assert PA.choose_balanced_splits(128, 8, 4000, 1 << 22, True, 256) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("seqs,nkv,group", [(32, 32, 1), (128, 8, 4), (61, 16, 20)])
@pytest.mark.parametrize("window", [None, 70])
def test_wide_chunks_match_reference(seqs, nkv, group, window):
    """One split on 64 keys a wave (more than 768 workgroups) against the gather: lengths around a wave's and a workgroup's chunk, several
    passes of 16 rows, blocks in any order, NaN behind a sequence's last key."""
    PA.native.require_hip()
    g = torch.Generator(device="cuda").manual_seed(seqs)
    bs, D, most = 16, 128, 300
    per = -(-most // bs)
    lens = [(1, 63, 64, 65, 255, 256, 257, 300)[i % 8] for i in range(seqs)]
    assert PA.two_a_cu(seqs * nkv, D)
    cache = torch.full((seqs * per, 2, nkv, bs, D), float("nan"), dtype=torch.bfloat16, device="cuda")
    bt = torch.randperm(seqs * per, generator=g, device="cuda").to(torch.int32).view(seqs, per)
    kv = torch.randn(seqs, 2, nkv, most, D, generator=g, device="cuda").bfloat16()
    for i, n in enumerate(lens):
        for b in range(-(-n // bs)):
            m = min(bs, n - b * bs)
            cache[int(bt[i, b]), :, :, :m] = kv[i, :, :, b * bs:b * bs + m]
    q = torch.randn(seqs, nkv * group, D, generator=g, device="cuda").bfloat16()
    one = torch.ones(seqs, dtype=torch.int32, device="cuda")
    meta = (bt, torch.arange(seqs, dtype=torch.int32, device="cuda"), one, torch.tensor(lens, dtype=torch.int32, device="cuda"))
    got = [torch.ops.sxe.paged_attention(q, cache, *meta, D ** -0.5, most, 1, window or 0, None, wide) for wide in (True, False)]
    want = PA.paged_attention_reference(q, cache, *meta, D ** -0.5, window)
    for y in got:  # bf16 weights and result: two roundings of 2^-9 on values that are averages of unit normals
        assert not y.isnan().any() and (y.float() - want.float()).norm() <= 2 ** -7 * want.float().norm()
    assert torch.equal(PA.paged_attention(q, cache, *meta, D ** -0.5, most, window=window, splits=1), got[0])


def test_short_splits_of_few_workgroups():
    """Splits of 128 keys are at most a workgroup a CU and stay within what partials may take; all else is as it was."""
    assert PA._decode_plan(1, 8, 1024, 1 << 14, False, 128, None) == (8, False) == PA._decode_plan(1, 8, 1024, 1 << 14, True, 128, None)
    for S in (1, 3, 8, 24, 33):
        for keys in (100, 256, 257, 1000, 2048, 2049, 8192):
            for nkv, dim, room in ((1, 128, 1 << 10), (8, 128, 1 << 14), (8, 128, 1 << 27), (8, 64, 1 << 14), (8, 256, 1 << 14)):
                was, n = PA.choose_balanced_splits(S, nkv, keys, room, True, dim), PA._decode_plan(S, nkv, keys, room, True, dim, None)[0]
                assert n == was or (dim == 128 and 256 < keys <= 2048 and was < n <= -(-keys // 128) and S * nkv * n <= 256 and n * room <= PA.PA_SPLIT_BYTES)


@pytest.mark.parametrize("target", [512, 4])
def test_graphs_by_lengths_only_where_the_splits_differ(target, monkeypatch):
    """A decode graph of sequences of like lengths and one of any lengths are two where attention takes other splits for them, not else."""
    from types import SimpleNamespace as N
    from shuffle_exchange_amd.inference.v2.decode_graphs import DecodeGraphRunner
    monkeypatch.setattr(PA, "PA_TARGET_WGS", target)  # few: chosen by the lengths, but for the short splits of few sequences
    seen = set()
    for nq, nkv, dim in ((32, 8, 128), (4, 2, 128), (12, 12, 64)):
        r = DecodeGraphRunner.__new__(DecodeGraphRunner)
        r.model, r._matters = N(nq=nq, nkv=nkv, head_dim=dim), {}
        for S in (2, 4, 12, 24, 64, 128):
            for kvb in (256, 512, 1024, 2048, 4096, 16384):
                plans = [PA.decode_plan(S, nkv, kvb, 4 * S * nq * dim, even, dim) for even in (True, False)]
                like, unlike = [N(seen_tokens=kvb - 1)] * S, [N(seen_tokens=kvb - 1)] + [N(seen_tokens=0)] * (2 * S)
                assert r._even(S, kvb, like) == (plans[0] != plans[1]) and not r._even(S, kvb, unlike)
                seen.add((dim, plans[0] != plans[1]))
    assert seen == {(dim, differ) for dim in (64, 128) for differ in (False, True)}

"""The weight-streaming GEMM of batched decode (csrc/kernels/stream_gemm.hip) against fp64: row counts, column remainders, K tails,
strided operands, e4m3 weights, bias and the gated form."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _native():
    from shuffle_exchange_amd.ops import native
    native.require_hip()


def _operands(M, N, K, fp8, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K + 24, generator=g, device="cuda").bfloat16()[:, 8:K + 8]  # rows 16 bytes into longer ones
    w = torch.randn(N, K, generator=g, device="cuda") * K ** -0.5
    if not fp8:
        w = w.bfloat16()
        return x, w, None, w.double()
    s = w.abs().amax(1) / 448
    q = (w / s[:, None]).to(torch.float8_e4m3fn)
    return x, q.view(torch.uint8), s, q.double() * s.double()[:, None]


def _rounding(values):
    """Products of bf16 are exact in fp32; left are fp32 sums and the rounding of the result. It is at most 2^-8 of a value (just above a power
    of two), which a result of a few values comes near; over many it is spread evenly, 2^-8 / sqrt(3) of the power of two below each, 1.7e-3
    of normal values together and more where a few large ones are most of their norm."""
    return 1.01 * 2 ** -8 if values.numel() < 256 else 3e-3


@pytest.mark.parametrize("M", [1, 5, 15, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(4, 16), (20, 1024), (6144, 96), (6148, 4112), (128, 2064), (8192, 2048)])
@pytest.mark.parametrize("fp8", [False, True])
def test_plain(M, N, K, fp8):
    x, w, s, ref = _operands(M, N, K, fp8, M + N + K)
    b = torch.randn(N, device="cuda").bfloat16()
    for bias in (None, b):
        got = torch.ops.sxe.stream_gemm(x, w, s, bias, False)
        want = x.double() @ ref.T + (0 if bias is None else b.double())
        assert (got.double() - want).norm() < _rounding(want) * want.norm()


@pytest.mark.parametrize("M", [1, 7, 8])
@pytest.mark.parametrize("N", [80, 4096, 4112, 8208])  # half tiles, then whole ones: at most one workgroup a CU, two, more
@pytest.mark.parametrize("K", [2048, 2056, 3072, 3080, 4096, 4104, 5000, 6152, 8200])
def test_pieces_in_flight(M, N, K):
    """Two at a time, or pieces of twice the size: any of the waves may have one more or one less than the others."""
    x, w, _, ref = _operands(M, N, K, False, M + N + K)
    want = x.double() @ ref.T
    assert (torch.ops.sxe.stream_gemm(x, w, None, None, False).double() - want).norm() < _rounding(want) * want.norm()
    assert (torch.ops.sxe.stream_gemm_normed(x, w, None, None, 0.0, False).double() - want).norm() < 1e-5 * want.norm()
    res, gw = torch.randn(M, N, device="cuda").bfloat16(), torch.ones(N, device="cuda").bfloat16()
    want = want + res.double()
    assert (torch.ops.sxe.stream_gemm_res(x, w, None, None, res, gw)[1].double() - want).norm() < _rounding(want) * want.norm()


def test_every_e4m3_value_is_exact():
    w = torch.arange(256, device="cuda", dtype=torch.uint8).view(16, 16)
    one = torch.ones(16, device="cuda")
    y = torch.ops.sxe.stream_gemm(torch.eye(16, device="cuda").bfloat16(), torch.where(w & 127 == 127, 0, w), one, None, False)
    want = torch.where(w & 127 == 127, 0, w).view(torch.float8_e4m3fn).float()
    assert torch.equal(y.float(), want.T) and not torch.ops.sxe.stream_gemm(torch.ones(1, 16, device="cuda").bfloat16(), w, one, None,
                                                                            False)[:, 7::8].isfinite().any()


@pytest.mark.parametrize("M", [5, 16, 32])
@pytest.mark.parametrize("N,K", [(32, 32), (96, 512), (64, 4096), (28672, 128)])
@pytest.mark.parametrize("fp8", [False, True])
def test_gated(M, N, K, fp8):
    x, w, s, ref = _operands(M, N, K, fp8, M + N + K)
    got = torch.ops.sxe.stream_gemm(x, w, s, None, True)
    g, u = (x.double() @ ref.T).chunk(2, -1)
    want = torch.nn.functional.silu(g) * u
    assert got.shape == (M, N // 2) and (got.double() - want).norm() < 3e-3 * want.norm()


@pytest.mark.parametrize("M", [5, 17])
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("fp8,N,K", [(False, 8256, 4112), (True, 16416, 4112), (True, 16448, 4096)])
def test_weights_read_past_the_caches(M, fp8, N, K, glu):
    """From 64 MB on the weight is loaded another way: the same bits as of its pieces, which are smaller."""
    x, w, s, _ = _operands(M, N, K, fp8, M + N + K)
    got = torch.ops.sxe.stream_gemm(x, w, s, None, glu)
    half = N // 2
    for a in range(0, half if glu else N, 2064):
        b = min(a + 2064, half if glu else N)
        part = torch.cat((w[a:b], w[half + a:half + b])) if glu else w[a:b]
        scale = None if s is None else torch.cat((s[a:b], s[half + a:half + b])) if glu else s[a:b]
        assert part.numel() * part.element_size() < 64 << 20
        assert torch.equal(got[:, a:b], torch.ops.sxe.stream_gemm(x, part.contiguous(), scale, None, glu))


def test_linear_routes_by_rows():
    """The rule's two sides agree: the streaming kernel, the library and the few-row kernel within one rounding of each other."""
    from shuffle_exchange_amd.ops.fp_quantizer import FP8Weight
    from shuffle_exchange_amd.ops.linear import glu_linear, linear
    w = (torch.randn(5120, 4096, device="cuda") / 64).bfloat16()
    fw = FP8Weight(w)
    with torch.no_grad():
        for M in (1, 4, 5, 16, 17, 33):
            x = torch.randn(M, 4096, device="cuda").bfloat16()
            want = x.double() @ w.double().T
            assert (linear(x, w).double() - want).norm() < 3e-3 * want.norm()
            if M <= 16:
                q = x.double() @ (fw.q.double() * fw.scale.double()[:, None]).T
                assert (linear(x, fw).double() - q).norm() < 3e-3 * q.norm()
            mid = glu_linear(x, w)
            assert (mid is not None) == (M <= 32)
            if mid is not None:
                g, u = want.chunk(2, -1)
                ref = torch.nn.functional.silu(g) * u
                assert (mid.double() - ref).norm() < 3e-3 * ref.norm()


@pytest.mark.parametrize("M", [1, 8, 9, 17, 32])
@pytest.mark.parametrize("N,K", [(16, 16), (48, 1032 - 8), (6160, 2064), (4096, 4096)])
@pytest.mark.parametrize("fp8", [False, True])
def test_residual_and_what_a_normed_product_needs(M, N, K, fp8):
    x, w, s, ref = _operands(M, N, K, fp8, M + N + K)
    res = torch.randn(M, N + 12, device="cuda").bfloat16()[:, 4:N + 4]
    gw = (1 + 0.3 * torch.randn(N, device="cuda")).bfloat16()
    y, h, sums = torch.ops.sxe.stream_gemm_res(x, w, s, None, res, gw)
    want = res.double() + x.double() @ ref.T
    assert (h.double() - want).norm() < _rounding(want) * want.norm()
    assert torch.equal(y, (h.float() * gw.float()).bfloat16())
    tiles, rows = sums.shape
    assert N // tiles in (8, 16) and rows in (8, 16, 32) and rows >= M and not sums[:, M:].any()
    squares = h.double().square().view(M, tiles, N // tiles).sum(-1)
    assert (sums[:, :M].T.double() - squares).abs().max() <= 1e-6 * squares.max()


@pytest.mark.parametrize("N,heads,dim,splits", [(16, 1, 64, 1), (2048, 16, 128, 5), (2032, 9, 128, 8), (512, 16, 128, 17), (64, 3, 256, 9)])
@pytest.mark.parametrize("fp8", [False, True])
def test_residual_of_a_row_in_splits(N, heads, dim, splits, fp8):
    from shuffle_exchange_amd.ops.paged_attention import merge_attention_parts
    _, w, s, ref = _operands(1, N, heads * dim, fp8, N + splits)
    po = torch.randn(splits, 1, heads, dim, device="cuda")
    pml = torch.stack([torch.randn(splits, 1, heads, device="cuda") * 4, torch.rand(splits, 1, heads, device="cuda") + 0.5], -1)
    if splits > 1:  # splits without keys: nothing is behind their maximum
        pml[1::3, ..., 0], pml[1::3, ..., 1], po[1::3] = float("-inf"), float("nan"), float("nan")
    res, gw = torch.randn(1, N, device="cuda").bfloat16(), (1 + 0.3 * torch.randn(N, device="cuda")).bfloat16()
    got = torch.ops.sxe.stream_gemm_res_splits(po, pml, w, s, res, gw)
    row = merge_attention_parts(po[pml[:, 0, 0, 0] > -1e30], pml[pml[:, 0, 0, 0] > -1e30], torch.float32).view(1, -1)
    want = res.double() + row.double() @ ref.T
    # the row's rounding to bf16 (2^-8 at most) on its way into the product, then that of the result
    assert (got[1].double() - want).norm() < _rounding(want) * (want.norm() + (want - res.double()).norm())
    assert torch.equal(got[0], (got[1].float() * gw.float()).bfloat16())
    squares = got[1].double().square().view(len(got[2]), -1).sum(-1)
    assert (got[2][:, 0].double() - squares).abs().max() <= 1e-6 * squares.max() and not got[2][:, 1:].any()


@pytest.mark.parametrize("M", [1, 8, 9, 17, 32])
@pytest.mark.parametrize("N,K,tiles", [(32, 16, 1), (96, 1024, 3), (6208, 2064, 129), (8192, 4096, 256), (16416, 4112, 600)])
@pytest.mark.parametrize("fp8", [False, True])
def test_products_behind_a_norm(M, N, K, tiles, fp8):
    """The sums come from any number of tiles; what they say of the rows is up to who made them. From 64 MB on weights pass the caches."""
    x, w, s, ref = _operands(M, N, K, fp8, M + N + K)
    sums = torch.rand(tiles, 8 if M <= 8 else 16 if M <= 16 else 32, device="cuda") * 3
    p = x.double() @ ref.T * (sums[:, :M].double().sum(0) / K + 1e-3).rsqrt()[:, None]
    got = torch.ops.sxe.stream_gemm_normed(x, w, s, sums, 1e-3, False)
    assert got.dtype == torch.float32 and (got.double() - p).norm() < 1e-5 * p.norm()
    g, u = p.chunk(2, -1)
    mid = torch.ops.sxe.stream_gemm_normed(x, w, s, sums, 1e-3, True)
    want = torch.nn.functional.silu(g) * u
    assert (mid.double() - want).norm() < _rounding(want) * want.norm()
    plain = torch.ops.sxe.stream_gemm_normed(x, w, s, None, 0.0, False)
    assert torch.equal(plain.bfloat16(), torch.ops.sxe.stream_gemm(x, w, s, None, False))


@pytest.mark.parametrize("M", [1, 9, 17, 32])
@pytest.mark.parametrize("nq,nkv,K", [(1, 1, 16), (4, 2, 1024), (48, 8, 2064)])  # one and two tiles a workgroup
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("normed", [False, True])
def test_rotated_heads_and_the_cache(M, nq, nkv, K, fp8, normed):
    x, w, s, ref = _operands(M, (nq + 2 * nkv) * 128, K, fp8, M + nq + K)
    sums = torch.rand(7, 8 if M <= 8 else 16 if M <= 16 else 32, device="cuda") if normed else None
    a = torch.rand(50, 64, device="cuda") * 6.28
    pos = torch.randint(0, 50, (M,), device="cuda")
    slots = torch.randperm(5 * 16, device="cuda")[:M]
    slots[::5] = -1
    cache = torch.full((5, 2, nkv, 16, 128), 7.0, device="cuda").bfloat16()
    got = torch.ops.sxe.stream_gemm_rope(x, w, s, sums, 1e-3, a.cos(), a.sin(), pos, slots, cache, nq, nkv)
    p = x.double() @ ref.T
    if normed:
        p = p * (sums[:, :M].double().sum(0) / K + 1e-3).rsqrt()[:, None]
    p = p.view(M, nq + 2 * nkv, 2, 64)
    c, sn = a.cos().double()[pos][:, None], a.sin().double()[pos][:, None]
    lo, hi = p.unbind(2)
    want = torch.stack([lo * c - hi * sn, hi * c + lo * sn], 2)
    want[:, nq + nkv:] = p[:, nq + nkv:]
    want = want.view(M, nq + 2 * nkv, 128)
    got = got.view(M, nq + 2 * nkv, 128)
    assert (got.double() - want).norm() < _rounding(want) * want.norm()
    expect = torch.full_like(cache, 7.0)
    for i, at in enumerate(slots.tolist()):
        if at >= 0:
            expect[at // 16, 0, :, at % 16], expect[at // 16, 1, :, at % 16] = got[i, nq:nq + nkv], got[i, nq + nkv:]
    assert torch.equal(cache, expect)


@pytest.mark.parametrize("quant", [None, "fp8"])
@pytest.mark.parametrize("hidden,heads,kv,experts", [(512, 4, 2, 0), (2304, 18, 2, 0), (512, 4, 2, 2)])  # half tiles and whole ones
def test_layers_of_chained_products(hidden, heads, kv, experts, quant, monkeypatch):
    """Prompts, decode steps and a pass whose logits are not one a sequence, by either route over the same cache. With experts every token
    has all of them, so that no near tie of the router goes another way."""
    from shuffle_exchange_amd.inference.v2 import RaggedInferenceEngineConfig, build_engine
    from shuffle_exchange_amd.inference.v2.model_implementations import llama as module
    from shuffle_exchange_amd.models import LlamaForCausalLM, MixtralForCausalLM, llama_config, mixtral_config
    torch.manual_seed(1)
    sizes = dict(hidden_size=hidden, intermediate_size=1408, num_hidden_layers=2, num_attention_heads=heads, num_key_value_heads=kv, head_dim=128,
                 vocab_size=1000, max_position_embeddings=512)
    model = (MixtralForCausalLM(mixtral_config("mixtral-tiny", num_local_experts=experts, num_experts_per_tok=experts, **sizes)) if experts
             else LlamaForCausalLM(llama_config("llama-tiny", **sizes))).to("cuda", torch.bfloat16)
    g = torch.Generator().manual_seed(2)
    chained, runs, calls = [], [], {}
    own = module.RaggedLlama._chain

    def counted(name):
        of = getattr(module, name)

        def call(*args):
            y = of(*args)
            calls[name] = calls.get(name, 0) + (y is not None)
            return y
        monkeypatch.setattr(module, name, call)
    for name in ("embed_normed", "stream_rope", "stream_res", "stream_res_splits", "stream_glu", "stream_head"):
        counted(name)
    for on in (True, False):
        def chain(self, *args):
            chained.append(on and own(self, *args) is not None)
            return own(self, *args) if on else None
        monkeypatch.setattr(module.RaggedLlama, "_chain", chain)
        g.manual_seed(2)
        e = build_engine(model, RaggedInferenceEngineConfig(kv_block_size=16, num_kv_blocks=200, weight_quant=quant))
        out = [e.put([i], [torch.randint(0, 1000, (n,), generator=g)]) for i, n in enumerate((7, 31, 3, 300))]
        for uids in ([0, 1, 2], [3], [0, 2]):
            for _ in range(2):
                out.append(e.put(uids, [torch.randint(0, 1000, (1,), generator=g) for _ in uids]))
        out.append(e.put([0, 1], [torch.randint(0, 1000, (n,), generator=g) for n in (5, 1)], want=[(1, 4, 0), ()]))
        runs.append(out)
    # three short prompts and one of 300 tokens, the steps' three graphs, each of a pass before its capture and the captured one, a mixed pass
    assert chained == [True] * 3 + [False] + [True] * 7 + [False] * 11
    splits = 4 if hidden <= 2048 and not experts else 0  # the graph of one sequence of 300 keys: two layers, twice
    want = {"embed_normed": 10, "stream_rope": 20}
    if not experts:  # else two launches of the norm a layer, and the head behind one
        want.update(stream_res=40 - splits, stream_glu=20, stream_head=6, **({"stream_res_splits": splits} if splits else {}))
    assert calls == want
    for a, b in zip(*runs):
        assert a.dtype == b.dtype and a.shape == b.shape
        # roundings to bf16 (2^-9 in the mean square) of a dozen tensors a layer, other ones by either route
        assert (a - b).norm() < 0.02 * b.norm()


@pytest.mark.parametrize("which", ["layers.1.input_layernorm", "layers.0.post_attention_layernorm", "norm"])
def test_norm_weights_anywhere_in_a_buffer(which):
    """A parameter that starts between two loads of four of its values: the norm is a launch of its own again."""
    from shuffle_exchange_amd.inference.v2 import RaggedInferenceEngineConfig, build_engine
    from shuffle_exchange_amd.models import LlamaForCausalLM, llama_config
    torch.manual_seed(3)
    cfg = llama_config("llama-tiny", hidden_size=512, intermediate_size=1408, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2,
                       head_dim=128, vocab_size=1000)
    model = LlamaForCausalLM(cfg).to("cuda", torch.bfloat16)
    norm, runs = model.get_submodule(which), []
    weight = (1 + 0.3 * torch.randn(516, device="cuda")).bfloat16()
    for start in (0, 2):
        norm.weight = torch.nn.Parameter(weight.roll(start)[start:start + 512])
        assert norm.weight.data_ptr() % 8 == 2 * start
        e, g = build_engine(model, RaggedInferenceEngineConfig(kv_block_size=16, num_kv_blocks=60)), torch.Generator().manual_seed(4)
        runs.append([e.put(list(range(5)), [torch.randint(0, 1000, (n,), generator=g) for n in lens]) for lens in ((3, 1, 8, 2, 5), (1, 1, 1, 1, 1))])
    for a, b in zip(*runs):  # roundings to bf16 (2^-9 in the mean square) of a dozen tensors a layer, other ones by either route
        assert (a - b).norm() < 0.02 * b.norm()


@pytest.mark.parametrize("n", [1, 8, 9, 32])
@pytest.mark.parametrize("K", [8, 1032, 2048, 4104])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_rows_of_the_embedding_with_their_squares(n, K, dtype):
    from shuffle_exchange_amd.ops.rows import embed, embed_normed
    g = torch.Generator(device="cuda").manual_seed(n + K)
    w = torch.randn(50, K, generator=g, device="cuda").bfloat16()
    gw = (1 + 0.3 * torch.randn(K, generator=g, device="cuda")).bfloat16()
    ids = torch.randint(-3, 54, (n,), generator=g, device="cuda").to(dtype)  # ids outside read zeros
    scaled, rows, sums = embed_normed(w, ids, gw)
    assert torch.equal(rows, embed(w, ids)) and torch.equal(scaled, (rows.float() * gw.float()).bfloat16())
    want = rows.double().square().sum(1)
    assert sums.shape == (1, 8 if n <= 8 else 16 if n <= 16 else 32) and not sums[0, n:].any()
    assert (sums[0, :n].double() - want).abs().max() <= 1e-6 * want.max()  # fp32 sums of exact squares, a tree of at most 25 steps
    assert embed_normed(w.float(), ids, gw) is None and embed_normed(w, ids, gw.float()) is None and embed_normed(w[:, 4:], ids, gw[4:]) is None
    assert embed_normed(w, ids.repeat(33), gw) is None

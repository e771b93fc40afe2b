"""Products of many rows (csrc/kernels/gemm_tn.hip) against 64 bits, and the calls of ops/linear.py that take them."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _native():
    from shuffle_exchange_amd.ops import native
    native.require_hip()


def _operands(M, N, K, apart=0):
    g = torch.Generator("cuda").manual_seed(M + 3 * N + 7 * K)
    x = torch.randn(M, K + apart, device="cuda", generator=g).bfloat16()[:, :K]
    w = (torch.randn(N, K + 2 * apart, device="cuda", generator=g) * K ** -0.5).bfloat16()[:, :K]
    return x, w, torch.randn(N, device="cuda", generator=g).bfloat16()


def _close(y, ref, x, w, factor=1.0):
    """One rounding to bf16 (2^-9) of fp32 sums of K exact products (each off by at most K 2^-24 of the magnitudes' sum)."""
    assert y.dtype == torch.bfloat16 and y.shape == ref.shape
    sums = x.double().abs() @ w.double().abs().t() * x.shape[1] * 2.0 ** -24
    bound = ref.abs() * 2.0 ** -8 + (sums if sums.shape == ref.shape else sums.amax()) * factor + 1e-30
    assert bool(((y.double() - ref).abs() <= bound).all())


# tiles: 256 x 256, 192 x 256, 128 x 256, 128 x 128, the plan's. Rows around a tile and its 16-row blocks, columns that end inside
# a store's 8, a lane's 32 and a tile's 256, one slab of K to more than the slots hold
@pytest.mark.parametrize("tile", [0, 1, 2, 3, -1])
@pytest.mark.parametrize("splits", [1, 3, 0])
@pytest.mark.parametrize("M,N,K,apart", [(1, 8, 64, 0), (15, 40, 128, 8), (128, 264, 192, 0), (193, 256, 320, 16), (257, 520, 64, 0),
                                         (385, 1000, 640, 8), (512, 272, 1024, 0)])
def test_products(M, N, K, apart, splits, tile):
    x, w, b = _operands(M, N, K, apart)
    ref = x.double() @ w.double().t()
    _close(torch.ops.sxe.gemm_tn(x, w, None, False, tile, splits), ref, x, w)
    _close(torch.ops.sxe.gemm_tn(x, w, b, False, tile, splits), ref + b.double(), x, w, 2.0)
    if N % 16 == 0:
        gate, up = ref.chunk(2, 1)
        # both sums' errors through silu(gate) up: |silu'| <= 1.1, values up to about 6
        _close(torch.ops.sxe.gemm_tn(x, w, None, True, tile, splits), F.silu(gate) * up, x, w, 16.0)


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("M", [base + rest for base in (0, 768) for rest in (1, 63, 64, 65, 127, 128, 129)])
def test_small_last_tiles(M, splits):
    """The last rows run as a tile of 64 or 128 rows: the sums are those of whole tiles, in the same order, whichever tile the rest has, and
    rows behind it that are not in use, zeros, stay zeros."""
    x, w, b = _operands(M, 528, 320)
    ref = x.double() @ w.double().t()
    for glu in (False, True):
        got = [torch.ops.sxe.gemm_tn(x, w, None if glu else b, glu, tile, splits) for tile in range(4)]
        assert all(torch.equal(got[0], y) for y in got[1:])
    _close(torch.ops.sxe.gemm_tn(x, w, None, False, 0, splits), ref, x, w)
    rows = torch.tensor([M // 2, M], device="cuda", dtype=torch.int32)
    xb, wb = torch.stack((x, x)), torch.stack((w, w))
    xb[0, M // 2:] = 0
    for tile in range(4):
        y = torch.ops.sxe.gemm_tn_batch(xb, wb, tile, rows)
        assert not y[0, M // 2:].any() and torch.equal(y[0, :M // 2], y[1, :M // 2])
        _close(y[1], ref, x, w)


@pytest.mark.parametrize("tile", [0, 1, 2, 3, -1])
@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (129, 264, 192), (321, 776, 640)])
def test_products_in_32_bits(M, N, K, tile):
    """Written to and added to a buffer in fp32: the sums before their rounding; nothing behind it is touched."""
    x, w, _ = _operands(M, N, K)
    ref, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    behind = torch.full((M * N + 8,), float("nan"), device="cuda")
    c = behind[:M * N].view(M, N)
    for times in (1, 2):  # each sum is off by at most K 2^-24 of the magnitudes' sum
        torch.ops.sxe.gemm_tn_into(x, w, c, times == 2, tile)
        assert bool(((c.double() - times * ref).abs() <= times * (K + 2) * 2.0 ** -24 * size).all())
    assert bool(behind[M * N:].isnan().all())
    with pytest.raises(RuntimeError):
        torch.ops.sxe.gemm_tn_into(x, w, c[:, :-1], False)


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("M,N,K,splits", [(1, 8, 128, 2), (129, 264, 320, 2), (321, 776, 640, 3), (65, 40, 704, 8)])
def test_split_products_in_32_bits(M, N, K, splits, tile):
    """The same of products that are split along K, and of a few rows and many tokens, which the plan splits."""
    x, w, _ = _operands(M, N, K)
    ref, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    behind = torch.full((M * N + 8,), float("nan"), device="cuda")
    c = behind[:M * N].view(M, N)
    for times in (1, 2):
        torch.ops.sxe.gemm_tn_into(x, w, c, times == 2, tile, splits)
        assert bool(((c.double() - times * ref).abs() <= times * (K + 2 + splits) * 2.0 ** -24 * size).all())
    assert bool(behind[M * N:].isnan().all())


def test_a_small_tables_gradient_fills_the_card():
    """515 x 768 of 8192 tokens have 15 tiles: split along the tokens, as the product in bf16 is, to the same sums."""
    x, w, _ = _operands(515, 768, 8192)
    c, one = torch.zeros(515, 768, device="cuda"), torch.zeros(515, 768, device="cuda")
    torch.ops.sxe.gemm_tn_into(x, w, c, False)
    torch.ops.sxe.gemm_tn_into(x, w, one, False, -1, 1)
    assert torch.equal(c.bfloat16(), torch.ops.sxe.gemm_tn(x, w, None, False)) and not torch.equal(c, one)


def test_head_gradient_into_the_optimizers_buffer():
    """A table that embeds and ends a model: both gradients meet in the buffer, as autograd's sum of them does."""
    from shuffle_exchange_amd.ops.cross_entropy import head_cross_entropy
    from shuffle_exchange_amd.ops.linear import Embedding
    torch.manual_seed(0)
    emb = Embedding(515, 128).cuda().bfloat16()
    ids = torch.randint(0, 515, (2, 75), device="cuda")
    p, valid = emb.weight, []

    def run():
        head_cross_entropy(emb(ids), p, ids).backward()
    run()
    want, p.grad = 2 * p.grad.float(), None
    buf = torch.full(p.shape, float("nan"), device="cuda")
    p._sxe_grad_target, p._sxe_grad_done, p._sxe_grad_local = (lambda q: (buf, bool(valid))), valid.append, True
    run()
    run()
    assert len(valid) == 4 and p.grad is None and (buf - want).norm() <= 2 ** -7 * want.norm()  # autograd's pieces were rounded to 8 bits


def test_infinities_and_nan_stay_in_their_rows():
    x, w, _ = _operands(300, 512, 256)
    x[7, 3], x[299, 0] = float("inf"), float("nan")
    for glu in (False, True):
        y = torch.ops.sxe.gemm_tn(x, w, None, glu)
        bad = ~torch.isfinite(y).all(1)
        assert bad.nonzero().flatten().tolist() == [7, 299] and bool(torch.isnan(y[299]).all())


@pytest.mark.parametrize("M,N,K,taken", [(1536, 2048, 2048, False), (1537, 2048, 2048, True), (1537, 2040, 2048, False), (300, 2048, 8192, True),
                                         (33, 2048, 8192, True), (300, 4096, 4096, False)])
def test_linear_takes_them(M, N, K, taken, monkeypatch):
    from shuffle_exchange_amd.ops import linear as L
    x, w, b = _operands(M, N, K)
    seen = [None]
    tiled = L._tiled
    monkeypatch.setattr(L, "_tiled", lambda *a: seen.append(tiled(*a)) or seen[-1])
    with torch.no_grad():
        y = L.linear(x.view(1, M, K), w, b)
        assert (seen[-1] is not None) == taken
        _close(y[0], x.double() @ w.double().t() + b.double(), x, w, 2.0)
        # what the kernel does not read goes where it went before: rows apart by no whole 16 bytes, another type
        odd = torch.randn(M, K + 4, device="cuda").bfloat16()[:, :K]
        assert torch.equal(L.linear(odd, w), F.linear(odd, w)) and seen[-1] is None
        with torch.autocast("cuda", torch.float16):
            assert L.linear(x, w).dtype == torch.float16
    n = len(seen)
    assert L.linear(x.requires_grad_(), w).requires_grad and len(seen) == n


def test_wide_weights_rule():
    from shuffle_exchange_amd.ops.linear import _tiled_faster as own
    assert own(1025, 6144, 3072) and own(1499, 6144, 3072) and not own(1024, 6144, 3072) and not own(1280, 6144, 3072)
    assert not own(1025, 6128, 3072) and not own(1025, 6144, 2048)


@pytest.mark.parametrize("C", [1, 16, 129, 257, 300])
@pytest.mark.parametrize("E,K,N", [(1, 64, 128), (3, 192, 320), (8, 64, 576)])
def test_expert_products(E, C, K, N):
    """All experts' products in a launch, with the weights as they lie and transposed, and the gradients of the layer that runs them."""
    from shuffle_exchange_amd.moe.experts import expert_products, grouped_mm
    g = torch.Generator("cuda").manual_seed(C)
    x = torch.randn(E, C, K, device="cuda", generator=g).bfloat16()
    w = (torch.randn(E, K, N, device="cuda", generator=g) * K ** -0.5).bfloat16()
    dy = torch.randn(E, C, N, device="cuda", generator=g).bfloat16()
    y, dx = expert_products(x, w), expert_products(dy, w, transposed=True)
    for tile in range(4):
        assert torch.equal(torch.ops.sxe.gemm_tn_batch(dy, w, tile), dx)
    for e in range(E):
        _close(y[e], x[e].double() @ w[e].double(), x[e], w[e].t())
        _close(dx[e], dy[e].double() @ w[e].double().t(), dy[e], w[e])
    xg, wg = x.clone().requires_grad_(), w.clone().requires_grad_()
    out = grouped_mm(xg, wg)
    out.backward(dy)
    assert torch.equal(out, y) and torch.equal(xg.grad, dx)
    for other in (x[:, :, :K - 32].contiguous(), x.float(), x.transpose(1, 2)):  # not covered: the caller's loop over the experts
        assert expert_products(other, w) is None


@pytest.mark.parametrize("rows", [(3, 515), (1545,), (4, 384)])
def test_training_products(rows):
    """Forward and data gradient of a layer that writes its weight gradient itself; its result may be changed in place, as RoPE does."""
    from shuffle_exchange_amd.ops import linear as L
    x, w, _ = _operands(1545, 2048, 2048)
    x = x.contiguous().view(*rows, 2048) if len(rows) == 1 or rows[0] * rows[1] == 1545 else x[:1536].contiguous().view(*rows, 2048)
    dy = torch.randn(*rows, 2048, device="cuda", generator=torch.Generator("cuda").manual_seed(1)).bfloat16()
    x.requires_grad_()
    p = torch.nn.Parameter(w.contiguous())
    buf = torch.zeros(2048, 2048, device="cuda")
    p._sxe_grad_target, p._sxe_grad_done = (lambda q: (buf, False)), (lambda q: None)
    y = L.linear(x, p)
    _close(y.detach().view(-1, 2048), x.detach().view(-1, 2048).double() @ w.double().t(), x.detach().view(-1, 2048), w)
    y.view(*rows, 16, 128)[..., :4, :].mul_(2.0)
    y.backward(dy)
    d = dy.clone()
    d.view(*rows, 16, 128)[..., :4, :].mul_(2.0)
    _close(x.grad.view(-1, 2048), d.view(-1, 2048).double() @ w.double(), d.view(-1, 2048), w.t())
    want = d.view(-1, 2048).double().t() @ x.detach().view(-1, 2048).double()
    assert (buf.double() - want).norm() <= 1e-5 * want.norm()
    # many columns to sum over: few rows take the transposed weight, too
    wide = (torch.randn(16384, 2048, device="cuda") * 128 ** -1).bfloat16()
    g = torch.randn(300, 16384, device="cuda").bfloat16()
    _close(L.data_grad(g, wide), g.double() @ wide.double(), g, wide.t())


# tokens: inside a slab of 64, whole slabs, more than the slots hold, pieces that end inside a slab; sizes that end inside a tile of 256 or
# 128, a block of 16, a store of 4 columns; one product or three
@pytest.mark.parametrize("E,T,T2,M,N", [(0, 1, 0, 8, 8), (0, 63, 0, 264, 40), (0, 64, 0, 128, 256), (0, 577, 0, 192, 1000), (0, 640, 0, 256, 512),
                                        (0, 128, 72, 256, 264), (0, 100, 30, 136, 256), (3, 70, 0, 264, 128), (3, 90, 65, 264, 128)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_weight_gradients(E, T, T2, M, N, accumulate):
    g = torch.Generator("cuda").manual_seed(T + M)
    batch = (E,) if E else ()
    a, b, a2, b2 = [torch.randn(*batch, t, n + 8, device="cuda", generator=g).bfloat16()[..., :n] for t in (T, T2) for n in (M, N)]
    before = torch.randn(*batch, M, N, device="cuda", generator=g)
    sums = a.double().transpose(-1, -2) @ b.double() + a2.double().transpose(-1, -2) @ b2.double()
    want = 0.5 * sums + (before.double() if accumulate else 0)
    # fp32 sums of T exact products each: T 2^-24 of the magnitudes' sum
    bound = (a.double().abs().transpose(-1, -2) @ b.double().abs() + a2.double().abs().transpose(-1, -2) @ b2.double().abs()) * (T + T2 + 8) * 2.0 ** -24
    bound += (want.abs() + before.double().abs()) * 2.0 ** -22
    forms = [None] if T2 or E else [None, 0, 1, 16 * 3, 16 * 2 + 1]  # 256 x 256, 128 x 256, splits
    for form in forms:
        c = before.clone() if accumulate else torch.full_like(before, float("nan"))
        if T2:
            torch.ops.sxe.wgrad_gemm2_(a, b, a2, b2, c, 0.5, accumulate)
        elif form is None:
            torch.ops.sxe.wgrad_gemm_(a, b, c, 0.5, accumulate)
        else:
            torch.ops.sxe.wgrad_gemm_variant_(a, b, c, 0.5, accumulate, form)
        assert bool(((c.double() - want).abs() <= bound).all()), form


def test_captured():
    """Replays with new inputs; the splits' sums are the graph's own memory."""
    x, w, _ = _operands(300, 2048, 8192)
    from shuffle_exchange_amd.ops.linear import linear
    with torch.no_grad():
        linear(x, w)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = linear(x, w)
        for seed in range(3):
            x.copy_(torch.randn(300, 8192, device="cuda", generator=torch.Generator("cuda").manual_seed(seed)).bfloat16())
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, linear(x, w))


@pytest.mark.parametrize("C", [1, 64, 100, 256, 320, 700])
def test_expert_products_of_rows_in_use(C):
    """Rows behind those in use are zeros and left out: the same bits as all rows, for no row, a row, edges of slabs and tiles, all rows; both
    products, and the weight gradient in one piece and in two, with tokens that end inside a slab."""
    from shuffle_exchange_amd.moe.experts import expert_products
    E, K, N = 6, 128, 320
    g = torch.Generator("cuda").manual_seed(C)
    R = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()
    w = R(E, K, N) * K ** -0.5

    def piece(used):
        rows = torch.tensor([min(C, u) for u in used], device="cuda", dtype=torch.int32)
        live = torch.arange(C, device="cuda")[None, :, None] < rows[:, None, None]
        return rows, R(E, C, K) * live, R(E, C, N) * live
    a, b = piece((0, 1, 63, 64, 257, C)), piece((65, 0, 256, 128, 1, C - 1))
    nan = lambda *s: torch.full(s, float("nan"), device="cuda", dtype=torch.bfloat16)
    for rows, x, dy in (a, b):
        nan(E, C, N), nan(E, C, K)  # what the results' memory may hold before
        assert torch.equal(expert_products(x, w, rows=rows), expert_products(x, w))
        assert torch.equal(expert_products(dy, w, transposed=True, rows=rows), expert_products(dy, w, transposed=True))
        for tile in range(4):
            assert torch.equal(torch.ops.sxe.gemm_tn_batch(dy, w, tile, rows), torch.ops.sxe.gemm_tn_batch(dy, w, tile))
    for accumulate in (False, True):
        def both(f):
            out = [torch.randn(E, K, N, device="cuda", generator=torch.Generator("cuda").manual_seed(1)) for _ in range(2)]
            f(out[0], False), f(out[1], True)
            assert torch.equal(*out)
        both(lambda c, r: torch.ops.sxe.wgrad_gemm_(a[1], a[2], c, 0.5, accumulate, a[0] if r else None))
        both(lambda c, r: torch.ops.sxe.wgrad_gemm2_(a[1], a[2], b[1], b[2], c, 1.0, accumulate, a[0] if r else None, b[0] if r else None))
        both(lambda c, r: torch.ops.sxe.wgrad_gemm2_(a[1], a[2], b[1], b[2], c, 1.0, accumulate, None, b[0] if r else None))
    with pytest.raises(RuntimeError):
        expert_products(a[1], w, rows=a[0].long())
    with pytest.raises(RuntimeError):
        expert_products(a[1], w, rows=a[0][:-1])


@pytest.mark.parametrize("N,K", [(512, 512), (768, 3072), (2304, 768), (1344, 1088), (3072, 768)])
@pytest.mark.parametrize("rows", [33, 300, 1025])
def test_narrow_products_of_training(N, K, rows):
    """Weights that are narrow one way, inside autograd functions: forward with a bias and data gradient on the own products, and what they do
    not cover on the library's."""
    from shuffle_exchange_amd.ops import linear as L
    g = torch.Generator("cuda").manual_seed(rows)
    R = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()
    x, w, b, dy = R(rows, K), R(N, K) * K ** -0.5, R(N), R(rows, N)
    with torch.no_grad():
        assert L._narrow(rows, N, K) and not L._narrow(32, N, K) and not L._narrow(10 ** 10 // (N * K) + 1, N, K)
        y = L.product(x, w, b)
        _close(y, x.double() @ w.double().t() + b.double(), x, w)
        assert torch.equal(L.product(x.view(1, rows, K), w, b)[0], y)
        dx = L._narrow_data_grad(dy, w)
        _close(dx, dy.double() @ w.double(), dy, w.t())
        assert torch.equal(L.data_grad(dy.view(1, rows, N), w)[0], dx)
        odd = R(rows + 1, N + 1)[1:, 1:]  # rows that start off 16 bytes
        assert L._narrow_data_grad(odd, w) is None and L._narrow_data_grad(dy.float(), w.float()) is None
        _close(L.data_grad(odd, w), odd.double() @ w.double(), odd, w.t())
    assert L._narrow_data_grad(dy.requires_grad_(), w) is None  # a graph is recorded


def test_gpt2_block_packed_attention():
    """Attention over the projection as it lies and the residual inside the second norm: values and gradients of the block by plain operators."""
    from shuffle_exchange_amd.models.gpt2 import GPT2Block, gpt2_config
    import torch.nn.functional as F
    torch.manual_seed(0)
    cfg = gpt2_config("gpt2-tiny", n_embd=128, n_head=2)
    blk = GPT2Block(cfg).cuda().bfloat16()
    x = torch.randn(2, 70, 128, device="cuda").bfloat16().requires_grad_()
    dy = torch.randn(2, 70, 128, device="cuda").bfloat16()
    y = blk(x)
    got = torch.autograd.grad(y, [x, *blk.parameters()], dy)
    P = {n: p.detach().double().requires_grad_() for n, p in blk.named_parameters()}
    xd = x.detach().double().requires_grad_()
    ln = lambda t, n: F.layer_norm(t, (128,), P[n + ".weight"], P[n + ".bias"], 1e-5)
    lin = lambda t, n: t @ P[n + ".weight"].t() + P[n + ".bias"]
    q, k, v = (t.transpose(1, 2) for t in lin(ln(xd, "ln_1"), "c_attn").view(2, 70, 3, 2, 64).unbind(2))
    s = (q @ k.transpose(-1, -2) / 8).masked_fill(torch.ones(70, 70, device="cuda", dtype=torch.bool).triu(1), float("-inf"))
    h = xd + lin((s.softmax(-1) @ v).transpose(1, 2).reshape(2, 70, 128), "c_proj")
    want = h + lin(F.gelu(lin(ln(h, "ln_2"), "c_fc"), approximate="tanh"), "mlp_proj")
    assert (y.double() - want).norm() <= 4e-3 * want.norm()  # roundings to 8 bits of the sums: 2^-9 each
    for a, b in zip(got, torch.autograd.grad(want, [xd, *P.values()], dy.double())):
        assert (a.double() - b).norm() <= 2e-2 * b.norm(), a.shape  # a chain of a dozen of them


@pytest.mark.parametrize("M,N,K,taken", [(33, 512, 512, True), (768, 3072, 2048, True), (769, 3072, 2048, False), (32, 3072, 2048, False), (85, 28672, 4096, True),
                                         (86, 28672, 4096, False), (300, 4096, 4096, True), (300, 4096, 448, False)])
def test_short_products_of_eager_passes(M, N, K, taken, monkeypatch):
    """Calls that wait for the host: own products from 33 rows on, with what these do not read, and what is captured, left to the library."""
    from shuffle_exchange_amd.ops import linear as L
    x, w, b = _operands(M, N, K)
    seen = [None]
    tiled = L._tiled
    monkeypatch.setattr(L, "_tiled", lambda *a: seen.append(tiled(*a)) or seen[-1])
    with torch.no_grad():
        y = L.linear(x, w, b, True)
        assert (seen[-1] is not None) == taken
        _close(y, x.double() @ w.double().t() + b.double(), x, w, 2.0)
        seen.append(None)
        odd = torch.randn(M, K + 4, device="cuda").bfloat16()[:, :K]
        assert torch.equal(L.linear(odd, w, None, True), F.linear(odd, w)) and seen[-1] is None
        n = len(seen)
        monkeypatch.setattr(L, "_capturing", lambda: True)
        if M > 32:
            assert torch.equal(L.linear(x, w, b, True), F.linear(x, w, b)) and len(seen) == n
    assert L.linear(x.requires_grad_(), w, b, True).requires_grad


@pytest.mark.parametrize("shape", [(5, 256), (2, 3, 1024), (1, 4128)])
def test_norms_and_gates_without_a_graph(shape):
    """The forward by itself and inside its autograd function: the same bits, for rows that lie apart, too."""
    from shuffle_exchange_amd.ops.activation import gated_act
    from shuffle_exchange_amd.ops.norm import layer_norm, rms_norm
    H = shape[-1]
    x = torch.randn(*shape[:-1], H + 8, device="cuda").bfloat16()[..., :H]
    r = torch.randn(*shape, device="cuda").bfloat16()
    w, b = torch.randn(H, device="cuda").bfloat16(), torch.randn(H, device="cuda").bfloat16()
    calls = [lambda: rms_norm(x, w, 1e-5), lambda: rms_norm(x, w, 1e-5, r), lambda: layer_norm(x, w, b), lambda: layer_norm(x, w, None, 1e-6, r),
             lambda: gated_act(x, "silu"), lambda: gated_act(x, "gelu")]
    for f in calls:
        with torch.no_grad():
            a = f()
        b_ = f()
        for s, t in zip(*(v if isinstance(v, tuple) else (v,) for v in (a, b_))):
            assert torch.equal(s, t) and s.shape == t.shape and s.dtype == t.dtype

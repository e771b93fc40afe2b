"""Which calls the kernels behind ops/linear.py take: those that read tensors' memory and differentiate by no operator.
Everything else -- transformed or fake tensors, traces, forward-mode derivatives, trainable biases -- runs the library's product."""
import pytest
import torch
import torch.autograd.forward_ad as fwAD
import torch.nn.functional as F

gpu = pytest.mark.gpu


def _operands(rows, dtype=torch.bfloat16, device="cuda", N=64, K=128):
    g = torch.Generator(device).manual_seed(rows)
    return (torch.randn(rows, K, generator=g, device=device).to(dtype), (torch.randn(N, K, generator=g, device=device) / K ** 0.5).to(dtype),
            torch.randn(N, generator=g, device=device).to(dtype))


def _close(got, want):
    # both are fp32 sums of exact products, rounded once to bf16 (2^-9 each)
    assert got.dtype == want.dtype and got.shape == want.shape
    assert (got.double() - want.double()).norm() <= 6e-3 * want.double().norm()


def test_plain_tensors():
    """What ``native.plain`` lets through, on the CPU."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx

    from shuffle_exchange_amd.ops.native import plain
    x, w, b = _operands(5, torch.float32, "cpu")
    assert plain(x, torch.nn.Parameter(w), None) and plain(x[1:, ::2])
    seen = []

    def look(t):
        seen.append(plain(t))
        return t * 2
    torch.func.vmap(look)(x)
    torch.func.jvp(look, (x,), (x,))
    torch.func.grad(lambda t: look(t).sum())(x)
    torch.func.functionalize(look)(x)
    with fwAD.dual_level():
        look(fwAD.make_dual(x, x))
        assert not plain(x)  # another operand of the call may be dual
    with FakeTensorMode() as mode:
        look(mode.from_tensor(x))
    make_fx(look)(x)
    torch.jit.trace(look, (x,), check_trace=False)

    class Twice(torch.autograd.Function):
        @staticmethod
        def forward(ctx, t):
            return t * 2

        @staticmethod
        def backward(ctx, g):
            return look(g)
    t = x.clone().requires_grad_()
    torch.autograd.grad(Twice.apply(t), t, torch.ones(3, *x.shape), is_grads_batched=True)
    assert len(seen) >= 8 and not any(seen)
    assert plain(x)


@gpu
@pytest.mark.parametrize("rows", [1, 4, 5, 16, 17, 32, 33])
def test_forward_mode(rows):
    from shuffle_exchange_amd.ops.linear import linear
    x, w, b = _operands(rows)
    t = _operands(rows + 100)[0][:rows]
    want = F.linear(t, w)
    with torch.no_grad(), fwAD.dual_level():
        y = fwAD.unpack_dual(linear(fwAD.make_dual(x, t), w, b))
        assert y.tangent is not None
        _close(y.tangent, want)
        dw = fwAD.unpack_dual(linear(x, fwAD.make_dual(w, w), b)).tangent
        _close(dw, F.linear(x, w))
    _close(torch.func.jvp(lambda a: linear(a, w, b), (x,), (t,))[1], want)


@gpu
@pytest.mark.parametrize("rows", [2, 8, 24])
def test_vmap(rows):
    from shuffle_exchange_amd.ops.linear import linear
    x, w, b = _operands(3 * rows)
    with torch.no_grad():
        _close(torch.func.vmap(lambda a: linear(a, w, b))(x.view(3, rows, -1)), F.linear(x, w, b).view(3, rows, -1))


@gpu
@pytest.mark.parametrize("rows", [4, 8, 32])
def test_traces(rows):
    """A trace of few rows runs more, and a fake tensor has no memory to look at."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from shuffle_exchange_amd.ops.linear import linear
    x, w, b = _operands(rows)
    with torch.no_grad():
        traced = torch.jit.trace(lambda a: linear(a, w, b), (x,), check_trace=False)
        many = _operands(100)[0]
        _close(traced(many), F.linear(many, w, b))
        with FakeTensorMode(allow_non_fake_inputs=True) as mode:
            assert linear(mode.from_tensor(x), w, b).shape == (rows, 64)


@gpu
def test_column_sum_transforms():
    from shuffle_exchange_amd.ops.linear import column_sum
    x = torch.randn(3, 400, 72, device="cuda")
    f = lambda a: column_sum(a, a.dtype)  # noqa: E731
    # sums of 400 values in another order: 400 x 2^-24 x the sum of magnitudes (330) at most, a tenth of that allowed here
    torch.testing.assert_close(torch.func.vmap(f)(x), x.sum(1), rtol=1e-5, atol=1e-3)
    torch.testing.assert_close(torch.func.jvp(f, (x[0],), (x[1],))[1], x[1].sum(0), rtol=1e-5, atol=1e-3)


@gpu
@pytest.mark.parametrize("rows", [4, 8, 32, 40])
def test_trainable_bias_alone(rows):
    """Bias-only training: the first layer's input and weight want no gradient, its bias does."""
    from shuffle_exchange_amd.ops.linear import linear
    x, w, b = _operands(rows)
    b.requires_grad_()
    y = linear(x, w, b)
    assert y.requires_grad
    y.float().sum().backward()
    assert torch.equal(b.grad, torch.full_like(b, rows))


@gpu
@pytest.mark.parametrize("rows", [4, 8, 32, 40])
def test_bias_forms(rows):
    """What the library's product takes as a bias is taken at every row count, and a bias of another length is refused."""
    from shuffle_exchange_amd.ops.linear import linear
    x, w, b = _operands(rows)
    for bias in (b[:1], b.repeat(2)[::2].contiguous(), torch.stack([b, b], 1)[:, 0]):
        with torch.no_grad():
            _close(linear(x, w, bias), F.linear(x, w, bias))
    with pytest.raises(RuntimeError), torch.no_grad():
        linear(x, w, b[:7])


@gpu
def test_autocast_type():
    from shuffle_exchange_amd.ops.linear import linear
    for rows in (4, 8, 32, 40):
        x, w, b = _operands(rows)
        with torch.no_grad(), torch.autocast("cuda", torch.float16):
            assert linear(x, w, b).dtype == F.linear(x, w, b).dtype == torch.float16


@gpu
@pytest.mark.parametrize("rows", [4, 8, 32, 40])
def test_operands_on_one_device(rows):
    """A bias or scale in host memory is refused before any launch."""
    from shuffle_exchange_amd.ops.fp_quantizer import FP8Weight
    from shuffle_exchange_amd.ops.linear import linear
    x, w, b = _operands(rows)
    q = FP8Weight(w)
    with torch.no_grad():
        with pytest.raises(RuntimeError):
            linear(x, w, b.cpu())
        if rows <= 16:
            for scale, bias in ((q.scale.cpu(), b), (q.scale, b.cpu())):
                q.scale = scale
                with pytest.raises(RuntimeError, match="operand is on cpu"):
                    q.linear(x, bias)
                q.scale = scale.cuda()


@gpu
def test_library_switch(monkeypatch):
    """SXE_SKINNY_MAX_M = 0: no product of linear() or of the gated form leaves the library."""
    from shuffle_exchange_amd.ops import linear as L
    monkeypatch.setattr(L, "SKINNY_MAX_M", 0)
    for rows in (1, 8, 32):
        x, w, _ = _operands(rows)
        with torch.no_grad():
            assert L.glu_linear(x, w) is None and torch.equal(L.linear(x, w), F.linear(x, w))


@gpu
@pytest.mark.parametrize("rows", [1, 8, 32, 100])
def test_flops_are_counted(rows):
    from torch.utils.flop_counter import FlopCounterMode

    from shuffle_exchange_amd.ops.fp_quantizer import FP8Weight
    from shuffle_exchange_amd.ops.linear import glu_linear, linear
    from shuffle_exchange_amd.profiling.flops_profiler.profiler import _register_sxe_formulas
    _register_sxe_formulas()
    x, w, b = _operands(rows)
    for weight in (w, FP8Weight(w)) if rows <= 16 else (w,):
        with torch.no_grad(), FlopCounterMode(display=False) as c:
            linear(x, weight, b)
        assert c.get_total_flops() == 2 * rows * 64 * 128
    if rows <= 32:
        with torch.no_grad(), FlopCounterMode(display=False) as c:
            assert glu_linear(x, w) is not None
        assert c.get_total_flops() == 2 * rows * 64 * 128


@gpu
def test_flops_of_a_head_with_a_buffer():
    """A column-wise head's products, forward, dh and dW: the same count where dW goes into the optimizer's buffer."""
    from torch.utils.flop_counter import FlopCounterMode

    from shuffle_exchange_amd.ops.cross_entropy import head_cross_entropy
    from shuffle_exchange_amd.profiling.flops_profiler.profiler import _register_sxe_formulas
    _register_sxe_formulas()
    w = torch.nn.Parameter(torch.randn(515, 128, device="cuda").bfloat16())
    h, ids = torch.randn(2, 64, 128, device="cuda").bfloat16().requires_grad_(), torch.randint(0, 515, (2, 64), device="cuda")
    buf, done, counts = torch.zeros(515, 128, device="cuda"), [], []
    for _ in range(2):
        with FlopCounterMode(display=False) as c:
            head_cross_entropy(h, w, ids).backward()
        counts.append(c.get_total_flops())
        w.grad = None
        w._sxe_grad_target, w._sxe_grad_done, w._sxe_grad_local = (lambda p: (buf, False)), done.append, True
    assert done and counts == [3 * 2 * 128 * 515 * 128] * 2


@gpu
@pytest.mark.parametrize("tokens", [3, 200])
def test_flops_of_routed_experts(tokens):
    from torch.utils.flop_counter import FlopCounterMode

    from shuffle_exchange_amd.ops.moe import route_logits, swiglu_experts
    from shuffle_exchange_amd.profiling.flops_profiler.profiler import _register_sxe_formulas
    _register_sxe_formulas()
    x = torch.randn(tokens, 128, device="cuda").bfloat16()
    up, down = (torch.randn(4, *s, device="cuda").bfloat16() / 16 for s in ((128, 256), (128, 128)))
    routing = route_logits(torch.randn(tokens, 4, device="cuda"), 2)
    with torch.no_grad(), FlopCounterMode(display=False) as c:
        swiglu_experts(x, routing, up, down)
    assert c.get_total_flops() == 2 * 2 * tokens * (128 * 256 + 128 * 128)


def test_streaming_rule():
    """Which side of the measured lines a product falls on; no size is refused by the rule itself."""
    from shuffle_exchange_amd.ops.linear import _stream_faster, glu_faster
    for N, K in ((3072, 2048), (4096, 4096), (28672, 4096), (4096, 14336), (8, 4096), (2048, 5632), (15360, 5120)):
        assert _stream_faster(5, N, K) and _stream_faster(16, N, K)
    for N, K in ((5120, 5120), (5120, 13824), (10240, 8192), (50257, 768)):
        assert not _stream_faster(5, N, K) and not _stream_faster(16, N, K)
    for N, K in ((2048, 2048), (4096, 4096), (4100, 1032)):
        assert _stream_faster(17, N, K) and _stream_faster(32, N, K) and not _stream_faster(33, N, K)
    for N, K in ((5120, 3072), (6144, 4096), (1024, 8192), (11264, 2048)):
        assert not _stream_faster(17, N, K)
    w = lambda N, K: torch.empty(N, K, device="meta")  # noqa: E731
    assert all(glu_faster(16, w(*s)) and glu_faster(24, w(*s)) for s in ((16384, 2048), (16384, 3072), (28672, 4096), (0, 8)))
    assert all(glu_faster(16, w(*s)) and not glu_faster(24, w(*s)) for s in ((17920, 2560), (27648, 5120), (7168, 4096)))
    assert not glu_faster(5, w(57344, 8192)) and glu_faster(16, object())


@gpu
@pytest.mark.parametrize("R,N,kernel", [(255, 768, False), (256, 768, True), (4096, 8192, True), (8192, 8192, True), (8192, 8200, False),
                                        (8191, 8200, True), (4095, 1001, False), (4096, 1001, True), (4096, 63, False), (256, 65544, False)])
def test_column_sum_rule(R, N, kernel):
    from shuffle_exchange_amd.ops import linear as L
    x = torch.randn(R, N, device="cuda").bfloat16()
    assert L._colsum_faster(x) == kernel
    want, size = x.double().sum(0), x.double().abs().sum(0)
    for dtype in (torch.bfloat16, torch.float32):
        got = L.column_sum(x, dtype)
        # fp32 sums of at most R / 128 + 14 steps a column (the general reduction has no more), and the rounding of the result
        assert got.dtype == dtype and ((got.double() - want).abs() <= (R / 128 + 14) * 2 ** -24 * size
                                       + (2 ** -8 if dtype == torch.bfloat16 else 0) * want.abs() + 1e-30).all()


@pytest.mark.parametrize("T,M,N,own", [(256, 57344, 8192, False), (512, 57344, 8192, True), (128, 16384, 8192, False), (256, 8192, 8192, True),
                                       (128, 128256, 4096, True), (64, 28672, 4096, True)])
def test_weight_gradient_rule(T, M, N, own):
    """Few tokens of the largest weights whose rows lie 32 KB apart are the library's."""
    from shuffle_exchange_amd.ops.linear import _wgrad_faster
    assert _wgrad_faster(T, M, N) == own


@pytest.mark.parametrize("rows,N,K,own", [(1499, 4096, 4096, False), (1501, 4096, 4096, True), (1536, 4096, 4096, False), (12999, 3072, 8192, True),
                                          (13001, 3072, 8192, False), (31000, 4096, 4096, False), (600, 4096, 14336, True), (33, 8192, 8192, False),
                                          (200, 8192, 8192, True), (33, 2048, 8192, True), (100, 2048, 8192, False), (64, 6144, 16384, False),
                                          (200, 6144, 16384, True), (100, 8192, 28672, True), (600, 2040, 8192, False)])
def test_many_row_rule(rows, N, K, own):
    from shuffle_exchange_amd.ops.linear import _tiled_faster
    assert _tiled_faster(rows, N, K) == own


@pytest.mark.parametrize("rows,N,K,own", [(255, 28672, 4096, False), (256, 28672, 4096, True), (1280, 28672, 4096, True), (1371, 28672, 4096, False),
                                          (1819, 16384, 2048, True), (1962, 28672, 3072, False), (512, 16384, 4096, False), (256, 57344, 8192, False),
                                          (400, 128256, 4096, False), (640, 57344, 4096, False), (1000, 27648, 5120, True), (1792, 16384, 2048, False)])
def test_transposed_weight_rule(rows, N, K, own):
    from shuffle_exchange_amd.ops.linear import _wt_few_faster
    assert _wt_few_faster(rows, N, K) == own


@gpu
def test_data_gradient_of_few_rows(monkeypatch):
    """The weight is transposed only for the own product: not where a graph is recorded (the transpose has no derivative), nor where the
    library's products are asked for."""
    from shuffle_exchange_amd.ops import linear as L, native
    native.require_hip()
    g = torch.Generator("cuda").manual_seed(2)
    w = (torch.randn(16384, 2048, generator=g, device="cuda") / 128).bfloat16()
    gy = torch.randn(300, 16384, generator=g, device="cuda").bfloat16()
    seen = []
    transposed = L._transposed_weight
    monkeypatch.setattr(L, "_transposed_weight", lambda t: seen.append(1) or transposed(t))
    want = gy.double() @ w.double()
    with torch.no_grad():
        dx = L.data_grad(gy, w)
        assert seen == [1] and (dx.double() - want).norm() <= 6e-3 * want.norm()
        assert torch.equal(L.data_grad(F.pad(gy, (0, 4))[:, :16384], w), gy @ w) and seen == [1]  # rows off 16 bytes
    wg = w.clone().requires_grad_()
    with torch.enable_grad():
        dx = L.data_grad(gy, wg)
        dw, = torch.autograd.grad(dx, wg, torch.ones_like(dx))
    assert seen == [1] and (dw.double() - (gy.double().t() @ torch.ones_like(dx).double())).norm() <= 6e-3 * dw.double().norm()
    monkeypatch.setattr(L, "SKINNY_MAX_M", 0)
    with torch.no_grad():
        assert torch.equal(L.data_grad(gy, w), gy @ w) and seen == [1]


@pytest.mark.parametrize("rows,N,K", [(512, 2048, 512), (2048, 1024, 2816), (300, 2304, 768), (300, 16384, 2048)])
def test_products_of_training_compile(rows, N, K):
    """No question that compilation cannot answer (where an operand lies) is on the way of a product or its data gradient: without a
    GPU, on fake tensors of one."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from shuffle_exchange_amd.ops.linear import data_grad, product

    class Product(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x, w):
            ctx.save_for_backward(x, w)
            return product(x, w)

        @staticmethod
        def backward(ctx, gy):
            x, w = ctx.saved_tensors
            return data_grad(gy, w), gy.t() @ x
    torch._dynamo.reset()
    with FakeTensorMode():
        x, w = (torch.empty(n, K, device="cuda", dtype=torch.bfloat16, requires_grad=True) for n in (rows, N))
        y = torch.compile(Product.apply, fullgraph=True, backend=lambda graph, inputs: graph)(x, w)
    assert y.shape == (rows, N)


def test_optimizers_buffer_is_for_backward():
    """``local_grad_target``: where the backward adds a parameter's gradient up, not where its caller asks for it or for others."""
    from shuffle_exchange_amd.ops.linear import keep_local, local_grad_target
    p, q, buf, seen = torch.nn.Parameter(torch.ones(3)), torch.nn.Parameter(torch.ones(3)), torch.zeros(3), []
    p._sxe_grad_target, p._sxe_grad_local = (lambda t: (buf, False)), True
    assert keep_local(q) is None

    class Scale(torch.autograd.Function):
        @staticmethod
        def forward(ctx, number, x, w):
            ctx.w = keep_local(w)
            return number * x * w

        @staticmethod
        def backward(ctx, gy):
            seen.append(local_grad_target(ctx.w, ctx) is not None)
            return None, gy, gy
    run = lambda: Scale.apply(1.0, q * 2, p).sum()  # noqa: E731
    run().backward()
    run().backward(inputs=[q])
    torch.autograd.grad(run(), [p])
    torch.autograd.grad(run(), [q])
    assert seen == [True, False, False, False]
    p.grad = None
    run().backward(inputs=[p])
    assert seen[4]


@gpu
def test_narrow_products_of_a_captured_step(monkeypatch):
    """Own kernels for what the host would wait for; in a captured graph, where it waits for nothing, the library's."""
    from shuffle_exchange_amd.ops import linear as L
    x, w, b = _operands(300, N=768, K=512)
    wide = _operands(300, N=2048, K=8192)  # the own product's on the device, too
    gy, took = F.linear(x, w), []
    for name in ("_tiled", "_narrow_data_grad"):
        monkeypatch.setattr(L, name, lambda *a, own=getattr(L, name): took.append(own(*a)) or took[-1])

    def run():
        took.clear()
        return [L.product(x, w, b), L.data_grad(gy, w), L.product(*wide[:2])], [t is not None for t in took]
    with torch.no_grad():
        want, own = run()
        assert own == [True, True, True]
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got, own = run()
        assert own == [False, True]  # the data gradient's and the wide product
        for _ in range(3):
            for t in got:
                t.zero_()
            graph.replay()
            torch.cuda.synchronize()
            for t, o in zip(got, want):
                _close(t, o)


@gpu
@pytest.mark.parametrize("R,N,kernel", [(128, 768, True), (64, 50257, True), (2048, 3072, True), (1000, 50257, False), (16, 524288, False)])
def test_bias_gradient_rule(R, N, kernel):
    """Into the optimizer's buffer by the kernel where that is the faster way; else autograd gets the general reduction's sums."""
    from shuffle_exchange_amd.ops.linear import _Linear
    x, w, b = torch.zeros(R, 8, device="cuda").bfloat16(), torch.zeros(N, 8, device="cuda").bfloat16(), torch.nn.Parameter(torch.zeros(N, device="cuda").bfloat16())
    buf, done = torch.zeros(N, device="cuda"), []
    b._sxe_grad_target, b._sxe_grad_done, b._sxe_grad_local = (lambda p: (buf, False)), done.append, True
    _Linear.apply(x, w, b).backward(torch.ones(R, N, device="cuda").bfloat16())
    got = buf if kernel else b.grad.float()
    assert bool(done) == kernel and (b.grad is None) == kernel and torch.equal(got, torch.full_like(buf, R).bfloat16().float())


@gpu
def test_glu_rule_and_switch(monkeypatch):
    """SwiGLU of many rows in the product's launch, not of few rows of the largest weights, nor where the library's products are asked for."""
    from shuffle_exchange_amd.ops import linear as L
    w = torch.zeros(8192, 2048, device="cuda", dtype=torch.bfloat16)
    x = torch.zeros(301, 2048, device="cuda", dtype=torch.bfloat16)
    large = torch.empty(1, 8192, device="cuda", dtype=torch.bfloat16).expand(32776, 8192)  # never read
    xl = torch.zeros(1024, 8192, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        assert L.glu_tiled(x, w) is not None and L.glu_tiled(x[:300], w) is None and L.glu_tiled(xl, large) is None
        monkeypatch.setattr(L, "SKINNY_MAX_M", 0)
        assert L.glu_tiled(x, w) is None


@pytest.mark.parametrize("rows,N,K,own", [(17, 32000, 4096, True), (32, 16384, 4096, True), (24, 8192, 4096, False), (24, 8192, 3072, True),
                                          (24, 9216, 3072, False), (33, 32000, 4096, False), (24, 32000, 4104, False)])
def test_few_row_rule_of_wide_weights(rows, N, K, own):
    from shuffle_exchange_amd.ops.linear import _stream_faster
    assert _stream_faster(rows, N, K) == own


@pytest.mark.parametrize("rows,N,K,own", [(17, 4096, 14336, False), (24, 4096, 14336, True), (32, 8192, 28672, True), (24, 4096, 11008, True),
                                          (24, 4096, 24576, True), (17, 8192, 5120, False), (17, 8192, 5632, True),
                                          (24, 4096, 16384, False), (24, 4096, 8192, False), (33, 4096, 14336, False), (24, 3840, 15360, False),
                                          (24, 5120, 13824, False), (24, 2048, 22016, False), (24, 12288, 12288, False)])
def test_few_row_rule_of_long_rows(rows, N, K, own):
    from shuffle_exchange_amd.ops.linear import _stream_faster
    assert _stream_faster(rows, N, K) == own

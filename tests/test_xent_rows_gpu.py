"""Cross-entropy rows that start off a 16-byte boundary (csrc/kernels/xent.hip) against fp64: odd vocabularies, short rows, masked
logits, ignored targets, gradients in place and beside, operands that start differently."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _native():
    from shuffle_exchange_amd.ops import native
    native.require_hip()


@pytest.mark.parametrize("V", [1, 5, 8, 9, 31, 511, 513, 2049, 4096, 4100, 50257])
@pytest.mark.parametrize("offset", [0, 3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_rows(V, offset, dtype):
    R = 9
    g = torch.Generator(device="cuda").manual_seed(V + offset)
    flat = torch.randn(R * V + offset, generator=g, device="cuda") * 3
    flat = flat.to(dtype)
    logits = flat[offset:].view(R, V)
    if V > 16:
        logits[1, V // 2:] = float("-inf")  # a masked half, whole groups of eight among it
        logits[2, :V - 1] = torch.finfo(dtype).min
    tgt = torch.randint(0, max(1, V // 2), (R,), generator=g, device="cuda")
    tgt[2], tgt[4] = V - 1, -100
    ref = logits.double()
    lse = ref.logsumexp(-1)
    want = torch.where(tgt == -100, 0., lse - ref.gather(1, tgt.clamp_min(0)[:, None])[:, 0])
    one = torch.nn.functional.one_hot(tgt.clamp_min(0), V)
    dl = torch.rand(R, generator=g, device="cuda")
    grad = torch.where((tgt == -100)[:, None], 0., dl.double()[:, None] * ((ref - lse[:, None]).exp() - one))
    eps = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -10, torch.float32: 1e-5}[dtype]
    tol = dict(rtol=eps, atol=2e-6)  # a rounding of the result; fp32 sums and the device's exp and log (about 2^-21)

    keep = logits.clone()
    loss, got_lse = torch.ops.sxe.xent_fwd(logits, tgt, -100, False, None, 1.0)
    torch.testing.assert_close(got_lse.double(), lse, rtol=2e-6, atol=4e-6)
    torch.testing.assert_close(loss.double(), want, rtol=2e-6, atol=2e-5)
    beside = torch.ops.sxe.xent_bwd(logits, tgt, got_lse, dl, -100, False)
    assert torch.equal(logits, keep)
    torch.testing.assert_close(beside.double(), grad, **tol)
    torch.ops.sxe.xent_bwd(logits, tgt, got_lse, dl, -100, True)
    torch.testing.assert_close(logits.double(), grad, **tol)
    torch.ops.sxe.xent_fwd(keep, tgt, -100, True, None, 0.25)
    full = torch.where((tgt == -100)[:, None], 0., 0.25 * ((ref - lse[:, None]).exp() - one))
    torch.testing.assert_close(keep.double(), full, **tol)


@pytest.mark.parametrize("tokens", [1, 63, 64, 130, 500, 2100])  # columns behind the last token, of a block, blocks of each width
@pytest.mark.parametrize("V", [65, 129, 1001, 9999])        # one share and several, rounds of 64 rows and their rest
def test_column_head_matches_fp64(V, tokens):
    """The head with a token per column. A logit (|x| < 6) is rounded to bf16, and with it the loss moves by 2 * 6 * 2^-8 at most. A
    probability moves by 2^-8 |x|, in a norm by less than 2 * 2^-8; the gradient is rounded and so is the product of it: 2^-8 (2 + 2)."""
    from shuffle_exchange_amd.ops.cross_entropy import head_cross_entropy, _columns_ok
    g = torch.Generator("cuda").manual_seed(V + tokens)
    h = torch.randn(1, tokens, 64, generator=g, device="cuda").bfloat16().requires_grad_()
    w = torch.randn(V, 64, generator=g, device="cuda").mul_(0.125).bfloat16().requires_grad_()
    tgt = torch.randint(0, V, (1, tokens), generator=g, device="cuda")
    tgt[0, tokens // 2 + 1:tokens // 2 + 3] = -100
    assert _columns_ok(h, w, tgt)
    loss = head_cross_entropy(h, w, tgt)
    h2, w2 = h.detach().double().requires_grad_(), w.detach().double().requires_grad_()
    want = torch.nn.functional.cross_entropy((h2 @ w2.t())[0], tgt[0])
    (0.5 * loss).backward()
    (0.5 * want).backward()
    assert abs(loss.item() - want.item()) < 12 * 2 ** -8
    for a, b in ((h.grad, h2.grad), (w.grad, w2.grad)):
        assert (a.double() - b).norm() <= 2 ** -6 * b.norm()


@pytest.mark.parametrize("tokens", [64, 65])  # as they are, rounded up
def test_column_head_of_unaligned_states(tokens):
    """Hidden states that start off 16 bytes give what their copy gives."""
    from shuffle_exchange_amd.ops.cross_entropy import head_cross_entropy, _columns_ok
    g = torch.Generator("cuda").manual_seed(tokens)
    w = torch.randn(1001, 128, generator=g, device="cuda").mul_(0.1).bfloat16().requires_grad_()
    tgt = torch.randint(0, 1001, (1, tokens), generator=g, device="cuda")
    flat = torch.randn(tokens * 128 + 1, generator=g, device="cuda").bfloat16()
    got = []
    for h in (flat[1:].view(1, tokens, 128), flat[1:].clone().view(1, tokens, 128)):
        h.requires_grad_()
        assert _columns_ok(h, w, tgt)
        loss = head_cross_entropy(h, w, tgt)
        got.append((loss.detach(), *torch.autograd.grad(loss, (h, w))))
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("tokens", [64, 70])
def test_column_head_gradients_of_gradients(tokens):
    """What a recorded backward gives, and its derivatives with respect to the head's two operands (the softmax's own derivative is not
    among them, as over a token per row): as the product and the row form give them, up to the roundings of logits and gradients
    (see above: 2^-6 of the norm)."""
    from shuffle_exchange_amd.ops.cross_entropy import cross_entropy, head_cross_entropy, _columns_ok
    g = torch.Generator("cuda").manual_seed(tokens)
    h = torch.randn(1, tokens, 64, generator=g, device="cuda").bfloat16().requires_grad_()
    w = torch.randn(1001, 64, generator=g, device="cuda").mul_(0.125).bfloat16().requires_grad_()
    tgt = torch.randint(0, 1001, (1, tokens), generator=g, device="cuda")
    vh, vw = torch.randn_like(h), torch.randn_like(w)
    assert _columns_ok(h, w, tgt)
    got = []
    for loss in (head_cross_entropy(h, w, tgt), cross_entropy(torch.nn.functional.linear(h, w), tgt)):
        dh, dw = torch.autograd.grad(loss, (h, w), create_graph=True)
        got.append((dh.detach(), dw.detach(), torch.autograd.grad(dh, w, vh, retain_graph=True)[0], torch.autograd.grad(dw, h, vw)[0]))
    for a, b in zip(*got):
        assert (a.double() - b.double()).norm() <= 2 ** -6 * b.double().norm()


def test_column_head_masked_vocabulary():
    """Rows of -inf logits (a hidden state of infinities) and a share with nothing else: NaN and zeros where the row form has them."""
    x = torch.randn(200, 64, device="cuda").bfloat16()
    x[:120] = float("-inf")
    x[:, 3] = float("nan")
    tgt = torch.full((64,), 150, device="cuda")
    loss, lse = torch.ops.sxe.xent_cols_fwd(x, tgt, -100)
    rows, rlse = torch.ops.sxe.xent_fwd(x.t().contiguous(), tgt, -100, False, None, 1.0)
    torch.testing.assert_close(loss, rows, equal_nan=True, rtol=1e-5, atol=1e-5)  # sums of 200 terms in another order: 200 * 2^-24
    torch.testing.assert_close(lse, rlse, equal_nan=True, rtol=1e-5, atol=1e-5)
    dl = torch.ones(64, device="cuda")
    got = torch.ops.sxe.xent_cols_bwd(x, tgt, rlse, dl, -100)
    want = torch.ops.sxe.xent_bwd(x.t().contiguous(), tgt, rlse, dl, -100, False).t()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())

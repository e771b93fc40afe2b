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

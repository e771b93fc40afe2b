"""Column sums (csrc/kernels/colsum.hip, sxe_colsum.h) against fp64: remainders of rows and columns, both sides of the split, strided and
expanded rows, every type; and their users' gradients."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _native():
    from shuffle_exchange_amd.ops import native
    native.require_hip()


@pytest.mark.parametrize("R", [1, 127, 513, 2048, 2049, 5000])
@pytest.mark.parametrize("N", [1, 8, 63, 72, 2304])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_column_sum(R, N, dtype):
    g = torch.Generator(device="cuda").manual_seed(R + N)
    base = torch.randn(R, N + 16, generator=g, device="cuda").to(dtype)
    for x in (base[:, :N], base[:, 8:N + 8], base[:, 1:N + 1], base[:, :N].contiguous(), base[:1, :N].expand(R, N)):
        want, size = x.double().sum(0), x.double().abs().sum(0)
        for out in (dtype, torch.float32):
            y = torch.ops.sxe.column_sum(x, out)
            # fp32 sums over at most R / 128 + 14 steps a column, and the rounding of the result
            eps = (R / 128 + 14) * 2 ** -24
            rnd = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11, torch.float32: 0}[out]
            assert y.shape == (N,) and y.dtype == out
            assert ((y.double() - want).abs() <= eps * size + rnd * want.abs() + 1e-30).all()


def test_empty_and_nonfinite():
    assert torch.equal(torch.ops.sxe.column_sum(torch.empty(0, 5, device="cuda"), torch.float32), torch.zeros(5, device="cuda"))
    assert torch.ops.sxe.column_sum(torch.empty(4, 0, device="cuda"), torch.float32).shape == (0,)
    x = torch.ones(300, 16, device="cuda")
    x[7, 3], x[8, 4], x[9, 4] = float("nan"), float("inf"), float("-inf")
    y = torch.ops.sxe.column_sum(x, torch.float32)
    assert y[3].isnan() and y[4].isnan() and torch.equal(y[5:], torch.full((11,), 300., device="cuda"))


@pytest.mark.parametrize("rows,H", [(3, 768), (2500, 776), (130, 104)])
def test_users(rows, H):
    """The norm's and the biased activation's backward against autograd in fp64 of the same bf16 operands."""
    from shuffle_exchange_amd.ops.activation import bias_gelu
    from shuffle_exchange_amd.ops.norm import layer_norm
    x, dy = torch.randn(2, rows, H, device="cuda").bfloat16()
    w, b = (1 + 0.1 * torch.randn(2, H, device="cuda")).bfloat16()

    def grads(f, dt):
        leaves = [t.to(dt, copy=True).requires_grad_() for t in (x, w, b)]
        f(*leaves).backward(dy.to(dt))
        return [t.grad.double() for t in leaves if t.grad is not None]
    ln = zip(grads(lambda x, w, b: layer_norm(x, w, b), torch.bfloat16),
             grads(lambda x, w, b: torch.nn.functional.layer_norm(x, (H,), w, b), torch.float64))
    ge = zip(grads(lambda x, w, b: bias_gelu(x, b), torch.bfloat16),
             grads(lambda x, w, b: torch.nn.functional.gelu(x + b, approximate="tanh"), torch.float64))
    for got, want in (*ln, *ge):
        assert (got - want).norm() < 6e-3 * want.norm()  # roundings of bf16 terms and results: 2^-8 each at most


def test_traces():
    """The op has a shape function like the other kernels of a training step."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    import shuffle_exchange_amd.ops.fake_kernels  # noqa: F401
    with FakeTensorMode() as mode:
        x = mode.from_tensor(torch.empty(12, 40, device="cuda", dtype=torch.bfloat16))
        y = torch.ops.sxe.column_sum(x, torch.float32)
        assert y.shape == (40,) and y.dtype == torch.float32 and y.device == x.device

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


@pytest.mark.parametrize("M", [1, 5, 15, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(4, 16), (20, 1024), (6144, 96), (6148, 4112), (128, 2064), (8192, 2048)])
@pytest.mark.parametrize("fp8", [False, True])
def test_plain(M, N, K, fp8):
    x, w, s, ref = _operands(M, N, K, fp8, M + N + K)
    b = torch.randn(N, device="cuda").bfloat16()
    for bias in (None, b):
        got = torch.ops.sxe.stream_gemm(x, w, s, bias, False)
        want = x.double() @ ref.T + (0 if bias is None else b.double())
        # products of bf16 are exact in fp32; left are fp32 sums and the rounding of the result: at most 2^-8 of a value (just above a power
        # of two), which a result of four values with a bias drawn anew each time comes near
        assert (got.double() - want).norm() < 1.01 * 2 ** -8 * want.norm()


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

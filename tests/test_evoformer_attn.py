"""DS4Sci_EvoformerAttention vs the plain formula (fp32, CPU), values and all five gradients."""
import pytest
import torch

from shuffle_exchange_amd.ops.deepspeed4science import DS4Sci_EvoformerAttention
from shuffle_exchange_amd.ops.deepspeed4science import evoformer_attn as ea


def test_evoformer_matches_formula_with_grads(monkeypatch):
    monkeypatch.setattr(ea, "CHUNK", 8)
    torch.manual_seed(0)
    B, N, L, H, D = 1, 3, 20, 2, 16
    Q, K, V = (torch.randn(B, N, L, H, D, requires_grad=True) for _ in range(3))
    b1 = torch.randn(B, N, 1, 1, L, requires_grad=True)
    b2 = torch.randn(B, 1, H, L, L, requires_grad=True)
    out = ea.evoformer_attention(Q, K, V, b1, b2, chunk=8)
    s = torch.einsum("bnqhd,bnkhd->bnhqk", Q, K) / D ** 0.5 + b1 + b2
    ref = torch.einsum("bnhqk,bnkhd->bnqhd", torch.softmax(s, -1), V)
    torch.testing.assert_close(out, ref, atol=1e-5, rtol=1e-5)
    g = torch.randn_like(out)
    got = torch.autograd.grad(out, (Q, K, V, b1, b2), g)
    exp = torch.autograd.grad(ref, (Q, K, V, b1, b2), g)
    for a, b in zip(got, exp):
        torch.testing.assert_close(a, b, atol=1e-5, rtol=1e-4)
    o2 = DS4Sci_EvoformerAttention(Q, K, V, [b1, b2])
    torch.testing.assert_close(o2, ref, atol=1e-5, rtol=1e-5)
    o3 = DS4Sci_EvoformerAttention(Q, K, V, [])
    s3 = torch.einsum("bnqhd,bnkhd->bnhqk", Q, K) / D ** 0.5
    torch.testing.assert_close(o3, torch.einsum("bnhqk,bnkhd->bnqhd", torch.softmax(s3, -1), V), atol=1e-5,
                               rtol=1e-5)


def _formula(Q, K, V, b1, b2):
    D = Q.shape[-1]
    q, k, v = (t.float().transpose(-2, -3) for t in (Q, K, V))  # [B, N, H, L, D]
    s = q @ k.transpose(-1, -2) / D ** 0.5 + b1.float() + b2.float()
    return (torch.softmax(s, -1) @ v).transpose(-2, -3)


@pytest.mark.gpu
@pytest.mark.parametrize("D,L", [(32, 70), (64, 133), (64, 256)])
def test_evoformer_hip_kernels_vs_fp32(D, L):
    """Fused HIP forward / backward (evoformer.hip) vs the fp32 formula: output, dQ, dK, dV, dbias1,
    dbias2, for sequence lengths that are not tile multiples."""
    from shuffle_exchange_amd.ops import native
    native.require_hip()
    torch.manual_seed(0)
    B, N, H = 2, 3, 2
    mk = lambda *s: torch.randn(*s, device="cuda")
    Q, K, V = (mk(B, N, L, H, D).bfloat16().requires_grad_(True) for _ in range(3))
    b1 = (mk(B, N, 1, 1, L) * 2).bfloat16().requires_grad_(True)
    b2 = mk(B, 1, H, L, L).bfloat16().requires_grad_(True)
    assert ea._hip_ok(Q, K, V)
    out = DS4Sci_EvoformerAttention(Q, K, V, [b1, b2])
    g = mk(*out.shape).bfloat16()
    grads = torch.autograd.grad(out, (Q, K, V, b1, b2), g)
    ref_in = [t.detach().float().requires_grad_(True) for t in (Q, K, V, b1, b2)]
    ref = _formula(*ref_in)
    rgrads = torch.autograd.grad(ref, ref_in, g.float())
    assert (out.float() - ref).abs().max().item() < 2e-2
    for name, a, b in zip("QKV12", grads, rgrads):
        err = ((a.float() - b).norm() / b.norm()).item()
        assert err < 2e-2, (name, err)


@pytest.mark.gpu
@pytest.mark.parametrize("B,N,L,H,D", [(1, 1, 1, 1, 32), (1, 17, 31, 3, 32), (1, 9, 64, 4, 64), (2, 33, 129, 2, 32), (1, 5, 200, 8, 32),
                                       (1, 70, 128, 1, 64)])
@pytest.mark.parametrize("bias", ["bf16", "fp32", "mask", "pair", "none"])
def test_evoformer_tiles_and_biases(B, N, L, H, D, bias):
    """Tile edges, a single key, more rows than one part of dbias2, every bias form; masked keys (-inf, the type's lowest
    value, -1e9) and a row without any key left."""
    torch.manual_seed(1)
    mk = lambda *s: torch.randn(*s, device="cuda")
    Q, K, V, g = (mk(B, N, L, H, D).bfloat16() for _ in range(4))
    dt = torch.float32 if bias == "fp32" else torch.bfloat16
    b1 = b2 = None
    if bias in ("bf16", "fp32", "mask"):
        b1 = mk(B, N, 1, 1, L)
        b1[mk(B, N, 1, 1, L) > 1.5] = -1e9
        b1[mk(B, N, 1, 1, L) > 2] = float("-inf")
        b1[mk(B, N, 1, 1, L) > 2] = torch.finfo(torch.float32).min
        b1[..., 0] = 0.5
        b1[0, N - 1] = float("-inf")
        b1 = b1.to(dt)
    if bias in ("bf16", "fp32", "pair"):
        b2 = (mk(B, 1, H, L, L) * 2).to(dt)
    base = torch.empty(Q.numel() + 1, dtype=torch.bfloat16, device="cuda")  # a q that starts 2 bytes behind an aligned address
    q = base[1:].view(Q.shape).copy_(Q)
    ins = [t.requires_grad_(True) if t is not None else None for t in (q.detach(), K, V, b1, b2)]
    out = ea.evoformer_attention(*ins)
    live = [t for t in ins if t is not None]
    grads = torch.autograd.grad(out, live, g)
    ref = [t.detach().double().requires_grad_(True) if t is not None else None for t in ins]
    r = [t.transpose(-2, -3) for t in ref[:3]]
    s = r[0] @ r[1].transpose(-1, -2) / D ** 0.5
    for t in ref[3:]:
        s = s if t is None else s + t
    p = torch.softmax(s, -1)
    want = (torch.where(torch.isnan(p), torch.zeros_like(p), p) @ r[2]).transpose(-2, -3)
    keep = torch.ones(B, N, 1, 1, 1, device="cuda", dtype=torch.bool)
    if b1 is not None:
        keep[0, N - 1] = False  # no key left: the output is zero and nothing flows back
        assert out[0, N - 1].abs().max() == 0 and all(not t[0, N - 1].any() for t in grads[:3])
    s2 = s.masked_fill(~keep, 0.0)  # the reference's own gradient of that row is nan: leave the row out of it
    want_live = ((torch.softmax(s2, -1) * keep) @ r[2]).transpose(-2, -3)
    rg = torch.autograd.grad(want_live, [t for t in ref if t is not None], g.double())
    # p, ds and the results are rounded to 8 bits (2^-9 each, relative to their largest): 4 x 2^-9. A single key has dS = 0
    # exactly; what is left of it is the rounding of o in delta, at most 2^-9 sum |do o| a row
    slack = 2 ** -9 * (g.abs() * out.abs()).double().sum(-1).norm().item() * D ** 0.5 * (L == 1)
    assert (out.double() - want).norm() <= 8e-3 * want.norm() + 1e-6
    for a, b in zip(grads, rg):
        assert a.dtype == (dt if a.shape != Q.shape else torch.bfloat16)
        assert torch.isfinite(a).all() and (a.double() - b).norm() <= 8e-3 * b.norm() + slack, a.shape


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_evoformer_biases_reused_before_backward(dtype):
    """A program may write the next crop's mask and pair bias into the same buffers before this crop's backward."""
    torch.manual_seed(2)
    mk = lambda *s: torch.randn(*s, device="cuda")
    Q, K, V, g = (mk(1, 5, 70, 2, 32).bfloat16() for _ in range(4))
    b1, b2 = mk(1, 5, 1, 1, 70).to(dtype), mk(1, 1, 2, 70, 70).to(dtype)

    def grads(change):
        ins = [t.detach().clone().requires_grad_(True) for t in (Q, K, V)]
        m, p = b1.clone(), b2.clone()
        out = ea.evoformer_attention(*ins, m, p)
        if change:
            m.fill_(float("nan"))
            p.fill_(float("nan"))
        return torch.autograd.grad(out, ins, g)
    for a, b in zip(grads(True), grads(False)):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_evoformer_without_gradients():
    """The call that no backward follows gives the same bits, and a dual tensor's tangent is not dropped without a word."""
    import torch.autograd.forward_ad as fwAD
    torch.manual_seed(3)
    Q, K, V = (torch.randn(1, 5, 70, 2, 32, device="cuda").bfloat16() for _ in range(3))
    b1, b2 = torch.randn(1, 5, 1, 1, 70, device="cuda"), torch.randn(1, 1, 2, 70, 70, device="cuda").bfloat16().requires_grad_()
    want = ea.evoformer_attention(Q, K, V, b1, b2)
    with torch.no_grad():
        assert torch.equal(ea.evoformer_attention(Q, K, V, b1, b2), want)
    assert want.requires_grad and not ea.evoformer_attention(Q, K, V, b1).requires_grad
    with fwAD.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        ea.evoformer_attention(fwAD.make_dual(Q, torch.ones_like(Q)), K, V, b1, None)


@pytest.mark.gpu
@pytest.mark.parametrize("D,L", [(32, 127), (32, 128), (32, 129), (32, 256), (32, 257), (32, 383), (32, 384), (32, 385), (64, 65), (64, 257)])
@pytest.mark.parametrize("N", [1, 2, 7])
def test_evoformer_key_blocks(D, L, N):
    """Edges of the key blocks that dQ and the pair bias' gradient share, odd and even numbers of rows, and a row whose keys are all
    masked by the same finite number: its softmax is that of the other terms."""
    torch.manual_seed(4)
    B, H = 2, 3
    mk = lambda *s: torch.randn(*s, device="cuda")
    Q, K, V, g = (mk(B, N, L, H, D).bfloat16() for _ in range(4))
    b1 = (mk(B, N, 1, 1, L) > 1).float() * -1e9
    b1[..., 0] = 0
    b1[1, N - 1] = -1e9
    ins = [t.requires_grad_(True) for t in (Q, K, V, b1, (mk(B, 1, H, L, L) * 2).bfloat16())]
    out = ea.evoformer_attention(*ins)
    grads = torch.autograd.grad(out, ins, g)
    ref = [t.detach().double().requires_grad_(True) for t in ins]
    q, k, v = (t.transpose(-2, -3) for t in ref[:3])
    want = (torch.softmax(q @ k.transpose(-1, -2) / D ** 0.5 + ref[3] + ref[4], -1) @ v).transpose(-2, -3)
    # as above: p, ds and the results are rounded to 8 bits, 4 x 2^-9
    assert (out.double() - want).norm() <= 8e-3 * want.norm()
    for a, b in zip(grads, torch.autograd.grad(want, ref, g.double())):
        assert torch.isfinite(a).all() and (a.double() - b).norm() <= 8e-3 * b.norm(), a.shape


@pytest.mark.gpu
@pytest.mark.parametrize("D,N,L", [(32, 191, 40), (32, 193, 40), (64, 191, 40), (64, 193, 40), (64, 447, 40), (64, 449, 40), (32, 49, 400)])
@pytest.mark.parametrize("pair", [torch.bfloat16, torch.float32, None])
def test_evoformer_rows_of_a_workgroup(D, N, L, pair):
    """Both sides of the grids from which on a workgroup takes two of the N rows, with a last workgroup of one."""
    torch.manual_seed(6)
    H = 8
    mk = lambda *s: torch.randn(*s, device="cuda")
    ins = [mk(1, N, L, H, D).bfloat16() for _ in range(3)] + [(mk(1, N, 1, 1, L) > 1).float() * -30.0]
    g = mk(1, N, L, H, D).bfloat16()
    ins = [t.requires_grad_(True) for t in ins + ([(mk(1, 1, H, L, L) * 2).to(pair)] if pair else [])]
    out = ea.evoformer_attention(*ins)
    grads = torch.autograd.grad(out, ins, g)
    ref = [t.detach().double().requires_grad_(True) for t in ins]
    q, k, v = (t.transpose(-2, -3) for t in ref[:3])
    want = (torch.softmax(sum(ref[4:], q @ k.transpose(-1, -2).contiguous() / D ** 0.5 + ref[3]), -1) @ v).transpose(-2, -3)
    # as above: p, ds and the results are rounded to 8 bits, 4 x 2^-9
    assert (out.double() - want).norm() <= 8e-3 * want.norm()
    for a, b in zip(grads, torch.autograd.grad(want, ref, g.double())):
        assert torch.isfinite(a).all() and (a.double() - b).norm() <= 8e-3 * b.norm(), a.shape


@pytest.mark.gpu
@pytest.mark.parametrize("D,N,L", [(32, 5, 70), (32, 5, 257), (32, 5, 400), (32, 200, 40), (64, 5, 133), (64, 400, 40)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_evoformer_masked_queries(D, N, L, dtype):
    """Queries whose keys are all masked by one large finite number of the pair bias: their softmax is that of the other terms, forward
    and backward, also where they share keys with a part of the row mask; and a row mask that is large above zero."""
    torch.manual_seed(7)
    H = 8
    mk = lambda *s: torch.randn(*s, device="cuda")
    Q, K, V, g = (mk(1, N, L, H, D).bfloat16() for _ in range(4))
    b1 = (mk(1, N, 1, 1, L) > 1).float() * -1e9
    b1[..., 0] = 0
    b1[0, 1] = mk(L) + 3e4
    b1[0, 2] = 0
    b1[0, 2, 0, 0, 0] = 1e9
    b2 = (mk(1, 1, H, L, L) * 2).to(dtype)
    b2[0, 0, 1] = -1e9
    b2[0, 0, 2, L - 1] = -3e8
    b2[0, 0, 3, 5] = -20480.0 + (mk(L) > 0) * -128.0
    b2[0, 0, 4, 3, 1:] = -1e9  # a key is left: nothing to move
    b2[0, 0, 5, :, L // 3:] = -1e9
    ins = [t.requires_grad_(True) for t in (Q, K, V, b1, b2)]
    out = ea.evoformer_attention(*ins)
    grads = torch.autograd.grad(out, ins, g)
    ref = [t.detach().double().requires_grad_(True) for t in ins]
    q, k, v = (t.transpose(-2, -3) for t in ref[:3])
    want = (torch.softmax(q @ k.transpose(-1, -2).contiguous() / D ** 0.5 + ref[3] + ref[4], -1) @ v).transpose(-2, -3)
    # p, ds and the results are rounded to 8 bits, 4 x 2^-9
    assert (out.double() - want).norm() <= 8e-3 * want.norm()
    for a, b in zip(grads, torch.autograd.grad(want, ref, g.double())):
        assert torch.isfinite(a).all() and (a.double() - b).norm() <= 8e-3 * b.norm(), a.shape
        if a.shape == Q.shape:  # and of the head whose keys are all masked alone
            assert (a[:, :, :, 1].double() - b[:, :, :, 1]).norm() <= 8e-3 * b[:, :, :, 1].norm()


@pytest.mark.gpu
@pytest.mark.parametrize("D,N,dtype", [(64, 400, torch.bfloat16), (32, 191, torch.bfloat16), (32, 193, torch.bfloat16), (64, 3, torch.float32)])
def test_evoformer_packed_biases(D, N, dtype):
    """What the forward keeps for the backward: the pair bias in its own type, and a key of the mask takes 20 bytes."""
    q = torch.randn(1, N, 40, 8, D, device="cuda").bfloat16()
    b2 = torch.randn(1, 1, 8, 40, 40, device="cuda").to(dtype)
    _, _, mask, pair = torch.ops.sxe.evoformer_fwd(q, q, q, None, b2, True)
    assert pair.dtype == dtype and pair.shape == (2, 8, 128, 128) and mask.nbytes == 20 * N * 128

"""gfx950 flash attention (fwd + bwd) vs an fp32 PyTorch reference: causal / full, MHA / GQA,
packed-QKV strided inputs with fused RoPE."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.float() - b.float()).norm() / (b.float().norm() + 1e-12)).item()


@pytest.fixture(scope="module", autouse=True)
def _native():
    from shuffle_exchange_amd.ops import native
    native.require_hip()


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,S,H,Hk", [(2, 256, 4, 4), (1, 384, 8, 2), (2, 128, 4, 1)])
def test_flash_fwd_bwd(causal, B, S, H, Hk):
    from shuffle_exchange_amd.ops.attention import attention, reference_attention
    torch.manual_seed(0)
    D = 128
    q = torch.randn(B, S, H, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    k = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    v = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    o = attention(q, k, v, causal=causal)
    q2, k2, v2 = (t.detach().float().requires_grad_() for t in (q, k, v))
    o2 = reference_attention(q2, k2, v2, causal=causal)
    assert _rel(o, o2) < 1e-2
    do = torch.randn_like(o2)
    (o.float() * do).sum().backward()
    (o2 * do).sum().backward()
    assert _rel(q.grad, q2.grad) < 2e-2
    assert _rel(k.grad, k2.grad) < 2e-2
    assert _rel(v.grad, v2.grad) < 2e-2


@pytest.mark.parametrize("hpw", ["1", "2", "4", "3"])
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("B,S,H,Hk", [(1, 384, 8, 2), (2, 256, 12, 3)])
def test_flash_bwd_dkdv_head_groups(hpw, D, B, S, H, Hk, monkeypatch):
    """Causal GQA backward with the dK/dV workgroups sweeping `hpw` query heads each
    (SXE_FA_DKDV_HPW, read per call): 1 and 2 write fp32 partials summed by the reduce kernel, a
    whole group (4 of G=4, 3 of G=3) writes dK/dV directly, a non-divisor falls back to 1."""
    from shuffle_exchange_amd.ops.attention import attention, reference_attention
    monkeypatch.setenv("SXE_FA_DKDV_HPW", hpw)
    torch.manual_seed(H + D)
    q = torch.randn(B, S, H, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    k = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    v = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    o = attention(q, k, v, causal=True)
    q2, k2, v2 = (t.detach().float().requires_grad_() for t in (q, k, v))
    o2 = reference_attention(q2, k2, v2, causal=True)
    do = torch.randn_like(o2)
    (o.float() * do).sum().backward()
    (o2 * do).sum().backward()
    assert _rel(q.grad, q2.grad) < 2e-2
    assert _rel(k.grad, k2.grad) < 2e-2
    assert _rel(v.grad, v2.grad) < 2e-2


@pytest.mark.parametrize("one_sweep", ["0", "1"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,S,H,Hk", [(1, 256, 4, 4), (1, 384, 8, 2)])
def test_flash_bwd_d256_sweeps(one_sweep, causal, B, S, H, Hk, monkeypatch):
    """Head dim 256 backward with dV and dK in two sweeps (default) or one (SXE_FA_DKDV_ONE_SWEEP=1,
    read per call), MHA and causal GQA (split + reduce), against the fp32 oracle."""
    from shuffle_exchange_amd.ops.attention import attention, reference_attention
    monkeypatch.setenv("SXE_FA_DKDV_ONE_SWEEP", one_sweep)
    torch.manual_seed(S + H)
    D = 256
    q = torch.randn(B, S, H, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    k = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    v = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    o = attention(q, k, v, causal=causal)
    q2, k2, v2 = (t.detach().float().requires_grad_() for t in (q, k, v))
    o2 = reference_attention(q2, k2, v2, causal=causal)
    do = torch.randn_like(o2)
    (o.float() * do).sum().backward()
    (o2 * do).sum().backward()
    assert _rel(q.grad, q2.grad) < 2e-2
    assert _rel(k.grad, k2.grad) < 2e-2
    assert _rel(v.grad, v2.grad) < 2e-2


@pytest.mark.parametrize("waves", ["4", "8"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,Sq,Sk,H,Hk,D", [(1, 512, 512, 8, 2, 128), (2, 256, 768, 4, 1, 128),
                                            (1, 512, 512, 4, 4, 64), (1, 384, 384, 4, 2, 128),
                                            (2, 512, 512, 8, 8, 128)])
def test_flash_bwd_dq_waves(waves, causal, B, Sq, Sk, H, Hk, D, monkeypatch):
    """dQ and dK/dV kernels with 4 or 8 waves per workgroup (SXE_FA_DQ_WAVES / SXE_FA_DKDV_WAVES,
    read per call; 8 needs the axis a multiple of 256 -- and head dim 128 for dK/dV -- else 4 runs)
    against the fp32 oracle, incl. q_len != kv_len and GQA (split + partials under the mask)."""
    from shuffle_exchange_amd.ops.attention import attention, reference_attention
    monkeypatch.setenv("SXE_FA_DQ_WAVES", waves)
    monkeypatch.setenv("SXE_FA_DKDV_WAVES", waves)
    torch.manual_seed(Sq + Sk + D)
    q = torch.randn(B, Sq, H, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    k = torch.randn(B, Sk, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    v = torch.randn(B, Sk, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    o = attention(q, k, v, causal=causal)
    q2, k2, v2 = (t.detach().float().requires_grad_() for t in (q, k, v))
    o2 = reference_attention(q2, k2, v2, causal=causal)
    do = torch.randn_like(o2)
    (o.float() * do).sum().backward()
    (o2 * do).sum().backward()
    assert _rel(q.grad, q2.grad) < 2e-2
    assert _rel(k.grad, k2.grad) < 2e-2
    assert _rel(v.grad, v2.grad) < 2e-2


def test_flash_lse():
    from shuffle_exchange_amd.ops.attention import attention_with_lse, reference_attention
    q = torch.randn(1, 256, 2, 128, device="cuda", dtype=torch.bfloat16)
    k = torch.randn(1, 256, 2, 128, device="cuda", dtype=torch.bfloat16)
    v = torch.randn(1, 256, 2, 128, device="cuda", dtype=torch.bfloat16)
    o, lse = attention_with_lse(q, k, v, causal=True)
    o2, lse2 = reference_attention(q.float(), k.float(), v.float(), causal=True, return_lse=True)
    assert _rel(o, o2) < 1e-2
    assert (lse - lse2).abs().max().item() < 1e-2


def test_packed_qkv_rope():
    from shuffle_exchange_amd.ops.attention import attention_qkv_rope, reference_attention
    from shuffle_exchange_amd.ops.rope import RopeCache, _ref_rope
    torch.manual_seed(1)
    B, S, nq, nkv, D = 2, 256, 8, 2, 128
    cache = RopeCache(D, 512, 500000.0, device="cuda")
    base = torch.randn(B, S, (nq + 2 * nkv) * D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    qkv = base.view(B, S, nq + 2 * nkv, D) * 1.0
    o = attention_qkv_rope(qkv, nq, nkv, cache)
    ref_in = base.detach().float().view(B, S, nq + 2 * nkv, D).requires_grad_()
    pos = torch.arange(S, device="cuda").repeat(B)
    rot = _ref_rope(ref_in[:, :, :nq + nkv].reshape(B * S, nq + nkv, D), cache.cos, cache.sin, pos).view(B, S, nq + nkv, D)
    q2, k2, v2 = rot[:, :, :nq], rot[:, :, nq:], ref_in[:, :, nq + nkv:]
    o2 = reference_attention(q2, k2, v2, causal=True)
    assert _rel(o, o2) < 1e-2
    do = torch.randn_like(o2)
    (o.float() * do).sum().backward()
    (o2 * do).sum().backward()
    assert _rel(base.grad.view_as(ref_in), ref_in.grad) < 2e-2


@pytest.mark.slow
def test_flash_perf_report():
    """Not a pass/fail perf gate: prints TFLOP/s of fwd and fwd+bwd at the Llama-3-8B shape."""
    from shuffle_exchange_amd.ops.attention import attention
    B, S, H, Hk, D = 4, 2048, 32, 8, 128
    q = torch.randn(B, S, H, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    k = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    v = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    flops = 4 * B * H * S * S * D / 2
    for _ in range(3):
        o = attention(q, k, v)
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(10):
        o = attention(q, k, v)
    e1.record()
    torch.cuda.synchronize()
    tf = flops / (e0.elapsed_time(e1) / 10 / 1e3) / 1e12
    g = torch.randn_like(o)
    e0.record()
    for _ in range(10):
        torch.autograd.grad(attention(q, k, v), (q, k, v), g)
    e1.record()
    torch.cuda.synchronize()
    tfb = 3.5 * flops / (e0.elapsed_time(e1) / 10 / 1e3) / 1e12
    print(f"\n[flash] fwd {tf:.0f} TFLOP/s, fwd+bwd {tfb:.0f} TFLOP/s (model FLOPs, 3.5x fwd)")


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,S,H,Hk,D", [(2, 100, 4, 4, 64), (1, 200, 8, 2, 128), (2, 128, 4, 2, 80),
                                        (1, 77, 2, 1, 96), (2, 300, 12, 12, 64)])
def test_flash_padded_shapes_run_hip(causal, B, S, H, Hk, D, monkeypatch):
    """Head dims below 128 and sequence lengths that are not multiples of 128 run the HIP kernels on
    padded copies (kv_len masks the padded keys) -- never SDPA -- and match the fp32 reference."""
    import torch.nn.functional as F
    from shuffle_exchange_amd.ops import attention as A
    calls = []
    monkeypatch.setattr(A, "_sdpa", lambda *a, **k: calls.append(1) or F.scaled_dot_product_attention(*a))
    torch.manual_seed(0)
    q = torch.randn(B, S, H, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    k = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    v = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    o = A.attention(q, k, v, causal=causal)
    assert not calls
    q2, k2, v2 = (t.detach().float().requires_grad_() for t in (q, k, v))
    o2 = A.reference_attention(q2, k2, v2, causal=causal)
    assert o.shape == o2.shape
    assert _rel(o, o2) < 1e-2
    do = torch.randn_like(o2)
    (o.float() * do).sum().backward()
    (o2 * do).sum().backward()
    for a, b in ((q.grad, q2.grad), (k.grad, k2.grad), (v.grad, v2.grad)):
        assert a.shape == b.shape and _rel(a, b) < 2e-2


def test_smoke_shape_llama_d64_uses_hip():
    """The driver's smoke shape (hidden 256, 4 heads -> D = 64, S = 128) runs the HIP kernels."""
    from shuffle_exchange_amd.ops import attention as A
    from shuffle_exchange_amd.ops.rope import RopeCache
    B, S, nq, nkv, D = 2, 128, 4, 2, 64
    cache = RopeCache(D, 256, 10000.0, device="cuda")
    qkv = torch.randn(B, S, nq + 2 * nkv, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    o = A.attention_qkv_rope(qkv * 1.0, nq, nkv, cache)
    o.float().square().mean().backward()
    assert o.shape == (B, S, nq, D) and torch.isfinite(qkv.grad).all()


def _no_sdpa(monkeypatch):
    from shuffle_exchange_amd.ops import attention as A

    def boom(*a, **k):
        raise AssertionError("SDPA ran")
    monkeypatch.setattr(A, "_sdpa", boom)
    return A


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("B,S,H,Hk", [(2, 256, 4, 2), (1, 384, 4, 4)])
def test_flash_native_head_dims(causal, D, B, S, H, Hk, monkeypatch):
    """Head dims 64 and 256 run their own kernel instantiations in place (no padding copy, no SDPA)."""
    A = _no_sdpa(monkeypatch)
    torch.manual_seed(0)
    q = torch.randn(B, S, H, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    k = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    v = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    assert A.hip_supported(q, k, v)
    o = A.attention(q, k, v, causal=causal)
    q2, k2, v2 = (t.detach().float().requires_grad_() for t in (q, k, v))
    o2 = A.reference_attention(q2, k2, v2, causal=causal)
    assert _rel(o, o2) < 1e-2
    do = torch.randn_like(o2)
    (o.float() * do).sum().backward()
    (o2 * do).sum().backward()
    for a, b in ((q.grad, q2.grad), (k.grad, k2.grad), (v.grad, v2.grad)):
        assert _rel(a, b) < 2e-2


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("Sq,Sk,D", [(128, 384, 128), (256, 1024, 64), (100, 300, 96), (1, 517, 128),
                                     (384, 128, 128), (200, 200, 256)])
def test_flash_cross_and_prefix_lengths(causal, Sq, Sk, D, monkeypatch):
    """q_len != kv_len (prefix / chunked-prefill / cross attention): bottom-right aligned causal mask
    like flash-attn, on the HIP kernels (padded where the lengths are not multiples of 128)."""
    if causal and Sq > Sk:
        pytest.skip("causal with more queries than keys leaves fully masked rows (not a real use)")
    A = _no_sdpa(monkeypatch)
    torch.manual_seed(1)
    B, H, Hk = 2, 4, 2
    q = torch.randn(B, Sq, H, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    k = torch.randn(B, Sk, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    v = torch.randn(B, Sk, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    o = A.attention(q, k, v, causal=causal)
    q2, k2, v2 = (t.detach().float().requires_grad_() for t in (q, k, v))
    o2 = A.reference_attention(q2, k2, v2, causal=causal)
    assert o.shape == o2.shape and _rel(o, o2) < 1e-2
    do = torch.randn_like(o2)
    (o.float() * do).sum().backward()
    (o2 * do).sum().backward()
    for a, b in ((q.grad, q2.grad), (k.grad, k2.grad), (v.grad, v2.grad)):
        assert a.shape == b.shape and _rel(a, b) < 2e-2
    ol, lse = A.attention_with_lse(q.detach(), k.detach(), v.detach(), causal=causal)
    _, lse2 = A.reference_attention(q2.detach(), k2.detach(), v2.detach(), causal=causal, return_lse=True)
    assert (lse - lse2).abs().max().item() < 2e-2


@pytest.mark.parametrize("dma", ["0", "1"])
@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,Sq,Sk,H,Hk,D", [(2, 256, 256, 4, 4, 128), (1, 512, 512, 8, 2, 128),
                                            (2, 256, 256, 4, 2, 64), (1, 256, 768, 4, 1, 128),
                                            (1, 512, 1024, 4, 2, 64), (1, 1024, 1024, 2, 2, 128)])
def test_flash_fwd_variants(dma, waves, causal, B, Sq, Sk, H, Hk, D, monkeypatch):
    """Every forward variant (4 and 8 waves per workgroup, SXE_FA_FWD_WAVES; K/V through registers
    or by LDS-DMA, SXE_FA_FWD_DMA; both read per call) against the fp32 oracle: head dims 64 / 128,
    causal / full, q_len != kv_len, GQA."""
    A = _no_sdpa(monkeypatch)
    monkeypatch.setenv("SXE_FA_FWD_WAVES", str(waves))
    monkeypatch.setenv("SXE_FA_FWD_DMA", dma)
    torch.manual_seed(2)
    q = torch.randn(B, Sq, H, D, device="cuda", dtype=torch.bfloat16)
    k = torch.randn(B, Sk, Hk, D, device="cuda", dtype=torch.bfloat16)
    v = torch.randn(B, Sk, Hk, D, device="cuda", dtype=torch.bfloat16)
    assert A.hip_supported(q, k, v)
    o, lse = A.attention_with_lse(q, k, v, causal=causal)
    o2, lse2 = A.reference_attention(q.float(), k.float(), v.float(), causal=causal, return_lse=True)
    assert _rel(o, o2) < 1e-2
    assert (lse - lse2).abs().max().item() < 2e-2


@pytest.mark.parametrize("Sq,Sk,kv_len,qoff,causal", [(256, 128, 64, 0, False),    # one tile
                                                       (256, 128, 65, 0, False),    # and one key
                                                       (256, 256, 200, 0, True),    # rows past the keys
                                                       (512, 128, 128, -384, True),  # rows that see nothing
                                                       (256, 640, 640, 384, True),
                                                       (512, 512, 512, 17, True)])   # diagonal inside tiles
@pytest.mark.parametrize("D", [64, 128])
def test_flash_fwd_waves_in_turns(D, Sq, Sk, kv_len, qoff, causal, monkeypatch):
    """The eight-wave forward, whose waves take turns at the matrix core, does per query what the
    four-wave one does in the same order: the outputs and LSEs are the same bits."""
    from shuffle_exchange_amd.ops import native
    native.require_hip()
    torch.manual_seed(3)
    q = torch.randn(2, Sq, 4, D, device="cuda", dtype=torch.bfloat16)
    k = torch.randn(2, Sk, 2, D, device="cuda", dtype=torch.bfloat16)
    v = torch.randn(2, Sk, 2, D, device="cuda", dtype=torch.bfloat16)
    out = []
    for waves in ("8", "4"):
        monkeypatch.setenv("SXE_FA_FWD_WAVES", waves)
        out.append(torch.ops.sxe.flash_attn_fwd(q, k, v, causal, D ** -0.5, kv_len, qoff))
    for a, b in zip(*out):
        assert torch.equal(a, b)
    # in pairs the sums of every other tile meet at the end, each against a maximum of its own: the probabilities are
    # rounded to bf16 at other places (2^-8 of each, twice, of sum p |v|), and so is the result
    size = torch.ops.sxe.flash_attn_fwd(q, k, v.abs(), causal, D ** -0.5, kv_len, qoff)[0].float()
    monkeypatch.setenv("SXE_FA_FWD_WAVES", "16")
    o, lse = torch.ops.sxe.flash_attn_fwd(q, k, v, causal, D ** -0.5, kv_len, qoff)
    assert bool(((o.float() - out[1][0].float()).abs() <= 2 ** -7 * (out[1][0].float().abs() + 1.01 * size)).all())
    torch.testing.assert_close(lse, out[1][1], rtol=2 ** -18, atol=2 ** -16)
    if causal and qoff == 0:  # a value that no query before it sees, at the start of half a tile
        v[:, 96] = float("nan")
        k[:, 96] = float("inf")
        for waves in ("8", "4", "16"):
            monkeypatch.setenv("SXE_FA_FWD_WAVES", waves)
            assert torch.ops.sxe.flash_attn_fwd(q, k, v, causal, D ** -0.5, kv_len, qoff)[0][:, :96].isfinite().all()


@pytest.mark.parametrize("Sq,Sk,causal", [(256, 128, False), (128, 384, True), (384, 384, True), (512, 128, True)])
@pytest.mark.parametrize("D", [64, 128])
def test_flash_bwd_pairs(D, Sq, Sk, causal, monkeypatch):
    """dQ and dK / dV by pairs of waves that take every other tile (none, one, or a different number of them): the four-wave form's
    products, their fp32 sums of a few tiles added in another order (2^-24 of the sizes of the terms each, which are below 16 here) and
    rounded once to bf16."""
    torch.manual_seed(4)
    q, do = (torch.randn(2, Sq, 4, D, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    k, v = (torch.randn(2, Sk, 2, D, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    o, lse = torch.ops.sxe.flash_attn_fwd(q, k, v, causal, D ** -0.5)
    out = []
    for waves in ("4", "16"):
        monkeypatch.setenv("SXE_FA_DQ_WAVES", waves)
        monkeypatch.setenv("SXE_FA_DKDV_WAVES", waves)
        out.append([torch.full_like(t, float("nan")) for t in (q, k, v)])
        torch.ops.sxe.flash_attn_bwd(do, q, k, v, o, lse, *out[-1], causal, D ** -0.5)
    for a, b in zip(*out):
        assert bool(((a.float() - b.float()).abs() <= 2 ** -7 * a.float().abs() + 2 ** -18).all())


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,S,H,Hk,D", [(1, 4096, 10, 2, 64),   # 320 workgroups of 128 rows: the second half of the grid runs backwards
                                        (1, 2176, 20, 5, 128),  # 340, no whole 256 rows
                                        (1, 2048, 64, 16, 128),  # 512 of 256: eight waves; K/V heads fill the chip
                                        (4, 1024, 64, 16, 64),  # 1024 of 256
                                        (1, 512, 8, 1, 128)])   # dK / dV of 8 query heads in parts
def test_flash_default_launch_rules(B, S, H, Hk, D, causal, monkeypatch):
    """The launches that the sizes choose against the fp32 oracle, per head (bf16 results of fp32 sums: as the tests above)."""
    A = _no_sdpa(monkeypatch)
    torch.manual_seed(5)
    q = torch.randn(B, S, H, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    k = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    v = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    do = torch.randn(B, S, H, D, device="cuda", dtype=torch.bfloat16)
    o = A.attention(q, k, v, causal=causal)
    o.backward(do)
    G = H // Hk
    for hk in (0, Hk - 1):
        q2, do2 = (t[:, :, hk * G:(hk + 1) * G].detach().float() for t in (q, do))
        q2.requires_grad_()
        k2, v2 = (t[:, :, hk:hk + 1].detach().float().requires_grad_() for t in (k, v))
        o2 = A.reference_attention(q2, k2, v2, causal=causal)
        o2.backward(do2)
        assert _rel(o[:, :, hk * G:(hk + 1) * G], o2) < 1e-2
        assert _rel(q.grad[:, :, hk * G:(hk + 1) * G], q2.grad) < 2e-2
        assert _rel(k.grad[:, :, hk:hk + 1], k2.grad) < 2e-2 and _rel(v.grad[:, :, hk:hk + 1], v2.grad) < 2e-2


def _chunked_reference(q, k, v, do, causal, chunk=1024):
    """fp32 attention output and gradients for long sequences, one query block at a time (the full
    score matrix of S = 16k would not be materialised at once). q [B, S, H, D], k/v [B, S, Hk, D]."""
    B, S, H, D = q.shape
    G = H // k.shape[2]
    qf, kf, vf, dof = (t.detach().float() for t in (q, k, v, do))
    kf = kf.repeat_interleave(G, dim=2).requires_grad_()
    vf = vf.repeat_interleave(G, dim=2).requires_grad_()
    out = torch.empty_like(qf)
    dq = torch.empty_like(qf)
    scale = 1.0 / math.sqrt(D)
    for s0 in range(0, S, chunk):
        qc = qf[:, s0:s0 + chunk].clone().requires_grad_()
        sc = torch.einsum("bqhd,bkhd->bhqk", qc, kf) * scale
        if causal:
            qi = torch.arange(s0, min(S, s0 + chunk), device=q.device)[:, None]
            ki = torch.arange(S, device=q.device)[None, :]
            sc = sc.masked_fill(ki > qi, float("-inf"))
        o = torch.einsum("bhqk,bkhd->bqhd", torch.softmax(sc, -1), vf)
        out[:, s0:s0 + chunk] = o.detach()
        (o * dof[:, s0:s0 + chunk]).sum().backward()
        dq[:, s0:s0 + chunk] = qc.grad
    Hk = k.shape[2]
    dk = kf.grad.view(B, S, Hk, G, D).sum(3)
    dv = vf.grad.view(B, S, Hk, G, D).sum(3)
    return out, dq, dk, dv


@pytest.mark.parametrize("S,causal", [(8192, True), (8192, False), (16384, True)])
def test_flash_long_sequence_default_launch(S, causal, monkeypatch):
    """Long-context shapes (the SP-32k per-rank slices, H4/1 GQA) with the DEFAULT launch selection
    -- no env forcing: from 8k tokens the 8-wave dQ / dK/dV kernels are chosen -- against a chunked
    fp32 reference. Long-range accumulation and online-softmax rescaling errors show up here, not at
    the S <= 768 of the other tests."""
    for var in [v for v in list(__import__("os").environ) if v.startswith("SXE_FA_")]:
        monkeypatch.delenv(var, raising=False)
    from shuffle_exchange_amd.ops.attention import attention
    torch.manual_seed(S + causal)
    B, H, Hk, D = 1, 4, 1, 128
    q = torch.randn(B, S, H, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    k = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    v = torch.randn(B, S, Hk, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    o = attention(q, k, v, causal=causal)
    do = torch.randn_like(o)
    o.backward(do)
    ro, rdq, rdk, rdv = _chunked_reference(q, k, v, do, causal)
    assert _rel(o, ro) < 1e-2
    assert _rel(q.grad, rdq) < 2e-2
    assert _rel(k.grad, rdk) < 2e-2
    assert _rel(v.grad, rdv) < 2e-2

"""Dual-layout backward paths (GPU): the LM-head gradient kernel that writes g and g^T
(xent_grad_dual), the fused LM-head loss on that path, and the fused QKV projection + attention
node whose weight gradient runs as a TN GEMM -- each against a plain fp32 PyTorch reference."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _native():
    from shuffle_exchange_amd.ops import native
    native.require_hip()


def _rel(a, b):
    return ((a.float() - b.float()).norm() / (b.float().norm() + 1e-12)).item()


def test_xent_grad_dual_kernel():
    torch.manual_seed(0)
    T, V = 192, 1280
    logits = (torch.randn(T, V, device="cuda") * 3).to(torch.bfloat16)
    tgt = torch.randint(0, V, (T,), device="cuda")
    tgt[5] = -100
    tgt[100] = V - 1
    ref_in = logits.float()
    lse = torch.logsumexp(ref_in, dim=-1)
    sa = torch.tensor([0.25], device="cuda")
    sb = torch.tensor([3.0], device="cuda")
    ref = torch.softmax(ref_in, dim=-1)
    ref[torch.arange(T, device="cuda")[tgt >= 0], tgt[tgt >= 0]] -= 1.0
    ref *= 0.75
    ref[tgt < 0] = 0
    buf = logits.clone()
    gT = torch.ops.sxe.xent_grad_dual(buf, tgt, lse, -100, sa, sb)
    assert gT.shape == (V, T)
    assert _rel(buf, ref) < 1e-2
    assert torch.equal(gT, buf.t().contiguous())
    assert buf[5].abs().max().item() == 0.0


def test_fused_linear_xent_dual_path_matches_reference():
    from shuffle_exchange_amd.ops import cross_entropy as CE
    torch.manual_seed(1)
    T, H, V = 256, 128, 2048
    h = (torch.randn(T, H, device="cuda") * 0.5).to(torch.bfloat16).requires_grad_()
    W = (torch.randn(V, H, device="cuda") * 0.05).to(torch.bfloat16).requires_grad_()
    tgt = torch.randint(0, V, (T,), device="cuda")
    tgt[:9] = -100
    assert CE._dual_ok(h, W)
    loss = CE.fused_linear_cross_entropy(h, W, tgt)
    (loss * 0.5).backward()
    h2, W2 = h.detach().float().requires_grad_(), W.detach().float().requires_grad_()
    ref = F.cross_entropy(h2 @ W2.t(), tgt, ignore_index=-100)
    (ref * 0.5).backward()
    assert abs(loss.item() - ref.item()) < 1e-2 * abs(ref.item())
    assert _rel(h.grad, h2.grad) < 3e-2 and _rel(W.grad, W2.grad) < 3e-2


def test_fused_linear_xent_dual_writes_grad_target():
    """The LM-head weight gradient lands in the optimizer's fp32 accumulator (accumulate on)."""
    from shuffle_exchange_amd.ops import cross_entropy as CE
    torch.manual_seed(2)
    T, H, V = 128, 128, 1024
    h = (torch.randn(T, H, device="cuda") * 0.5).to(torch.bfloat16).requires_grad_()
    W = torch.nn.Parameter((torch.randn(V, H, device="cuda") * 0.05).to(torch.bfloat16))
    buf = torch.full((V, H), 1.0, device="cuda")
    done = []
    W._sxe_grad_target = lambda p: (buf, True)
    W._sxe_grad_done = lambda p: done.append(1)
    tgt = torch.randint(0, V, (T,), device="cuda")
    CE.fused_linear_cross_entropy(h, W, tgt).backward()
    assert W.grad is None and done == [1]
    W2 = W.detach().float().requires_grad_()
    F.cross_entropy(h.detach().float() @ W2.t(), tgt).backward()
    assert _rel(buf - 1.0, W2.grad) < 3e-2


@pytest.mark.parametrize("target", [False, True])
def test_qkv_proj_attention_matches_unfused(target):
    from shuffle_exchange_amd.ops.attention import _QKVProjAttn, qkv_proj_attention, reference_attention
    from shuffle_exchange_amd.ops.linear import Linear
    from shuffle_exchange_amd.ops.rope import RopeCache, _ref_rope
    torch.manual_seed(3)
    B, S, H, nq, nkv, D = 2, 256, 512, 4, 2, 128
    cache = RopeCache(D, 512, 500000.0, device="cuda")
    proj = Linear(H, (nq + 2 * nkv) * D, bias=False, init_std=0.02).to(device="cuda", dtype=torch.bfloat16)
    x = (torch.randn(B, S, H, device="cuda") * 0.5).to(torch.bfloat16).requires_grad_()
    buf = torch.zeros(proj.weight.shape, device="cuda")
    if target:
        proj.weight._sxe_grad_target = lambda p: (buf, True)
        proj.weight._sxe_grad_done = lambda p: None
    seen = []
    orig = _QKVProjAttn.apply
    _QKVProjAttn.apply = lambda *a: (seen.append(1), orig(*a))[1]
    try:
        o = qkv_proj_attention(x, proj, nq, nkv, cache)
    finally:
        _QKVProjAttn.apply = orig
    assert seen == [1], "fused node not taken"
    x2 = x.detach().float().requires_grad_()
    w2 = proj.weight.detach().float().requires_grad_()
    qkv = (x2 @ w2.t()).view(B, S, nq + 2 * nkv, D)
    pos = torch.arange(S, device="cuda").repeat(B)
    rot = _ref_rope(qkv[:, :, :nq + nkv].reshape(B * S, nq + nkv, D), cache.cos, cache.sin, pos).view(B, S, nq + nkv, D)
    o2 = reference_attention(rot[:, :, :nq], rot[:, :, nq:], qkv[:, :, nq + nkv:], causal=True)
    assert _rel(o, o2) < 2e-2
    do = torch.randn_like(o2)
    (o.float() * do).sum().backward()
    (o2 * do).sum().backward()
    assert _rel(x.grad, x2.grad) < 3e-2
    dw = buf if target else proj.weight.grad
    assert proj.weight.grad is None if target else True
    assert _rel(dw, w2.grad) < 3e-2


def _train(stage, gas, stash, steps=2):
    import shuffle_exchange_amd as sxe
    from shuffle_exchange_amd.models import LlamaForCausalLM, llama_config
    from shuffle_exchange_amd.ops import mlp
    torch.manual_seed(0)
    cfg = llama_config("llama-tiny", hidden_size=256, intermediate_size=512, num_attention_heads=4,
                       num_key_value_heads=2, vocab_size=1024, num_hidden_layers=2)
    model = LlamaForCausalLM(cfg).to(device="cuda", dtype=torch.bfloat16)
    ds = {"train_micro_batch_size_per_gpu": 2, "gradient_accumulation_steps": gas, "bf16": {"enabled": True},
          "zero_optimization": {"stage": stage}, "optimizer": {"type": "AdamW", "params": {"lr": 1e-3}},
          "gradient_clipping": 1.0}
    engine, _, _, _ = sxe.initialize(model=model, config=ds)
    calls = []
    orig = mlp._may_stash
    mlp.STASH = stash
    mlp._may_stash = lambda w, g: calls.append(orig(w, g)) or calls[-1]
    try:
        g = torch.Generator(device="cuda").manual_seed(1)
        for _ in range(steps * gas):
            ids = torch.randint(0, cfg.vocab_size, (2, 128), device="cuda", generator=g)
            loss = engine(ids, labels=ids)
            engine.backward(loss)
            engine.step()
    finally:
        mlp._may_stash, mlp.STASH = orig, True
    torch.cuda.synchronize()
    return [p.detach().float().clone() for p in engine.module.parameters()], calls


@pytest.mark.parametrize("stage,gas", [(3, 2), (3, 3), (2, 2)])
def test_wgrad_stash_bit_identical(stage, gas):
    """Holding a micro-step's bf16 weight gradient and folding it with the next one (acc2_bf16_)
    is the same fp32 sum as writing every micro-step: parameters after two steps are identical."""
    on, calls = _train(stage, gas, True)
    off, _ = _train(stage, gas, False)
    assert any(calls), "no weight gradient was held"
    assert all(torch.equal(a, b) for a, b in zip(on, off))


def test_acc2_bf16_kernel():
    n = 1000003
    a = torch.randn(n, device="cuda").to(torch.bfloat16)
    b = torch.randn(n, device="cuda").to(torch.bfloat16)
    d = torch.randn(n, device="cuda")
    ref = d + a.float() + b.float()
    torch.ops.sxe.acc2_bf16_(d, a, b, True)
    assert torch.equal(d, ref)
    torch.ops.sxe.acc2_bf16_(d, a, b, False)
    assert torch.equal(d, a.float() + b.float())


@pytest.mark.parametrize("n", [1, 3, 4, 1023, 2047, 2048, 2049, 4100, 100003])
@pytest.mark.parametrize("accumulate", [False, True])
def test_acc2_bf16_sizes(n, accumulate):
    """Edges of a workgroup's 2048 elements; what lies behind the operands stays."""
    torch.manual_seed(0)
    room = torch.randn(n + 8, device="cuda")
    a, b = (torch.randn(n + 8, device="cuda").bfloat16() for _ in range(2))
    want = room.clone()
    want[:n] = (want[:n] if accumulate else 0) + a[:n].float() + b[:n].float()
    torch.ops.sxe.acc2_bf16_(room[:n], a[:n], b[:n], accumulate)
    assert torch.equal(room, want)

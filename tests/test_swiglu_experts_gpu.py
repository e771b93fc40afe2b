"""Routed SwiGLU experts over [E, K, N] weights (csrc/kernels/experts_kn.hip, experts_kn_tile.hip) against fp64, and Mixtral decode steps replayed
from graphs against eager ones."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _native():
    from shuffle_exchange_amd.ops import native
    native.require_hip()


def _reference(x, logits, k, w_gu, w_down):
    top, idx = logits.double().topk(k, -1)
    wt = torch.softmax(top, -1)
    out = torch.zeros(x.shape[0], w_down.shape[2], dtype=torch.float64, device=x.device)
    for e in range(w_gu.shape[0]):
        t, c = (idx == e).nonzero(as_tuple=True)
        g, u = (x[t].double() @ w_gu[e].double()).chunk(2, -1)
        out.index_add_(0, t, (torch.nn.functional.silu(g) * u) @ w_down[e].double() * wt[t, c, None])
    return out


@pytest.mark.parametrize("T", [1, 2, 7, 16, 33, 100, 256])
@pytest.mark.parametrize("E,k,K,I,N", [(8, 2, 256, 192, 128), (4, 1, 32, 64, 256), (8, 2, 2080, 1088, 384), (3, 3, 96, 64, 128),
                                       (8, 2, 2080, 1088, 4096)])  # the last: from 64 MB on weights are loaded another way
@pytest.mark.parametrize("skew", [False, True])
def test_streaming_kernels(T, E, k, K, I, N, skew, monkeypatch):
    from shuffle_exchange_amd.ops import moe
    monkeypatch.setattr(moe, "KN_ROWS", 1 << 20)
    g = torch.Generator(device="cuda").manual_seed(T + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = rnd(T, K).bfloat16()
    w_gu, w_down = (rnd(E, K, 2 * I) * K ** -0.5).bfloat16(), (rnd(E, I, N) * I ** -0.5).bfloat16()
    logits = rnd(T, E)
    if skew:  # every token to the same experts: more rows than one pass holds
        logits[:, :k] += 100
    assert moe.swiglu_experts_ok(x, w_gu, w_down)
    got = moe.swiglu_experts(x, moe.route_logits(logits, k), w_gu, w_down)
    ref = _reference(x, logits, k, w_gu, w_down)
    # the hidden row and the output are rounded to bf16 (2^-9 each)
    assert ((got.double() - ref).norm() / ref.norm()).item() < 5e-3
    monkeypatch.setattr(moe, "KN_ROWS", 0)  # the tile products behind the same routing
    tiles = moe.swiglu_experts(x, moe.route_logits(logits, k), w_gu, w_down)
    assert ((tiles.double() - ref).norm() / ref.norm()).item() < 8e-3


@pytest.mark.parametrize("T", [1, 127, 128, 129, 300, 1025])
@pytest.mark.parametrize("E,k,K,I,N", [(8, 2, 256, 192, 128), (4, 1, 32, 64, 384), (2, 2, 96, 136, 272), (70, 2, 160, 128, 256)])
@pytest.mark.parametrize("skew", [False, True])
def test_tile_kernels(T, E, k, K, I, N, skew):
    """Prefill's products: row tiles and halves of them, column remainders, one to five slabs of K, more experts than lanes."""
    from shuffle_exchange_amd.ops import moe
    g = torch.Generator(device="cuda").manual_seed(T + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = rnd(T, K).bfloat16()
    w_gu, w_down = (rnd(E, K, 2 * I) * K ** -0.5).bfloat16(), (rnd(E, I if I % 32 == 0 else K, N) * I ** -0.5).bfloat16()
    logits = rnd(T, E)
    if skew:
        logits[:, :k] += 100
    rows, _, _, offs, _ = moe.route_logits(logits, k).lists
    h = torch.ops.sxe.expert_swiglu_kn_tile(x, w_gu, offs, rows)
    a = h if I % 32 == 0 else x[rows.long()]
    y = torch.ops.sxe.expert_down_kn_tile(a, w_down, offs)
    o = offs.tolist()
    for e in range(E):
        r = slice(o[e], o[e + 1])
        gate, up = (x[rows[r].long()].double() @ w_gu[e].double()).chunk(2, -1)
        want, wy = torch.nn.functional.silu(gate) * up, a[r].double() @ w_down[e].double()
        # fp32 sums and one rounding of the result (2^-9)
        assert (h[r].double() - want).norm() <= 3e-3 * want.norm()
        assert (y[r].double() - wy).norm() <= 3e-3 * wy.norm()


@pytest.mark.parametrize("E,N,counts", [(8, 4096, [730] * 8), (8, 4096, [768, 767, 577, 640, 641, 705, 704, 769]), (8, 4096, [5840] + [0] * 7),
                                        (8, 4096, [1, 64, 65, 128, 129, 192, 193, 5068]), (70, 1040, [300] * 69 + [299]), (70, 1040, [0, 600] * 35)])
@pytest.mark.parametrize("K", [64, 160])
def test_tiles_of_either_height(E, N, counts, K):
    """Rows for which tiles of 192 may end sooner: the same sums whichever the kernel takes by the rows that the experts have."""
    g = torch.Generator(device="cuda").manual_seed(K)
    R = sum(counts)
    h = torch.randn(R, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(E, K, N, generator=g, device="cuda") * K ** -0.5).bfloat16()
    offs = torch.tensor([0] + counts, device="cuda").cumsum(0).int()
    y = torch.ops.sxe.expert_down_kn_tile(h, w, offs)
    for e, (a, b) in enumerate(zip(offs.tolist(), offs.tolist()[1:])):
        want = h[a:b].double() @ w[e].double()
        assert (y[a:b].double() - want).norm() <= 3e-3 * want.norm()  # fp32 sums and one rounding of the result (2^-9)


def _tile_activation(gate, up):
    """silu(gate) up of [I, 64] pairs that the products hold exactly, one term each."""
    offs, rows = torch.tensor([0, 64], device="cuda", dtype=torch.int32), torch.arange(64, device="cuda", dtype=torch.int32)
    return torch.ops.sxe.expert_swiglu_kn_tile(torch.eye(64, device="cuda").bfloat16(), torch.cat([gate, up]).t().contiguous()[None], offs, rows)


def test_tile_activation_in_32_bits():
    """A million gates whose exponents are large. A value that is off by e of itself before the rounding to bf16 rounds the other way with
    a chance of 2^8 e at the most (a spacing is 2^-8 of the value, or more): 5 units of 2^-24 let 80 of 2^20 differ, four standard
    deviations more are 116."""
    g = torch.Generator("cuda").manual_seed(3)
    gate = -(16 + 64 * torch.rand(16384, 64, device="cuda", generator=g)).bfloat16()
    up = (1 + torch.rand(16384, 64, device="cuda", generator=g)).bfloat16()
    y = _tile_activation(gate, up)
    want = (torch.nn.functional.silu(gate.double()) * up.double()).t()
    assert int((y != want.bfloat16()).sum()) <= 116
    torch.testing.assert_close(y.double(), want, rtol=2 ** -8, atol=0)


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), -500.0, -88.5, -87.0, -0.0])
def test_tile_activation_of_extremes(value):
    """As x / (1 + exp(-x)) in 32 bits: NaN of -inf, zeros far below (from -87 on, where the result is under 2^-119)."""
    gate = torch.zeros(128, 64, device="cuda").bfloat16()
    gate[:, 5] = value
    y = _tile_activation(gate, torch.ones_like(gate))[5]
    v = gate[:, 5].double()
    torch.testing.assert_close(y.double(), v / (1 + (-v).exp()), equal_nan=True, rtol=2 ** -8, atol=2.0 ** -119)


def test_mixtral_decode_graphs_match_eager():
    from shuffle_exchange_amd.inference.v2 import RaggedInferenceEngineConfig, build_engine
    from shuffle_exchange_amd.models import MixtralForCausalLM, mixtral_config
    torch.manual_seed(0)
    with torch.device("cuda"):
        model = MixtralForCausalLM(mixtral_config("mixtral-tiny", hidden_size=512, intermediate_size=256, num_attention_heads=4,
                                                  num_key_value_heads=2)).to(torch.bfloat16)
    engines = [build_engine(model, RaggedInferenceEngineConfig(num_kv_blocks=64, decode_graphs=g)) for g in (True, False)]
    gen = torch.Generator().manual_seed(1)
    prompts = [torch.randint(0, 512, (n,), generator=gen) for n in (5, 40, 17)]
    for e in engines:
        e.put([0, 1, 2], prompts)
    for step in range(5):  # 1 - 3 sequences: two buckets, replayed with eager work in between
        live = [0, 1, 2][:1 + step % 3]
        toks = [torch.randint(0, 512, (1,), generator=gen) for _ in live]
        a, b = (e.put(live, toks) for e in engines)
        torch.cuda.synchronize()
        assert (a - b).abs().max() <= 2e-2 * b.abs().max(), step
    assert engines[0]._decode_graphs.replays == 5 and engines[1]._decode_graphs is False

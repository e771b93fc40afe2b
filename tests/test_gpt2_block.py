"""A GPT-2 block whose second norm is not its own, or is looked at."""
import dataclasses

import pytest
import torch

from .dist_utils import run_dist


def _model():
    from shuffle_exchange_amd.models.gpt2 import GPT2LMHeadModel, gpt2_config
    torch.manual_seed(0)
    cfg = dataclasses.replace(gpt2_config("gpt2"), n_layer=2, n_embd=128, n_head=2, vocab_size=100, n_positions=64)
    return GPT2LMHeadModel(cfg), torch.randint(0, 100, (2, 64), generator=torch.Generator().manual_seed(1))


def test_norm_of_the_programs_own():
    """One that takes no residual, and one that a hook looks at: it sees one tensor."""
    model, ids = _model()
    want, seen = model(ids, labels=ids), []
    for blk in model.h:
        blk.ln_2.register_forward_hook(lambda mod, args, out: seen.append(out.shape))
    torch.testing.assert_close(model(ids, labels=ids), want)
    assert seen == [(2, 64, 128)] * 2
    for blk in model.h:
        norm = torch.nn.LayerNorm(128, blk.ln_2.eps)
        norm.load_state_dict(blk.ln_2.state_dict())
        blk.ln_2 = norm
    torch.testing.assert_close(model(ids, labels=ids), want)


def _case_fused_under_engine(rank, world, stage):
    import shuffle_exchange_amd as sxe
    from shuffle_exchange_amd.ops.linear import is_own_call
    from shuffle_exchange_amd.ops.norm import LayerNorm
    model, ids = _model()
    eng, _, _, _ = sxe.initialize(model=model, config={"train_micro_batch_size_per_gpu": 2, "zero_optimization": {"stage": stage},
                                                       "optimizer": {"type": "AdamW", "params": {"lr": 1e-2}}})
    own = [is_own_call(blk.ln_2, LayerNorm) for blk in model.h]
    seen = []
    model.h[0].ln_2.register_forward_pre_hook(lambda mod, args: seen.append(len(args)))
    model.h[1].ln_2.register_full_backward_hook(lambda mod, gin, gout: seen.append(len(gout)))
    eng.backward(eng(ids, labels=ids))
    return own, [is_own_call(blk.ln_2, LayerNorm) for blk in model.h], seen


@pytest.mark.parametrize("stage", [0, 1, 2, 3])
def test_engines_hooks_look_at_nothing(stage):
    """The residual sum stays in the norm's launch under every engine, whose hooks only wait for parameters; not beside a program's."""
    (own, hooked, seen), = run_dist(_case_fused_under_engine, 1, stage)
    assert own == [True, True] and hooked == [False, False] and seen == [1, 1]

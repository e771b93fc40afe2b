"""A GPT-2 block whose second norm is not its own, or is looked at."""
import dataclasses

import torch


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

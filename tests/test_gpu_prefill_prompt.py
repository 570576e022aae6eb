"""forward() of a long causal prompt: whichever rows' logits are asked for, and however the prompt is cut
into prefill calls, they are the rows of the all-logits forward bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,chunk", [(65, 4096), (300, 128), (300, 4096)])
def test_forward_returns_the_rows_asked_for(monkeypatch, tokens, chunk):
    import ssd.models.subnetwork_draft as sdm
    from ssd.engine.speculative import TargetRunner
    from ssd.models.llama import LlamaShape, MI355XLlama

    target = TargetRunner(MI355XLlama.synthetic(LlamaShape(256, 2, 4, 2, 64, 512, 1000), seed=3))
    ids = torch.randint(0, 1000, (1, tokens), generator=torch.Generator().manual_seed(4))
    full = target(ids, past_key_values=target.new_cache(tokens + 64))
    assert full.logits.shape == (1, tokens, 1000) and full.hidden_states.shape == (1, tokens, 256)
    monkeypatch.setattr(sdm, "PREFILL_CHUNK", chunk)
    for keep in (0, 1, 64, 65, 200, 1000):
        cache = target.new_cache(tokens + 64)
        out = target(ids.cuda(), torch.arange(tokens)[None], cache, logits_to_keep=keep)
        want = full.logits[:, -keep:] if keep else full.logits
        assert torch.equal(out.logits, want) and torch.equal(out.hidden_states, full.hidden_states)
        assert cache.get_seq_length() == tokens
    assert target(ids, past_key_values=target.new_cache(tokens), compute_logits=False).logits is None
    with pytest.raises(RuntimeError):
        target(torch.full((1, tokens), 1 << 40), past_key_values=target.new_cache(tokens))

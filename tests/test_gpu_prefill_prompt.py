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


@pytest.fixture(scope="module")
def target():
    from ssd.engine.speculative import TargetRunner
    from ssd.models.llama import LlamaShape, MI355XLlama

    return TargetRunner(MI355XLlama.synthetic(LlamaShape(256, 2, 4, 2, 64, 512, 1000), seed=3))


@pytest.mark.parametrize("bad", [torch.zeros(1, 65, 2, dtype=torch.int64), torch.zeros(1, 65, 1, dtype=torch.int64),
                                 torch.full((1, 65), 4_000_000_000, dtype=torch.uint32),
                                 torch.full((1, 65), 1 << 40, dtype=torch.uint64), torch.full((1, 65), 3e9),
                                 torch.full((1, 65), float("nan"))], ids=lambda t: f"{tuple(t.shape)}-{t.dtype}".replace("torch.", ""))
def test_long_prompts_refuse_what_short_ones_refuse(target, bad):
    """Ids that are no [1, tokens] table or do not fit int32, from a prompt that runs on the prefill kernels and
    from one of 8 tokens on the decode kernels. The cache is left as it was."""
    for n in (65, 8):
        cache = target.new_cache(192)
        with pytest.raises((RuntimeError, ValueError)):
            target(bad[:, :n], past_key_values=cache)
        assert cache.get_seq_length() == 0


@pytest.mark.parametrize("dtype", [torch.int32, torch.int16, torch.uint8, torch.float32])
def test_long_prompts_take_ids_of_any_type(target, dtype):
    ids = torch.randint(0, 200, (1, 70), generator=torch.Generator().manual_seed(1))
    want = target(ids, past_key_values=target.new_cache(80)).logits
    for x in (ids.to(dtype), ids.to(dtype).cuda()):
        assert torch.equal(target(x, past_key_values=target.new_cache(80)).logits, want)


@pytest.mark.parametrize("kind", ["list", "pageable", "pinned", "device"])
def test_prefill_chunk_has_taken_its_ids_when_it_returns(target, kind):
    """The transfer of the ids is not waited for, so a caller who reuses a buffer of any kind must not change them. The
    stream is held busy until after the buffer is overwritten."""
    ids = torch.randint(0, 1000, (70,), generator=torch.Generator().manual_seed(2), dtype=torch.int32)
    cache = target.new_cache(128)
    cache.ensure(target.num_kv_heads, target.head_dim, target.model.device)
    want = target.prefill_chunk(ids.tolist(), 0, cache, True).clone()
    buf = {"list": ids.tolist(), "pageable": ids.clone(), "pinned": ids.pin_memory(), "device": ids.cuda()}[kind]
    torch.cuda.synchronize()
    torch.cuda._sleep(20_000_000)  # about 10 ms
    got = target.prefill_chunk(buf, 0, cache, True)
    buf[:] = [0] * 70 if kind == "list" else torch.zeros(70, dtype=torch.int32)
    assert torch.equal(got, want)


@pytest.mark.parametrize("tokens,past,decode", [(64, 0, True), (65, 0, False), (65, 6240, False), (65, 6241, True),
                                                (100, 9600, False), (100, 12000, True), (255, 24480, False),
                                                (255, 24481, True), (256, 30000, False)])
def test_short_prompts_after_a_long_past_run_on_the_decode_kernels(target, tokens, past, decode):
    """Past the line the rows' bits are the decode forward's (an explicit causal mask always takes that one),
    before it they are not."""
    ids = torch.randint(0, 1000, (1, tokens), generator=torch.Generator().manual_seed(5))
    cache = target.new_cache(past + tokens)
    cache.ensure(target.num_kv_heads, target.head_dim, target.model.device)
    gen = torch.Generator(device="cuda").manual_seed(6)
    cache.k.normal_(generator=gen)
    cache.vt.normal_(generator=gen)
    out = []
    for mask in (None, torch.ones(tokens, tokens).tril().bool()[None, None]):
        cache.reset()
        cache.advance(past)
        out.append(target(ids, past_key_values=cache, tree_attention_mask=mask).hidden_states)
    assert torch.equal(*out) == decode
    torch.testing.assert_close(out[0].float(), out[1].float(), rtol=0.1, atol=0.1)


def test_prefill_workspace_follows_the_prompts(target):
    """A short prompt does not hold the buffers of a long one; they grow, and results stay."""
    target._pw = None
    ids = torch.randint(0, 1000, (1, 2000), generator=torch.Generator().manual_seed(7))
    first, rows = None, []
    for n in (65, 256, 257, 100, 1024, 2000):
        out = target(ids[:, :n], past_key_values=target.new_cache(n)).hidden_states
        rows.append(target._pw.m_cap)
        first = out if first is None else first
        assert torch.equal(out[:, :65], first)
    assert rows == [256, 256, 1024, 1024, 1024, 2000]

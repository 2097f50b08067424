"""A prompt whose ids lie outside an embedding table is refused before any K/V row is written,
with the ids on the device or on the host; a prompt after it is unaffected."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["device", "host"])
def test_refused_prompt_leaves_the_cache(dev, where):
    from moss_tts_lite_amd.fast import FastDecoder
    from tests._decode_case import build_case, small_config
    cfg = small_config()
    model, _ = build_case(cfg, seed=3, dev=dev)
    dec = FastDecoder(model)
    ids = torch.arange(20).reshape(-1, 1) % cfg.vocab
    ids = ids.to(dev) if where == "device" else ids
    h = dec.prefill_rows(ids).clone()
    k, v = model.k_cache.clone(), model.v_cache.clone()
    for bad in (cfg.vocab, -1):
        wrong = ids.clone()
        wrong[7, 0] = bad
        with pytest.raises(ValueError, match="outside its embedding table"):
            dec.prefill_rows(wrong)
        torch.cuda.synchronize()
        assert torch.equal(model.k_cache, k) and torch.equal(model.v_cache, v)
    assert torch.equal(dec.prefill_rows(ids), h)
    # the ids are read when the call is made: overwriting them afterwards changes nothing
    if where == "device":
        again = ids.clone()
        h2 = dec.prefill_rows(again)
        again.fill_(cfg.vocab + 5)
        torch.cuda.synchronize()
        assert torch.equal(h2, h)


@pytest.mark.parametrize("where", ["device", "host"])
def test_refused_prompt_leaves_the_returned_rows(dev, where):
    # the rows of the last prompt are a view of a buffer: prompts refused after it, of any
    # length, do not write into it, and the next accepted one is right
    from moss_tts_lite_amd.fast import FastDecoder
    from tests._decode_case import build_case, small_config
    cfg = small_config()
    model, _ = build_case(cfg, seed=4, dev=dev)
    dec = FastDecoder(model)
    ids = (torch.arange(20).reshape(-1, 1) * 7 % cfg.vocab).to(dev if where == "device" else "cpu")
    other = (ids + 11) % cfg.vocab
    want = [dec.prefill_rows(t).clone() for t in (ids, other)]
    rows = dec.prefill_rows(ids)
    for length in (20, 5, 20):
        wrong = other[:length].clone()
        wrong[length // 2, 0] = cfg.vocab
        with pytest.raises(ValueError, match="outside its embedding table"):
            dec.prefill_rows(wrong)
        torch.cuda.synchronize()
        assert torch.equal(rows, want[0])
    assert torch.equal(dec.prefill_rows(other), want[1])
    assert torch.equal(dec.prefill_rows(ids), want[0])

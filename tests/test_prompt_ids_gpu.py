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

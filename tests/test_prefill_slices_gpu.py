"""Context encoding behind a cached prefix, where the attention walks slices of the keys in separate work-groups: against the oracle, at lengths around
the edges of tiles (64 keys), query blocks (32) and slices, with 1 .. 8 query heads on a kv head."""
import pytest
import torch

from oracle import DecoderConfig, PagedDecoderOracle
from oracle.synth import make_weights
from tests.helpers import prefill_inputs

pytestmark = pytest.mark.gpu

BS, MAXLEN = 16, 1024


@pytest.mark.parametrize("heads,kv,hd", [(8, 1, 64), (7, 1, 128), (6, 2, 128), (4, 2, 64), (2, 2, 128)])
def test_rest_of_a_prompt_behind_a_cached_prefix(heads, kv, hd):
    from vllm_neuron_amd._native import NativeModel
    cfg = DecoderConfig(num_layers=1, hidden_size=128, num_heads=heads, num_kv_heads=kv, head_dim=hd, intermediate_size=192, vocab_size=256)
    w = make_weights(cfg, seed=2)
    model = NativeModel(num_layers=1, hidden_size=128, num_heads=heads, num_kv_heads=kv, head_dim=hd, intermediate_size=192, vocab_size=256,
                        rms_norm_eps=cfg.rms_norm_eps, rope_theta=cfg.rope_theta, rope_type=0, rope_factor=1.0, num_blocks=1 + MAXLEN // BS,
                        block_size=BS, max_num_seqs=1, max_model_len=MAXLEN, weight_dtype=0, quant_type=0, tp_degree=1, tp_rank=0, device_id=0)
    model.load_state_dict(w)
    model.finalize()
    oracle = PagedDecoderOracle(cfg, w, 1 + MAXLEN // BS, BS, compute="bf16")
    g = torch.Generator().manual_seed(heads * hd)
    prompt = torch.randint(0, 256, (MAXLEN,), generator=g).tolist()
    blocks = (torch.randperm(MAXLEN // BS, generator=g) + 1).tolist()
    first = prefill_inputs(prompt[:MAXLEN], blocks, BS, MAXLEN)
    model.forward(**first)
    oracle.forward(**first)
    # (new tokens, tokens with the prefix): one tile, two, slices that end with a tile, one key into the next, a single query, a ragged block
    for new, full in [(1, 64), (2, 130), (31, 191), (33, 193), (33, 257), (64, 384), (65, 385), (100, 640), (1, 1023), (17, 1000), (130, 1024)]:
        inp = prefill_inputs(prompt[:full], blocks, BS, MAXLEN, full - new)
        got, ref = model.forward(**inp), oracle.forward(**inp)
        assert (got - ref).abs().max().item() < 0.06, (new, full)       # the bar of the model tests: logits of order 4, bf16 rounding points
    model.close()


def _overflowing(cfg, kind):
    """Weights whose `kind` projection of token 255, and of no other, is past what bf16 holds: no other token has feature 0.  Keys and queries get a
    product of +-inf with each other, or NaN where the rotation brings both signs together."""
    w = make_weights(cfg, seed=2)
    embed, proj = w["model.embed_tokens.weight"], w[f"model.layers.0.self_attn.{kind}_proj.weight"]
    embed[:255, 0], embed[255, 0] = 0.0, 4.0
    proj[:, 0] = 2.0 ** 127
    return w


# where the token stands: last (its own query), in the part that is computed, in the cached part behind which slices of their own begin.  The first pair
# of lengths has one slice (a tile of keys), the others two to six.
@pytest.mark.parametrize("kind", ["q", "k", "v"])
@pytest.mark.parametrize("new,full", [(20, 60), (1, 1023), (100, 640), (17, 1000)])
def test_what_is_not_finite_stays_so(kind, new, full):
    cfg = DecoderConfig(num_layers=1, hidden_size=128, num_heads=6, num_kv_heads=2, head_dim=128, intermediate_size=192, vocab_size=256)
    from vllm_neuron_amd._native import NativeModel
    w = _overflowing(cfg, kind)
    model = NativeModel(num_layers=1, hidden_size=128, num_heads=6, num_kv_heads=2, head_dim=128, intermediate_size=192, vocab_size=256,
                        rms_norm_eps=cfg.rms_norm_eps, rope_theta=cfg.rope_theta, rope_type=0, rope_factor=1.0, num_blocks=1 + MAXLEN // BS,
                        block_size=BS, max_num_seqs=1, max_model_len=MAXLEN, weight_dtype=0, quant_type=0, tp_degree=1, tp_rank=0, device_id=0)
    model.load_state_dict(w)
    model.finalize()
    g = torch.Generator().manual_seed(full)
    prompt = torch.randint(0, 255, (full,), generator=g).tolist()
    blocks = (torch.randperm(MAXLEN // BS, generator=g) + 1).tolist()
    for at in {full - 1, full - new, 3, None}:
        seq = [255 if i == at else t for i, t in enumerate(prompt)]
        oracle = PagedDecoderOracle(cfg, w, 1 + MAXLEN // BS, BS, compute="bf16")
        for lo in (0, full - new):
            inp = prefill_inputs(seq[:full] if lo else seq[:full - new], blocks, BS, MAXLEN, lo)
            got, ref = model.forward(**inp), oracle.forward(**inp)
        bad = torch.isnan(ref)
        assert bad.all() or not bad.any()
        assert (kind == "q" and at != full - 1 or at is None) == (not bad.any()), at      # what the test means to ask
        assert torch.equal(torch.isnan(got), bad), at
        if not bad.any():
            assert (got - ref).abs().max().item() < 0.06, at
    model.close()

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

"""Decode attention of short contexts (one work-group per sequence and kv head, no partials) and the change to context splits as a batch outgrows it,
with the captured graph of each form replayed, against the oracle."""
import pytest
import torch

from oracle import PagedDecoderOracle
from oracle.synth import make_weights, zoo_config
from tests.helpers import decode_inputs, prefill_inputs
from tests.test_model_gpu import BS, MAXLEN, MB, NB, native_model

pytestmark = pytest.mark.gpu


# 128-wide heads: the longest of the batch crosses 128 tokens, beside one in its first tile and one at a tile's edge; 64-wide heads: up to the last
# short context (256)
@pytest.mark.parametrize("name,lengths", [("llama31_like", (125, 1, 62)), ("llama31_like", (128, 31, 96)), ("tinyllama_like", (249, 127, 3))])
def test_contexts_around_the_limit(name, lengths):
    cfg = zoo_config(name)
    w = make_weights(cfg, seed=1)
    model, oracle = native_model(cfg, w), PagedDecoderOracle(cfg, w, NB, BS, compute="bf16")
    g = torch.Generator().manual_seed(3)
    blocks = [[1 + i * MB + j for j in range(MB)] for i in range(len(lengths))]
    for i, n in enumerate(lengths):
        inp = prefill_inputs(torch.randint(0, cfg.vocab_size, (n,), generator=g).tolist(), blocks[i], BS, MAXLEN, 0)
        model.forward(**inp)
        oracle.forward(**inp)
    worst = 0.0
    for s in range(6):
        inp = decode_inputs(torch.randint(0, cfg.vocab_size, (len(lengths),), generator=g).tolist(), [n + s for n in lengths], blocks, BS, MAXLEN)
        worst = max(worst, (model.forward(**inp) - oracle.forward(**inp)).abs().max().item())
    assert worst < 0.06, worst            # as the other comparisons with the oracle's bf16 rounding points
    model.close()

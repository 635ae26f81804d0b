"""A prompt's chunk and generating requests in one attention launch (attn_mixed_kernel): where the run of requests stands before or behind the prompt, more
than one of either, contexts of one tile up to several splits, a prompt whose keys go over slices -- against the oracle, request by request."""
import pytest
import torch

import tests.test_model_gpu as M
from oracle import PagedDecoderOracle
from oracle.synth import make_weights, zoo_config
from tests.helpers import prefill_inputs

pytestmark = pytest.mark.gpu
BS, MAXLEN, NSEQ = 32, 768, 6
MB = MAXLEN // BS


# per step: (request, tokens scheduled); lengths already in the cache in front of it
STEPS = [
    ([1, 40, 0], [(0, 1), (1, 1), (2, 33)]),                        # a run, then a prompt; contexts of one tile
    ([600, 128, 129, 700], [(0, 20), (1, 1), (2, 1), (3, 1)]),      # a chunk far into its prompt (slices of its keys), then a run that needs splits
    ([126, 0, 127, 90], [(0, 1), (1, 70), (2, 1), (3, 2)]),         # two runs around a prompt, a second prompt of two tokens
    ([255, 200, 0, 129], [(0, 1), (1, 1), (2, 65), (3, 1)]),        # a tile for each of eight waves
    ([256, 200, 0], [(0, 1), (1, 1), (2, 65)]),                     # one token more
    ([500, 31, 0, 0, 300, 640], [(4, 1), (5, 1), (0, 1), (2, 96), (3, 17), (1, 1)]),
]


@pytest.mark.parametrize("name", ["llama31_like", "tinyllama_like", "qwen25_like"])
@pytest.mark.parametrize("step", range(len(STEPS)))
def test_runs_beside_prompts(monkeypatch, name, step):
    for key, value in dict(BS=BS, MAXLEN=MAXLEN, NSEQ=NSEQ, NB=1 + NSEQ * MB).items():
        monkeypatch.setattr(M, key, value)
    cfg = zoo_config(name)
    w = make_weights(cfg, seed=1)
    model, oracle = M.native_model(cfg, w), PagedDecoderOracle(cfg, w, M.NB, BS, compute="bf16")
    g = torch.Generator().manual_seed(7 + step)
    before, batch = STEPS[step]
    new = dict(batch)
    seqs = [torch.randint(0, cfg.vocab_size, (n + new[r],), generator=g).tolist() for r, n in enumerate(before)]
    blocks = [[1 + i * MB + j for j in range(MB)] for i in range(len(seqs))]
    for r, n in enumerate(before):
        if n:
            inp = prefill_inputs(seqs[r][:n], blocks[r], BS, MAXLEN, 0)
            model.forward(**inp)
            oracle.forward(**inp)
    ids, pos, slots, bt, full, comp = [], [], [], [], [], []
    for r, n in batch:
        lo, hi = before[r], before[r] + n
        ids += seqs[r][lo:hi]
        pos += range(lo, hi)
        slots += [blocks[r][p // BS] * BS + p % BS for p in range(lo, hi)]
        bt.append(blocks[r])
        full.append(hi)
        comp.append(lo)
    got = model.forward_chunked(torch.tensor(ids), torch.tensor(pos), torch.tensor(slots), torch.tensor(bt), torch.tensor(full), torch.tensor(comp))
    worst = 0.0
    for i, (r, n) in enumerate(batch):
        ref = oracle.forward(**prefill_inputs(seqs[r], blocks[r], BS, MAXLEN, before[r]))
        worst = max(worst, (got[i] - ref[0]).abs().max().item())
    assert worst < 0.06, worst            # as the other comparisons with the oracle's bf16 rounding points
    model.close()


# the splits of a run are merged by the work-group that ends last, which leaves the counters as it found them: a batch gives the same numbers again, whatever runs between
@pytest.mark.parametrize("rows", [1, 5])
def test_merged_splits_again(monkeypatch, rows):
    for key, value in dict(BS=BS, MAXLEN=MAXLEN, NSEQ=NSEQ, NB=1 + NSEQ * MB).items():
        monkeypatch.setattr(M, key, value)
    cfg = zoo_config("llama31_like")
    model = M.native_model(cfg, make_weights(cfg, seed=1))
    g = torch.Generator().manual_seed(rows)
    seqs = [torch.randint(0, cfg.vocab_size, (700 - 3 * r,), generator=g).tolist() for r in range(6)]
    blocks = [[1 + i * MB + j for j in range(MB)] for i in range(6)]
    for r in range(6):
        model.forward(**prefill_inputs(seqs[r], blocks[r], BS, MAXLEN, 0))

    def call(run, chunk):
        batch = [(r, len(seqs[r]) - 1, len(seqs[r])) for r in run] + [(5, 0, chunk)]
        ids = [t for r, lo, hi in batch for t in seqs[r][lo:hi]]
        pos = [p for r, lo, hi in batch for p in range(lo, hi)]
        slots = [blocks[r][p // BS] * BS + p % BS for r, lo, hi in batch for p in range(lo, hi)]
        return model.forward_chunked(torch.tensor(ids), torch.tensor(pos), torch.tensor(slots), torch.tensor([blocks[r] for r, _, _ in batch]),
                                     torch.tensor([hi for _, _, hi in batch]), torch.tensor([lo for _, lo, _ in batch]))
    first, other = call(range(rows), 40), call([2], 70)
    assert torch.isfinite(first).all()
    for _ in range(20):
        assert torch.equal(first, call(range(rows), 40)) and torch.equal(other, call([2], 70))
    model.close()

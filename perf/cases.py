"""What is measured: model calls as a serving loop makes them -- context encoding of one prompt, one token-generation step of a batch, one
ragged batch of a prompt chunk beside generating requests -- through `vllm_neuron_amd._native.NativeModel`, the object the plugin's model
runner drives.  Inputs are the host tensors vLLM hands over, outputs the fp32 logits it samples from (in the library's pinned buffer where the
runner reads them there).  Weights are seeded random numbers at the real shapes: N(0, 0.02) matrices, quantized by the library where the case
says so; `Weights` restates them for `exact`.

Families: Llama-style decoders (bf16, fp8 and int8 weights), and the four layer-stack designs, all bf16.  The 7b and 8b models have half of their
layers: with random weights the rounding of bf16 inputs alone puts two correct answers 2 - 3 % apart behind all 32.  For the same reason two options
are left out whose answers no tolerance could compare: experts (a token whose ninth is almost its eighth may take either) and fp8 activations
(an early value that rounds to the other side moves all later ones).  A generated token is written to its
own place in the cache before it is read, so a pass repeats on the same state; recurrent mixers (delta rule, Mamba-2, selective scan) advance
their state, so those are measured on prompts, which start from a zero state.
"""
import math
from types import SimpleNamespace

import torch

from vllm_neuron_amd._native import MI_Q, MI_W, NativeModel
from vllm_neuron_amd.models import config_from_dict, fill_sizes
from vllm_neuron_amd.worker.mi355x_model_loader import _decoder_geometry

BLOCK, STD = 32, 0.02
LLAMA3_ROPE = {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0, "original_max_position_embeddings": 8192}


def _hf(kind, vocab, width, inter, layers, heads, kv_heads, dim, eps, theta, scaling=None):
    return dict(model_type=kind, vocab_size=vocab, hidden_size=width, intermediate_size=inter, num_hidden_layers=layers, num_attention_heads=heads,
                num_key_value_heads=kv_heads, head_dim=dim, rms_norm_eps=eps, rope_theta=theta, rope_scaling=scaling, tie_word_embeddings=False)


LLAMAS = {
    "tinyllama_1b": _hf("llama", 32000, 2048, 5632, 22, 32, 4, 64, 1e-5, 1e4),
    "llama31_8b": _hf("llama", 128256, 4096, 14336, 16, 32, 8, 128, 1e-5, 5e5, LLAMA3_ROPE),
    "qwen25_7b": _hf("qwen2", 152064, 3584, 18944, 14, 28, 4, 128, 1e-6, 1e6),
}
LLAMA_LEN, BUCKETS = 2048, [256, 512, 1024, 2048]

STACK_VOCAB, STACK_LEN, WINDOW, LOW_RANK, BIAS_ROWS = 32768, 4096, 1024, 128, 32


def _stack(architecture, layer, layers=8, **extra):
    return {"architecture": architecture, "width": 2048, "vocab": STACK_VOCAB, "norm": {"eps": 1e-5}, "layers": [layer] * layers, **extra}


STACKS = {
    # grouped heads, distance slopes, window, squared-relu feed-forward
    "vimesun": _stack("Vimesun", {"type": "attention", "mixer": {"heads": 32, "kv_heads": 8, "dim": 64, "vdim": 64, "mask": {"size": WINDOW},
                                                                  "scale": 0.125}, "mlp": {"kind": "dense", "ff": 12288}},
                      residual_mult=0.5, max_positions=STACK_LEN),
    # latent attention and short convolutions, clipped gated feed-forward
    "rapodra": _stack("Rapodra", {"type": "latent_attention", "mixer": {"heads": 16, "dim": 128, "vdim": 128, "kv_rank": 512,
                                                                        "mask": {"size": WINDOW}, "scale": 128 ** -0.5},
                                  "mlp": {"kind": "dense", "ff": 7680, "limit": 7.0}},
                      canon={"taps": 4}, norm={"eps": 1e-5, "groups": 4}, logit_softcap=30.0),
    # gated delta rule
    "bokulorn": _stack("Bokulorn", {"type": "channel_delta", "mixer": {"heads": 16, "kv_heads": 16, "dim": 128, "vdim": 128, "conv": 4},
                                    "mlp": None}, embedding={"scale": 1.0}),
    # attention in chunks beside a Mamba-2 mixer
    "nusovik": _stack("Nusovik", {"type": "parallel", "mixer": {
        "left": {"heads": 32, "kv_heads": 8, "dim": 64, "vdim": 64, "scale": 0.125, "mask": {"size": WINDOW}, "bias_max": WINDOW // 2},
        "right": {"heads": 64, "vdim": 64, "state": 128, "groups": 1, "norm_groups": 1, "conv": 4}, "left_scale": 1.0, "right_scale": 1.0},
        "mlp": {"kind": "dense", "ff": 12288}}, embedding={"scale": 1.0}, logit_scale=1.0),
}
RECURRENT = ("bokulorn", "nusovik")


# ---- the cases ------------------------------------------------------------------------------------------------------------------------
# call "decode": `rows` sequences generate one token each, their contexts between `short` and `long` tokens;  "prefill": one prompt of
# `tokens`, the first `cached` of them already in the cache;  "chunk": a prompt chunk of `tokens` beside `rows` generating requests.
def _llama(model, weights, **case):
    return dict(model=model, weights=weights, **case)


def listed():
    return [
        # the smallest call: one short chat of a small model, a chain of short launches
        dict(_llama("tinyllama_1b", "bf16", call="decode", rows=1, short=40, long=40), name="decode 1b bf16, 1 row"),
        # the headline: four sequences of 1024 tokens, fp8 weights
        dict(_llama("llama31_8b", "f8e4m3", call="decode", rows=4, short=1024, long=1024), name="decode 8b fp8, 4 rows"),
        # a full batch (the default max_num_seqs) of uneven contexts
        dict(_llama("llama31_8b", "f8e4m3", call="decode", rows=32, short=37, long=1000), name="decode 8b fp8, 32 rows"),
        # int8 weights and qkv biases, an odd batch of uneven contexts
        dict(_llama("qwen25_7b", "int8", call="decode", rows=5, short=300, long=1900), name="decode 7b int8, 5 rows"),
        # the longest prompt of the largest bucket
        dict(_llama("llama31_8b", "f8e4m3", call="prefill", tokens=2031, cached=0), name="prefill 8b fp8, 2031"),
        # the same model unquantized, an odd length
        dict(_llama("llama31_8b", "bf16", call="prefill", tokens=1000, cached=0), name="prefill 8b bf16, 1000"),
        # int8 weights, most of the prompt found in the prefix cache: a short, ragged rest
        dict(_llama("qwen25_7b", "int8", call="prefill", tokens=700, cached=512), name="prefill 7b int8, 188 of 700"),
        # chunked prefill: a chunk of a prompt in the same batch as three requests that generate
        dict(_llama("llama31_8b", "f8e4m3", call="chunk", tokens=239, rows=3, short=500, long=900), name="chunk 8b fp8, 239 + 3"),
        # the layer-stack designs: long windowed prompt, token generation over latents, delta-rule prompt, Mamba-2 prompt
        dict(model="vimesun", weights="bf16", call="prefill", tokens=4000, cached=0, name="prefill vimesun, 4000"),
        dict(model="rapodra", weights="bf16", call="decode", rows=4, short=600, long=1500, name="decode rapodra, 4 rows"),
        dict(model="bokulorn", weights="bf16", call="prefill", tokens=2048, cached=0, name="prefill bokulorn, 2048"),
        dict(model="nusovik", weights="bf16", call="prefill", tokens=777, cached=0, name="prefill nusovik, 777"),
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.65:
        case = _llama(rng.choice(list(LLAMAS)), rng.choice(["bf16", "f8e4m3", "int8"]))
        most, call = 1500 if case["weights"] == "bf16" else LLAMA_LEN - 17, rng.choice(["decode", "prefill", "prefill", "chunk"])
        rows = _between(rng, 1, 32) if call == "decode" else rng.randint(1, 6)
    else:
        case = dict(model=rng.choice(list(STACKS)), weights="bf16")
        most, call = 4000, "prefill" if case["model"] in RECURRENT else rng.choice(["decode", "prefill"])
        rows = _between(rng, 1, 32)
    if call == "prefill":
        tokens = _between(rng, 17, most)
        cached = tokens // 2 // BLOCK * BLOCK if case["model"] in LLAMAS and rng.random() < 0.3 else 0
        return dict(case, call=call, tokens=tokens, cached=cached)
    long = min(_between(rng, 24, 2000), 16000 // rows)
    short = rng.randint(16, long)
    if call == "decode":
        return dict(case, call=call, rows=rows, short=short, long=long)
    return dict(case, call=call, tokens=_between(rng, 33, 1000), rows=rows, short=short, long=long)


# ---- weights: the library's counter-based N(0, std), restated for exact() ------------------------------------------------------------------
def _signed(x):
    return x - (1 << 64) if x >= 1 << 63 else x


def _shr(x, n):
    return (x >> n) & ((1 << (64 - n)) - 1)


def _mix(x):
    x = x + _signed(0x9E3779B97F4A7C15)
    x = (x ^ _shr(x, 30)) * _signed(0xBF58476D1CE4E5B9)
    x = (x ^ _shr(x, 27)) * _signed(0x94D049BB133111EB)
    return x ^ _shr(x, 31)


def _bf16(x):
    return x.to(torch.bfloat16).to(x.dtype)


class Weights:
    """Tensors in the order in which the library numbers them; float64 on the GPU, of the values the device holds."""

    def __init__(self, seed, kind="bf16"):
        self.seed, self.next, self.kind = seed, 1, kind

    def skip(self, n=1):
        self.next += n

    def plain(self, rows, cols, std):
        i = torch.arange(rows * cols, device="cuda", dtype=torch.int64) + _signed(self.next * 0x100000001B3 % (1 << 64))
        self.next += 1
        r = _mix(_mix(i) ^ self.seed)
        u1, u2 = (_shr(r, 40) + 1).double() / 16777217.0, (r & 0xFFFFFF).double() / 16777216.0
        return (std * torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(2.0 * math.pi * u2)).float().reshape(rows, cols)

    def bf16(self, rows, cols, std=STD):
        return _bf16(self.plain(rows, cols, std)).double()

    def f32(self, rows, cols, std=STD):
        return self.plain(rows, cols, std).double()

    def matrix(self, rows, cols):
        if self.kind == "bf16":
            return self.bf16(rows, cols)
        w, top = self.plain(rows, cols, STD), 448.0 if self.kind == "f8e4m3" else 127.0
        scale = w.abs().amax(1, keepdim=True) / top
        q = (w / scale).clamp(-top, top)
        return (q.to(torch.float8_e4m3fn).double() if self.kind == "f8e4m3" else torch.round(q).double()) * scale.double()


# ---- state --------------------------------------------------------------------------------------------------------------------------------
def _sequences(case, seed):
    """-> ([tokens of every sequence], new tokens of every sequence): the last of each is what logits are asked of"""
    g = torch.Generator().manual_seed(seed)
    vocab = LLAMAS[case["model"]]["vocab_size"] if case["model"] in LLAMAS else STACK_VOCAB

    def ids(n):
        return torch.randint(0, vocab, (n,), generator=g)
    if case["call"] == "prefill":
        return [ids(case["tokens"])], [case["tokens"] - case["cached"]]
    lens = [case["short"] + (case["long"] - case["short"]) * i // max(case["rows"] - 1, 1) for i in range(case["rows"])]
    order = torch.randperm(len(lens), generator=g).tolist()
    seqs, new = [ids(lens[i]) for i in order], [1] * len(lens)
    return ([ids(case["tokens"])] + seqs, [case["tokens"]] + new) if case["call"] == "chunk" else (seqs, new)


def _model(case, seqs):
    length = LLAMA_LEN if case["model"] in LLAMAS else STACK_LEN
    common = dict(num_blocks=1 + seqs * (length // BLOCK), block_size=BLOCK, max_num_seqs=4 if seqs <= 4 else 32,
                  max_model_len=length, device_id=0, use_graphs=1)
    if case["model"] in LLAMAS:
        quant = dict(weight_dtype=MI_W[case["weights"]], quant_type=MI_Q["per_channel_symmetric"],
                     quantize_lm_head=int(case["weights"] != "bf16"), prefill_fp8_activations=0)
        return NativeModel(**common, **quant, tp_degree=1, tp_rank=0, ctx_buckets=BUCKETS,
                           **_decoder_geometry(SimpleNamespace(**LLAMAS[case["model"]])))
    config = config_from_dict(STACKS[case["model"]])
    fill_sizes(config, lambda name: (BIAS_ROWS if name.endswith("rel") else LOW_RANK, 2048))
    return NativeModel(stack=dict(config.stack, compute_dtype=1), ctx_buckets=[length], **common)


def _call(seqs, tables, new):
    """The runner's tensors for one call over `seqs`, of which the last new[i] tokens are computed."""
    slots = [[int(tables[i][p // BLOCK]) * BLOCK + p % BLOCK for p in range(len(s) - n, len(s))] for i, (s, n) in enumerate(zip(seqs, new))]
    return dict(block_table=tables, full_context_lens=torch.tensor([len(s) for s in seqs]),
                computed_context_lens=torch.tensor([len(s) - n for s, n in zip(seqs, new)])), slots


def prepare(case, seed):
    seqs, new = _sequences(case, seed)
    model = _model(case, len(seqs))
    model.init_synthetic_weights(seed, STD)
    model.finalize()
    length = model.cfg.max_model_len
    free = torch.randperm(model.cfg.num_blocks - 1, generator=torch.Generator().manual_seed(seed)) + 1
    tables = torch.zeros(len(seqs), length // BLOCK, dtype=torch.long)
    for i, s in enumerate(seqs):
        n = -(-len(s) // BLOCK)
        tables[i, :n], free = free[:n], free[n:]

    def whole(i, n):                                # context encoding of the first n tokens of sequence i, `behind` of them cached
        inputs, slots = _call([seqs[i][:n]], tables[i:i + 1], [n])
        return dict(inputs, input_ids=seqs[i][None, :n], position_ids=torch.arange(n)[None], seq_ids=torch.tensor([i]),
                    slot_mapping=torch.tensor(slots))
    for i, (s, n) in enumerate(zip(seqs, new)):     # what earlier calls left in the cache
        if n < len(s):
            model.forward(**whole(i, len(s) - n), alias_ok=True)
    if case["call"] == "prefill":
        s, done = seqs[0], case["cached"]
        inputs = whole(0, len(s))
        inputs.update(computed_context_lens=torch.tensor([done]), slot_mapping=inputs["slot_mapping"][:, done:].contiguous())
        return SimpleNamespace(model=model, call=model.forward, inputs=dict(inputs, alias_ok=True))
    inputs, slots = _call(seqs, tables, new)
    if case["call"] == "decode":
        inputs.update(input_ids=torch.stack([s[-1:] for s in seqs]), position_ids=torch.tensor([[len(s) - 1] for s in seqs]),
                      seq_ids=torch.arange(len(seqs)), slot_mapping=torch.tensor(slots))
        return SimpleNamespace(model=model, call=model.forward, inputs=dict(inputs, alias_ok=True))
    inputs.update(input_ids=torch.cat([s[len(s) - n:] for s, n in zip(seqs, new)]), seq_ids=torch.arange(len(seqs)),
                  position_ids=torch.cat([torch.arange(len(s) - n, len(s)) for s, n in zip(seqs, new)]),
                  slot_mapping=torch.tensor([x for row in slots for x in row]))
    return SimpleNamespace(model=model, call=model.forward_chunked, inputs=inputs)


def run(state):
    logits = state.call(**state.inputs)
    logits.model = state.model      # a view of the model's own buffer, where it is one, lasts as long as that
    return logits


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------------------------
def _layer_sizes(model):
    """-> (weight numbers, flops per attended key, cache numbers per token) of a layer"""
    if model in LLAMAS:
        m = LLAMAS[model]
        q, kv, width = m["num_attention_heads"] * m["head_dim"], m["num_key_value_heads"] * m["head_dim"], m["hidden_size"]
        return width * (2 * q + 2 * kv + 3 * m["intermediate_size"]), 4 * q, 2 * kv
    width = 2048
    return {"vimesun": (width * (2 * 32 + 2 * 8) * 64 + 2 * width * 12288, 4 * 2048, 2 * 512),
            "rapodra": (width * (2048 + 512) + 2048 * width + 2 * 512 * 2048 + 3 * width * 7680, 4 * 2048, 512),
            "bokulorn": (width * (4 * 2048 + 16 + 2 * LOW_RANK) + 2 * LOW_RANK * 2048, 0, 0),
            "nusovik": (width * (2 * 2048 + 512 + 32 + 2 * 4096 + 256 + 64 + 4096 + 2 * 12288), 4 * 2048, 2 * 512)}[model]


def work(case):
    seqs, new = _sequences(case, 0)
    model, llama = case["model"], case["model"] in LLAMAS
    layers = LLAMAS[model]["num_hidden_layers"] if llama else 8
    width, vocab = (LLAMAS[model]["hidden_size"], LLAMAS[model]["vocab_size"]) if llama else (2048, STACK_VOCAB)
    size = 2 if case["weights"] == "bf16" else 1
    tokens = sum(new)
    weights, pair, cache = _layer_sizes(model)
    window = 1 << 30 if llama else WINDOW
    pairs = keys = 0
    for s, n in zip(seqs, new):
        pairs += sum(min(i + 1, window) for i in range(len(s) - n, len(s)))
        keys += min(len(s), window + n - 1)
    recurrence = {"bokulorn": 6 * 16 * 128 * 128, "nusovik": 4 * 64 * 64 * 128}.get(model, 0)
    return {"bytes": size * (layers * weights + vocab * width) + 2 * layers * cache * (keys + tokens) + 2 * tokens * width + 4 * len(seqs) * vocab,
            "flops": layers * (2 * weights * tokens + pair * pairs + recurrence * tokens) + 2 * vocab * width * len(seqs)}


def tolerance(case):
    # four times the distance to exact() (16 layers of 4096 wide: 1.1 - 1.5 %; 22 of 2048: 0.8 %; vimesun 0.4, rapodra 0.6, bokulorn 0.3, nusovik 0.9 - 1.6 %), 3 % at most
    return {"rel": {"vimesun": 0.018, "rapodra": 0.024, "bokulorn": 0.012}.get(case["model"], 0.03)}


# ---- the same logits in 64 bits ---------------------------------------------------------------------------------------------------------------
def _rms(x, eps):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _attend(q, k, v, scale, window=1 << 30, chunk=0, bias=None, sink=None):
    """q [T, H, d], k, v [T, G, d] of one sequence; bias(head, distances) joins the scores, exp(sink[h]) the denominator."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
    at = torch.arange(T, device=q.device)
    dist = at[:, None] - at[None, :]
    hidden = (dist < 0) | (dist >= window)
    if chunk:
        hidden |= at[:, None] // chunk != at[None, :] // chunk
    for h in range(H):
        s = (q[:, h] @ k[:, h * G // H].t()) * scale
        if bias is not None:
            s = s + bias(h, dist)
        s = s.masked_fill(hidden, -math.inf)
        if sink is None:
            out[:, h] = torch.softmax(s, -1) @ v[:, h * G // H]
        else:
            out[:, h] = torch.softmax(torch.cat([s, sink[h].expand(T, 1)], 1), -1)[:, :-1] @ v[:, h * G // H]
    return out


def _per_sequence(f, lens, *parts):
    return torch.cat([f(*x) for x in zip(*(p.split(lens) for p in parts))])


def _rotation(m, positions):
    d = m["head_dim"]
    freq = m["rope_theta"] ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
    r = m["rope_scaling"]
    if r:
        length = 2 * math.pi / freq
        low, high, old = r["low_freq_factor"], r["high_freq_factor"], r["original_max_position_embeddings"]
        blend = ((old / length - low) / (high - low)).clamp(0, 1)
        freq = (1 - blend) * freq / r["factor"] + blend * freq
    a = positions.double()[:, None] * freq
    c, s = a.cos()[:, None], a.sin()[:, None]

    def turn(x):
        u, v = x[..., :d // 2], x[..., d // 2:]
        return torch.cat([u * c - v * s, v * c + u * s], -1)
    return turn


def _exact_llama(case, seed, tokens, lens, last):
    m, w = LLAMAS[case["model"]], Weights(seed, case["weights"])
    width, hd, eps, inter = m["hidden_size"], m["head_dim"], m["rms_norm_eps"], m["intermediate_size"]
    H, G = m["num_attention_heads"], m["num_key_value_heads"]
    turn = _rotation(m, torch.cat([torch.arange(n, device="cuda") for n in lens]))
    x = w.bf16(m["vocab_size"], width, 1.0)[tokens]
    for _ in range(m["num_hidden_layers"]):
        h = _rms(x, eps)
        q, k, v = (h @ w.matrix(n * hd, width).t() for n in (H, G, G))
        wo, gate, up, down = (w.matrix(*s) for s in ((width, H * hd), (inter, width), (inter, width), (width, inter)))
        if m["model_type"] == "qwen2":
            q, k, v = (y + w.f32(1, y.shape[1], 0.25) for y in (q, k, v))
        q, k, v = turn(q.unflatten(1, (H, hd))), turn(k.unflatten(1, (G, hd))), v.unflatten(1, (G, hd))
        x = x + _per_sequence(lambda a, b, c: _attend(a, b, c, hd ** -0.5), lens, q, k, v).flatten(1) @ wo.t()
        h = _rms(x, eps)
        x = x + (torch.nn.functional.silu(h @ gate.t()) * (h @ up.t())) @ down.t()
    return _rms(x[last], eps) @ w.matrix(m["vocab_size"], width).t()


def _conv(x, taps):
    """sum_j taps[:, j] x_(t - n + 1 + j), zeros ahead of the sequence"""
    n, T = taps.shape[1], x.shape[0]
    padded = torch.cat([x.new_zeros(n - 1, x.shape[1]), x])
    return sum(taps[:, j] * padded[j:j + T] for j in range(n))


def _vimesun(x, w, lens):
    n1 = torch.nn.functional.layer_norm(x, (2048,), eps=1e-5)
    w.skip(2)
    q, k, v = (n1 @ w.bf16(n * 64, 2048).t() for n in (32, 8, 8))
    slopes = [2.0 ** (-8.0 * (h + 1) / 32) for h in range(32)]
    zero = torch.zeros(32, dtype=torch.float64, device="cuda")
    o = _per_sequence(lambda *p: _attend(*p, 0.125, WINDOW, 0, lambda h, d: -slopes[h] * d, zero), lens, _rms(q.unflatten(1, (32, 64)), 1e-5),
                      _rms(k.unflatten(1, (8, 64)), 1e-5), v.unflatten(1, (8, 64)))
    y = o.flatten(1) @ w.bf16(2048, 2048).t()
    w.skip(2)
    up, down = w.bf16(12288, 2048), w.bf16(2048, 12288)
    return x + 0.5 * (y + (n1 @ up.t()).clamp(min=0).pow(2) @ down.t())


def _group_rms(x):
    return _rms(x.unflatten(1, (4, 512)), 1e-5).flatten(1)


def _rapodra(x, w, lens):
    def mixed(x, taps):
        return _per_sequence(lambda h: h + _conv(h, taps), lens, _group_rms(x))
    w.skip(2)
    h = mixed(x, w.f32(2048, 4, 0.3))
    q, uk, uv, wo = h @ w.bf16(2048, 2048).t(), w.bf16(2048, 512), w.bf16(2048, 512), w.bf16(2048, 2048)
    c = _rms(h @ w.bf16(512, 2048).t(), 1e-5)
    w.skip()
    k, v = c @ uk.t(), c @ uv.t()
    o = _per_sequence(lambda *p: _attend(*p, 128 ** -0.5, WINDOW), lens, *(y.unflatten(1, (16, 128)) for y in (q, k, v)))
    x = x + _group_rms(o.flatten(1) @ wo.t())
    w.skip(2)
    h = mixed(x, w.f32(2048, 4, 0.3))
    gate, up, down = w.bf16(7680, 2048), w.bf16(7680, 2048), w.bf16(2048, 7680)
    g, u = (h @ gate.t()).clamp(max=7.0), (h @ up.t()).clamp(-7.0, 7.0)
    return x + _group_rms((g * torch.sigmoid(1.702 * g) * (u + 1)) @ down.t())


def _bokulorn(x, w, lens):
    H, d = 16, 128
    w.skip()
    h, T = _rms(x, 1e-5), x.shape[0]
    q, k, v = (torch.nn.functional.silu(_conv(h @ w.bf16(2048, 2048).t(), w.f32(2048, 4, 0.3))).unflatten(1, (H, d)) for _ in range(3))
    q, k = (y / torch.sqrt(y.pow(2).sum(-1, keepdim=True) + 1e-6) for y in (q, k))
    beta = torch.sigmoid(h @ w.bf16(H, 2048).t())
    w.skip()
    low = h @ w.bf16(LOW_RANK, 2048).t()
    keep = torch.exp(-torch.nn.functional.softplus(low @ w.bf16(2048, LOW_RANK).t())).unflatten(1, (H, d))
    w.skip()
    low = h @ w.bf16(LOW_RANK, 2048).t()
    gate = torch.sigmoid(low @ w.bf16(2048, LOW_RANK).t())
    w.skip()
    S, o = torch.zeros(H, d, d, dtype=torch.float64, device="cuda"), torch.empty_like(q)
    for t in range(T):
        S = keep[t, :, :, None] * S
        u = beta[t, :, None] * (v[t] - (k[t, :, None] @ S)[:, 0])
        S = S + k[t, :, :, None] * u[:, None]
        o[t] = (q[t, :, None] @ S)[:, 0]
    y = (_rms(o * d ** -0.5, 1e-5).flatten(1) * gate) @ w.bf16(2048, 2048).t()
    return x + y


def _nusovik(x, w, lens):
    T, eps = x.shape[0], 1e-5
    w.skip(2)
    up, down = w.bf16(12288, 2048), w.bf16(2048, 12288)
    z, xbc, dt = (x @ w.bf16(2 * 4096 + 256 + 64, 2048).t()).split([4096, 4096 + 256, 64], 1)
    xbc = torch.nn.functional.silu(_conv(xbc, w.f32(4096 + 256, 4, 0.3)))
    w.skip(5)                                       # its biases, decays, skip weights (zero) and norm (one)
    xs, b, c = xbc.split([4096, 128, 128], 1)
    xs, dt = xs.unflatten(1, (64, 64)), torch.nn.functional.softplus(dt)
    S, y = torch.zeros(64, 128, 64, dtype=torch.float64, device="cuda"), torch.empty_like(xs)
    for t in range(T):
        S = torch.exp(-dt[t])[:, None, None] * S + b[t, :, None] * (dt[t, :, None] * xs[t])[:, None]
        y[t] = (c[t, None, None] @ S)[:, 0]
    right = _rms(y.flatten(1) * torch.nn.functional.silu(z), eps) @ w.bf16(2048, 4096).t()
    q, k = (x @ w.bf16(n * 64, 2048).t() for n in (32, 8))
    wo = w.bf16(2048, 2048)
    w.skip(4)                                       # q and k: biases, norms
    gate = torch.sigmoid(x @ w.bf16(32, 2048).t())
    w.skip()                                        # sinks
    table = w.f32(BIAS_ROWS, 32)
    half, far = BIAS_ROWS // 2, WINDOW // 2
    n = torch.arange(WINDOW, dtype=torch.float64)
    rows = torch.where(n < half, n, half + torch.floor(torch.log(n.clamp(min=1) / half) / math.log(far / half) * half + 1e-9))
    rows = rows.clamp(max=BIAS_ROWS - 1).long().cuda()
    k, q = k.unflatten(1, (8, 64)), q.unflatten(1, (32, 64))
    o = _attend(_rms(q, eps), _rms(k, eps), k, 0.125, chunk=WINDOW, bias=lambda h, d: table[:, h][rows[d.clamp(0, WINDOW - 1)]],
                sink=torch.zeros(32, dtype=torch.float64, device="cuda"))
    x = x + _rms((o * gate[:, :, None]).flatten(1) @ wo.t() + right, eps)
    return x + _rms((x @ up.t()).clamp(min=0).pow(2) @ down.t(), eps)


def _exact_stack(case, seed, tokens, lens, last):
    w, model = Weights(seed), case["model"]
    x = w.bf16(STACK_VOCAB, 2048, 1.0)[tokens]
    at = torch.cat([torch.arange(n, device="cuda") for n in lens])
    if model == "vimesun":
        x = x + w.bf16(STACK_LEN, 2048, 0.1)[at]
    elif model == "nusovik":
        e = torch.arange(2048, device="cuda")
        a = at.double()[:, None] * 10000.0 ** (-2.0 * (e // 2).double() / 2048)
        x = x + torch.where(e % 2 == 0, torch.sin(a), torch.cos(a))
    step = {"vimesun": _vimesun, "rapodra": _rapodra, "bokulorn": _bokulorn, "nusovik": _nusovik}[model]
    for _ in range(8):
        x = step(x, w, lens)
    w.skip()
    x = x[last]
    x = {"vimesun": lambda: torch.nn.functional.layer_norm(x, (2048,), eps=1e-5), "rapodra": lambda: _group_rms(x)}.get(
        model, lambda: _rms(x, 1e-5))()
    z = x @ w.bf16(STACK_VOCAB, 2048).t()
    return 30.0 * torch.tanh(z / 30.0) if model == "rapodra" else z


@torch.no_grad()
def exact(case, seed):
    seqs, _ = _sequences(case, seed)
    lens = [len(s) for s in seqs]
    last = torch.tensor(lens, device="cuda").cumsum(0) - 1
    return (_exact_llama if case["model"] in LLAMAS else _exact_stack)(case, seed, torch.cat(seqs).cuda(), lens, last).cpu()

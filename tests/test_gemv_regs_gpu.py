"""Token generation of 5 .. 32 rows: the weight stream with the activations in registers (gemv_regs_kernel) at the edges of its splits, and the
sums it leaves to the next norm inside the models."""
import os
import subprocess
import sys

import pytest
import torch

from oracle.quant import dequantize_weight, quantize_weight
from tests.test_ops_gpu import WD, dev, quantize_on_device

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    from vllm_neuron_amd import _native
    _native.load_library()
    return _native


# rows: the first and last of each column group; K: fewer k-tiles than waves, an odd share per wave, the first beyond 4 / 8 / 16 tiles a wave, two to eight
# slices of uneven length, one k-tile more than eight slices hold (the kernels of 16 rows, and the GEMM); N: one row-tile, one more than the CUs, several
# passes, more than the passes whose scales fit
@pytest.mark.parametrize("wd", ["bf16", "f8e4m3", "int8"])
@pytest.mark.parametrize("M", [5, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(16, 64), (4112, 320), (272, 1088), (528, 2112), (144, 4096), (48, 4160), (2048, 6208), (16, 28672), (263680, 64), (8208, 1152), (32, 32832)])
def test_edges_of_the_register_gemv(lib, wd, M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    w = torch.randn(N, K, generator=g) * 0.05
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    bias = torch.randn(N, generator=g) * 0.1
    tiled, scale = quantize_on_device(lib, w, wd, "per_channel_symmetric")
    wq = w.to(torch.bfloat16).float() if wd == "bf16" else dequantize_weight(*quantize_weight(w, wd, "per_channel_symmetric"))
    ref = x.double() @ wq.double().t() + bias.double()
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    xd, bd = dev(x), dev(bias)
    lib.check(lib.load_library().mi_op_qlinear(xd.data_ptr(), M, tiled.data_ptr(), scale.data_ptr(), bd.data_ptr(), N, K, WD[wd], y.data_ptr(), 8, None))
    torch.cuda.synchronize()
    err = (y.cpu().double() - ref).abs().max().item()
    tol = 2e-5 * ref.abs().max().item() + 1e-5 * (K ** 0.5)     # as the other linear tests: fp32 sums in another order
    assert err < tol, (err, tol)


# every number of k-tiles a wave holds that has a kernel of its own, whole and with a last tile or whole waves missing (one-byte weights 5 .. 8, bf16 5 .. 8, 12, 14, 16)
@pytest.mark.parametrize("wd", ["bf16", "f8e4m3", "int8"])
@pytest.mark.parametrize("M", [5, 32])
@pytest.mark.parametrize("N,K", [(4096, K) for K in (1088, 1536, 1600, 1792, 1856, 2048, 2112, 2560, 2624, 3072, 3136, 3584, 3648, 4096)])
def test_k_tiles_of_a_wave(lib, wd, M, N, K):
    test_edges_of_the_register_gemv(lib, wd, M, N, K)


# up to 4 rows, where they go there: one row-tile a work-group, eight and more, one k-tile fewer than a wave has registers for, and one more (the LDS kernels)
@pytest.mark.parametrize("wd", ["bf16", "f8e4m3", "int8"])
@pytest.mark.parametrize("M", [1, 3, 4])
@pytest.mark.parametrize("N,K", [(16, 64), (4096, 320), (4112, 320), (272, 2048), (528, 2112), (48, 4096), (48, 4160), (32768, 128)])
def test_edges_of_few_rows(lib, wd, M, N, K):
    test_edges_of_the_register_gemv(lib, wd, M, N, K)


# up to 4 rows in the LDS kernels with K over the waves: batches of 5 .. 8 tiles, whole, and with tiles of the last wave missing; one and several passes; K beyond 16384
# and what the LDS holds: activations beside the weights, an odd and an even number of sub-chunks, waves with a part of one and with none of the last
@pytest.mark.parametrize("wd", ["bf16", "f8e4m3", "int8"])
@pytest.mark.parametrize("M", [1, 4])
@pytest.mark.parametrize("N,K", [(16, 4608), (4112, 5632), (144, 5568), (272, 6656), (4096, 7168), (16, 7104), (48, 9216), (4112, 14336), (528, 14272), (16, 16384), (48, 16448), (4112, 17472), (16, 18944), (8208, 20480), (272, 28672)])
def test_batches_of_the_few_row_kernels(lib, wd, M, N, K):
    test_edges_of_the_register_gemv(lib, wd, M, N, K)


def _quant(wd):
    return None if wd == "bf16" else dict(quantized=True, quantization_dtype=wd, quantization_type="per_channel_symmetric")


# ... with the norms in front, where slices of 2 .. 16 tiles go to 1, 2, 4 and 8 waves: against the oracle, at the bar of the other dispatch tests, and against 5 rows, whose weights the
# register kernel reads (the same products in another order; bf16 roundings of the activations in between make 2^-8 of a value, and as between any two kernels of this file 5 % of the spread
# is far beyond)
@pytest.mark.parametrize("wd", ["bf16", "f8e4m3", "int8"])
@pytest.mark.parametrize("hidden,inter,vocab", [(1024, 1088, 16), (1280, 6208, 12304), (2048, 5632, 32000), (2304, 2112, 8208), (3584, 4736, 16400), (4096, 14336, 4112)])
def test_norms_in_front_of_few_rows(wd, hidden, inter, vocab):
    from oracle import DecoderConfig, PagedDecoderOracle
    from oracle.synth import make_weights
    from tests.helpers import decode_inputs
    from vllm_neuron_amd._native import MI_Q, MI_W, NativeModel
    shape = dict(num_layers=1, hidden_size=hidden, num_heads=hidden // 64, num_kv_heads=hidden // 256, head_dim=64, intermediate_size=inter, vocab_size=vocab)
    cfg = DecoderConfig(**shape)
    w = make_weights(cfg, seed=4)
    model = NativeModel(**shape, rms_norm_eps=cfg.rms_norm_eps, rope_theta=cfg.rope_theta, rope_type=0, rope_factor=1.0, num_blocks=33, block_size=32, max_num_seqs=8,
                        max_model_len=32, weight_dtype=MI_W[wd], quant_type=MI_Q["per_channel_symmetric"], quantize_lm_head=1, tp_degree=1, tp_rank=0,
                        device_id=0, use_graphs=1, ctx_buckets=[32])
    model.load_state_dict(w)
    model.finalize()
    inputs = {rows: decode_inputs([i % vocab for i in range(rows)], [0] * rows, [[1 + i] for i in range(rows)], 32, 32) for rows in (5, 4, 1)}
    out = {rows: model.forward(**x).clone() for rows, x in inputs.items()}
    std = out[5].std().item()
    want = PagedDecoderOracle(cfg, w, 33, 32, compute="bf16", quant=_quant(wd)).forward(**inputs[4]).float()
    for rows in (4, 1):
        d = out[rows] - want[:rows]
        assert d.pow(2).mean().sqrt() < 0.02 * want.std() and d.abs().max() < 0.1 * want.std()
        assert torch.isfinite(out[rows]).all() and (out[rows] - out[5][:rows]).abs().max().item() < 0.05 * std
    model.close()


# the same sums at up to 4 rows: K of a narrow projection over several slices
@pytest.mark.parametrize("rows", [1, 4])
def test_sums_of_few_rows_left_to_the_next_norm(rows):
    for family in (_rapodra, _vimesun):
        test_sums_left_to_the_next_norm(family, rows)


def _rapodra():
    from tests import test_rapodra_gpu as T
    from tests.rapodra_cases import config, dense, latent
    cfg = config(256, 160, [latent(4, 32, 32, 64, 40, dense(6144)), latent(4, 32, 32, 64, 48, dense(6144), kv_from=0)], groups=2)
    return T, cfg


def _vimesun():
    from tests import test_vimesun_gpu as T
    from tests.vimesun_cases import att, config
    return T, config(256, 160, [att(4, 2, 32, 32, 40, 6144), att(4, 1, 32, 32, 48, 6144)])


# a feed-forward 24 times as deep as the row is wide: K goes over several slices, and the row norm behind it takes the sum over
@pytest.mark.parametrize("family", [_rapodra, _vimesun])
@pytest.mark.parametrize("rows", [5, 12, 32])
def test_sums_left_to_the_next_norm(family, rows):
    T, cfg = family()
    w = T.weights(cfg, 9)
    r = T.replay(cfg, w, "bfloat16", max_tokens=rows * 48, max_live=rows)
    toks = [T.tokens(cfg, w, n, 7000 + n) if family is _rapodra else T.tokens(cfg, n, 7000 + n) for n in (30, 31, 32)]
    refs = [T.reference(f"deep{i}", cfg, w, t, "bfloat16") for i, t in enumerate(toks)]
    ids = [T.uid() for _ in range(rows)]
    r.step([{"id": rid, "tokens": toks[i % 3][:20], "want": []} for i, rid in enumerate(ids)], [])
    worst = 0.0
    for p in range(20, 28):
        outs = r.step([{"id": rid, "tokens": [toks[i % 3][p]], "want": [0]} for i, rid in enumerate(ids)], ids if p == 27 else [])
        worst = max([worst] + [T.error(o, refs[i % 3][p:p + 1]) for i, o in enumerate(outs)])
    assert worst <= T.LIMIT["bfloat16"], worst
    r.engine.close()


@pytest.mark.parametrize("rows", [17, 32])
def test_fp8_activations_stay_with_prompts(rows):
    """A down projection deeper than eight slices of the registers (K > 32768) goes to the GEMM from 17 rows on: with bf16 activations there as well, whatever
    prompts have."""
    from oracle import DecoderConfig
    from oracle.synth import make_weights
    from tests.helpers import decode_inputs
    from vllm_neuron_amd._native import MI_Q, MI_W, NativeModel
    shape = dict(num_layers=1, hidden_size=128, num_heads=2, num_kv_heads=1, head_dim=64, intermediate_size=33792, vocab_size=256)
    w = make_weights(DecoderConfig(**shape), seed=4)
    out = []
    for a8 in (0, 1):
        model = NativeModel(**shape, rms_norm_eps=1e-5, rope_theta=1e4, rope_type=0, rope_factor=1.0, num_blocks=1 + rows, block_size=32, max_num_seqs=rows,
                            max_model_len=32, weight_dtype=MI_W["f8e4m3"], quant_type=MI_Q["per_channel_symmetric"], quantize_lm_head=1, tp_degree=1, tp_rank=0,
                            device_id=0, use_graphs=1, ctx_buckets=[32], prefill_fp8_activations=a8)
        model.load_state_dict(w)
        model.finalize()
        out.append(model.forward(**decode_inputs(range(rows), [0] * rows, [[1 + i] for i in range(rows)], 32, 32)).clone())
        model.close()
    assert torch.equal(*out)


def _logits_to_the_host(shape, wd, rows_of, max_rows=32):
    """Logits of the first step of a one-layer model, per number of rows, against the oracle at the bar of the other dispatch tests (a row-tile or a row in another place is off by the
    spread itself)."""
    from oracle import DecoderConfig, PagedDecoderOracle
    from oracle.synth import make_weights
    from tests.helpers import decode_inputs
    from vllm_neuron_amd._native import MI_Q, MI_W, NativeModel
    cfg, vocab = DecoderConfig(**shape), shape["vocab_size"]
    w = make_weights(cfg, seed=4)
    model = NativeModel(**shape, rms_norm_eps=cfg.rms_norm_eps, rope_theta=cfg.rope_theta, rope_type=0, rope_factor=1.0, num_blocks=33, block_size=32, max_num_seqs=max_rows,
                        max_model_len=32, weight_dtype=MI_W[wd], quant_type=MI_Q["per_channel_symmetric"], quantize_lm_head=1, tp_degree=1, tp_rank=0,
                        device_id=0, use_graphs=1, ctx_buckets=[32])
    model.load_state_dict(w)
    model.finalize()
    inputs = {rows: decode_inputs([i % vocab for i in range(rows)], [0] * rows, [[1 + i] for i in range(rows)], 32, 32) for rows in rows_of}
    want = PagedDecoderOracle(cfg, w, 33, 32, compute="bf16", quant=_quant(wd)).forward(**inputs[max(rows_of)]).float()
    out = {}
    for rows, x in inputs.items():
        for _ in range(2):         # eager pass, then the graph
            out[rows] = model.forward(**x).clone()
            d = out[rows] - want[:rows]
            assert torch.isfinite(d).all() and d.pow(2).mean().sqrt() < 0.02 * want.std() and d.abs().max() < 0.1 * want.std(), (wd, rows)
    model.close()
    return out


# logits of 16 and more rows to the host: single row-tiles, and from 8192 rows on (two of them a CU) four side by side: a last group of one, two, three and four, one and several a work-group
@pytest.mark.parametrize("vocab", [16, 80, 1024, 16448, 8176, 8192, 8208, 8224, 12272])
def test_logits_of_many_rows_to_the_host(vocab):
    shape = dict(num_layers=1, hidden_size=128, num_heads=2, num_kv_heads=1, head_dim=64, intermediate_size=256, vocab_size=vocab)
    for wd in ("bf16", "f8e4m3", "int8"):
        out = _logits_to_the_host(shape, wd, (16, 17, 32))
        # the same sums over K a row-tile, however many rows stand beside it; the projections in front differ in low bits between 16 and 17 rows, as between any two kernels
        assert torch.equal(out[17], out[32][:17]) and (out[16] - out[32][:16]).abs().max() < 0.05 * out[32].std()


# logits of up to 16 rows to the host: K so shallow that all go in groups of four row-tiles, and so deep that the line between those and single ones (rows * 540 >= bytes of a weight row) lies
# between 5 and 6 rows (bf16: 11 and 12); a last group of four, one, two and three, and below two row-tiles a CU
@pytest.mark.parametrize("vocab", [8176, 8192, 8208, 8224, 12272])
@pytest.mark.parametrize("hidden", [192, 3072])
def test_logits_of_few_rows_to_the_host(hidden, vocab):
    shape = dict(num_layers=1, hidden_size=hidden, num_heads=3, num_kv_heads=1, head_dim=64, intermediate_size=256, vocab_size=vocab)
    for wd in ("bf16", "f8e4m3", "int8"):
        out = _logits_to_the_host(shape, wd, (4, 5, 6, 11, 12, 16), 16)
        # single tiles and four have the same sums over K; the projections in front split theirs by the number of rows (bf16 3072 deep from 10 on)
        assert torch.equal(out[5], out[6][:5]) and torch.equal(out[11], out[12][:11])
        assert all((out[rows] - out[16][:rows]).abs().max() < 0.05 * out[16].std() for rows in out)


# ... and where they are sums of K slices
@pytest.mark.parametrize("wd", ["bf16", "f8e4m3", "int8"])
def test_logits_of_slices_to_the_host(wd):
    _logits_to_the_host(dict(num_layers=1, hidden_size=4224, num_heads=4, num_kv_heads=1, head_dim=64, intermediate_size=256, vocab_size=8208), wd, (4, 5, 16, 17, 32))


def _rapodra_of_many_words():
    from tests import test_rapodra_gpu as T
    from tests.rapodra_cases import config, dense, latent
    return T, config(256, 8208, [latent(4, 32, 32, 64, 40, dense(256))], groups=2)


# ... and bounded (bf16): groups of four with the last of one row-tile, against the oracle
@pytest.mark.parametrize("rows", [5, 16, 17])
def test_bounded_logits_to_the_host(rows):
    T, cfg = _rapodra_of_many_words()
    w = T.weights(cfg, 9)
    r = T.replay(cfg, w, "bfloat16", max_tokens=rows * 48, max_live=rows)
    toks = [T.tokens(cfg, w, n, 7000 + n) for n in (30, 31, 32)]
    refs = [T.reference(f"words{i}", cfg, w, t, "bfloat16") for i, t in enumerate(toks)]
    ids = [T.uid() for _ in range(rows)]
    r.step([{"id": rid, "tokens": toks[i % 3][:20], "want": []} for i, rid in enumerate(ids)], [])
    worst = 0.0
    for p in range(20, 24):
        outs = r.step([{"id": rid, "tokens": [toks[i % 3][p]], "want": [0]} for i, rid in enumerate(ids)], ids if p == 23 else [])
        worst = max([worst] + [T.error(o, refs[i % 3][p:p + 1]) for i, o in enumerate(outs)])
    assert worst <= T.LIMIT["bfloat16"], worst
    r.engine.close()


# Which of the two kernels takes 17 .. 32 rows of one-byte weights: the register kernel's sums over unsplit K are those of 16 rows bit for bit, the wide GEMM's are not.  Either side of the
# measured line by some us of 15 to 65 (profiles/few_rows_sweep.txt): shallow K stays, however full its tiles make the chip; deep and wide goes, unsplit and in slices; int8 later than fp8
@pytest.mark.parametrize("wd,N,K,rows,wide", [("f8e4m3", 49152, 6144, 17, True), ("int8", 49152, 6144, 32, True), ("f8e4m3", 10240, 8192, 20, True), ("int8", 20480, 5120, 32, False),
                                              ("f8e4m3", 28672, 3584, 17, False), ("f8e4m3", 16384, 3072, 32, False)])
def test_the_faster_kernel(lib, wd, N, K, rows, wide):
    g = torch.Generator().manual_seed(N + rows)
    w = torch.randn(N, K, generator=g) * 0.05
    x, bias = torch.randn(rows, K, generator=g).to(torch.bfloat16), torch.randn(N, generator=g) * 0.1
    tiled, scale = quantize_on_device(lib, w, wd, "per_channel_symmetric")
    xd, bd, out = dev(x), dev(bias), []
    for m in (16, rows):
        y = torch.full((m, N), float("nan"), dtype=torch.float32, device="cuda")
        lib.check(lib.load_library().mi_op_qlinear(xd.data_ptr(), m, tiled.data_ptr(), scale.data_ptr(), bd.data_ptr(), N, K, WD[wd], y.data_ptr(), 8, None))
        torch.cuda.synchronize()
        out.append(y.cpu())
    assert torch.isfinite(out[1]).all() and torch.equal(out[0], out[1][:16]) != wide
    assert (out[0] - out[1][:16]).abs().max().item() < 2e-5 * out[0].abs().max().item() + 1e-5 * (K ** 0.5)      # as above


# 17 .. 32 rows of one-byte weights leave the register kernel where deep K slices are summed by the next norm (2048 wide), where unsplit K fills the chip (fp8 gate | up
# of 24576 rows, from 25 rows on) and where it is deep besides (fp8 32768 x 5120, int8 32768 x 6144); not for sums of 256 wide
@pytest.mark.parametrize("wd,hidden,inter", [("f8e4m3", 256, 4096), ("f8e4m3", 3584, 12288), ("int8", 256, 16384), ("f8e4m3", 2048, 4096), ("int8", 2048, 17408), ("f8e4m3", 5120, 16384),
                                             ("int8", 6144, 16384)])
def test_rows_on_both_sides_of_the_wide_gemm(wd, hidden, inter):
    from oracle import DecoderConfig
    from oracle.synth import make_weights
    from tests.helpers import decode_inputs
    from vllm_neuron_amd._native import MI_Q, MI_W, NativeModel
    shape = dict(num_layers=2, hidden_size=hidden, num_heads=4, num_kv_heads=2, head_dim=64, intermediate_size=inter, vocab_size=512)
    model = NativeModel(**shape, rms_norm_eps=1e-5, rope_theta=1e4, rope_type=0, rope_factor=1.0, num_blocks=34, block_size=32, max_num_seqs=33,
                        max_model_len=32, weight_dtype=MI_W[wd], quant_type=MI_Q["per_channel_symmetric"], quantize_lm_head=1, tp_degree=1, tp_rank=0,
                        device_id=0, use_graphs=1, ctx_buckets=[32])
    model.load_state_dict(make_weights(DecoderConfig(**shape), seed=4))
    model.finalize()
    out = {}
    for rows in (16, 17, 31, 32, 33):
        for _ in range(2):             # eager pass, then the graph
            out[rows] = model.forward(**decode_inputs([7 * i % 512 for i in range(rows)], [0] * rows, [[1 + i] for i in range(rows)], 32, 32)).clone()
    std = out[16].std().item()
    for rows in (17, 31, 32, 33):      # sums in another order, roundings of bf16 activations behind them: as between any two kernels
        assert torch.isfinite(out[rows]).all() and (out[16] - out[rows][:16]).abs().max().item() < 0.05 * std and (out[33][:rows] - out[rows]).abs().max().item() < 0.05 * std
    model.close()


_OP = r"""
import sys, torch
sys.path.insert(0, %(root)r)
from vllm_neuron_amd import _native as lib
from tests.test_ops_gpu import WD, dev, quantize_on_device
lib.load_library()
for N, K in %(shapes)r:
    g = torch.Generator().manual_seed(N + K)
    tiled, scale = quantize_on_device(lib, torch.randn(N, K, generator=g) * 0.05, "f8e4m3", "per_channel_symmetric")
    x, y = dev(torch.randn(32, K, generator=g).to(torch.bfloat16)), {}
    for M in (16, 32):
        y[M] = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
        lib.check(lib.load_library().mi_op_qlinear(x.data_ptr(), M, tiled.data_ptr(), scale.data_ptr(), None, N, K, WD["f8e4m3"], y[M].data_ptr(), 8, None))
        torch.cuda.synchronize()
    assert torch.isfinite(y[32]).all() and (y[32][:16] - y[16]).abs().max() < 1e-4 * y[16].std()
    print("SAME" if torch.equal(y[32][:16], y[16]) else "OTHER", flush=True)
"""


def _kernels_of_32_rows(shapes, **env):
    """Per shape: whether 32 rows have the bits of 16, i.e. take the register kernel, whose sums do not depend on the rows beside them."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", _OP % {"root": root, "shapes": shapes}], env=dict(os.environ, **env), capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.stdout[-1500:], r.stderr[-1500:])
    return [x == "SAME" for x in r.stdout.split()[-len(shapes):]]


def test_switches_keep_32_rows_from_the_wide_gemm():
    """fp8, 192 tiles of 128 weight rows: the wide GEMM by size, the register kernel where that one is switched off or its token blocks are forced."""
    shape = [(24576, 3584)]
    assert _kernels_of_32_rows(shape) == [False]
    assert _kernels_of_32_rows(shape, MI355X_GEMM_WIDE="0") == [True] and _kernels_of_32_rows(shape, MI355X_GEMM_WIDE_BM="128") == [True]


def test_a_tile_more_than_the_chip_stays_in_registers():
    """fp8, tiles of 128 weight rows, one work-group a CU: 257 of them on 256 CUs are a second round for one (a last tile of 16 rows counts)."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert _kernels_of_32_rows([(128 * cus + 16, 3584), (128 * cus, 3584)]) == [True, False]


_ROUTES = r"""
import sys, torch
sys.path.insert(0, %(root)r)
from vllm_neuron_amd._native import MI_Q, MI_W, NativeModel
from tests.helpers import decode_inputs
res = {}
for wd, hidden, inter, heads, kv in %(shapes)r:
    m = NativeModel(num_layers=1, hidden_size=hidden, num_heads=heads, num_kv_heads=kv, head_dim=128, intermediate_size=inter, vocab_size=512, rms_norm_eps=1e-5,
                    rope_theta=1e4, rope_type=0, rope_factor=1.0, num_blocks=33, block_size=32, max_num_seqs=32, max_model_len=32, weight_dtype=MI_W[wd],
                    quant_type=MI_Q["per_channel_symmetric"], quantize_lm_head=1, tp_degree=1, tp_rank=0, device_id=0, use_graphs=1, ctx_buckets=[32])
    m.init_synthetic_weights(1, 0.02)
    m.finalize()
    for rows in (17, 28):
        res[wd, hidden, inter, heads, kv, rows] = m.forward(**decode_inputs([7 * i %% 512 for i in range(rows)], [0] * rows, [[1 + i] for i in range(rows)], 32, 32)).clone()
    m.close()
torch.save(res, sys.argv[1])
"""

# (weights, hidden, feed-forward, heads, kv heads) -> whether 17 and 28 rows go through the register kernel alone
_REGS_ALONE = {
    ("int8", 2048, 16384, 16, 4): (True, True),             # sums of int8 stay, up to K of 16384
    ("int8", 2048, 17408, 16, 4): (False, False),           # a little beyond
    ("int8", 1536, 17408, 12, 2): (True, True),             # narrow
    ("f8e4m3", 2048, 4096, 16, 4): (False, False),          # a sum of 4096 deep
    ("f8e4m3", 1024, 4096, 8, 2): (True, True),             # narrow
    ("f8e4m3", 2048, 14336, 16, 4): (True, True),           # deep and narrow: ten slices of K are 160 work-groups of the wide GEMM
    ("f8e4m3", 3584, 3584, 28, 14): (True, True),           # K of 3584; queries, keys and values are twice the width
    ("f8e4m3", 3584, 3584, 28, 28): (True, False)}          # three times: the wide GEMM from 25 rows on


def test_which_calls_of_17_to_32_rows_leave_the_register_kernel(tmp_path):
    root, got = os.path.dirname(os.path.dirname(os.path.abspath(__file__))), []
    for i, env in enumerate(({}, dict(MI355X_GEMM_WIDE="0"))):
        out = str(tmp_path / f"{i}.pt")
        r = subprocess.run([sys.executable, "-c", _ROUTES % {"root": root, "shapes": list(_REGS_ALONE)}, out], env=dict(os.environ, **env), capture_output=True, text=True,
                           timeout=300)
        assert r.returncode == 0, (r.stdout[-1500:], r.stderr[-1500:])
        got.append(torch.load(out, weights_only=True))
    for k, want in _REGS_ALONE.items():
        assert tuple(torch.equal(got[0][(*k, rows)], got[1][(*k, rows)]) for rows in (17, 28)) == want, k


# queries, keys and values by the wide GEMM from 25 rows on and earlier (their slices' sum rotates them and writes them to the pool, which the second step reads), the down
# projection by it from 17 rows on, logits to the host in groups of four row-tiles of which the last has one: against the oracle, at the bar of the other dispatch tests
@pytest.mark.parametrize("rows", [16, 17, 25, 32])
def test_two_steps_of_many_rows_against_the_oracle(rows):
    from oracle import DecoderConfig, PagedDecoderOracle
    from oracle.synth import make_weights
    from tests.helpers import decode_inputs
    from vllm_neuron_amd._native import MI_Q, MI_W, NativeModel
    shape = dict(num_layers=1, hidden_size=3584, num_heads=28, num_kv_heads=4, head_dim=128, intermediate_size=4096, vocab_size=8208)
    if not _oracle:
        cfg = DecoderConfig(**shape)
        _oracle.append((cfg, make_weights(cfg, seed=4)))
    cfg, w = _oracle[0]
    oracle = PagedDecoderOracle(cfg, w, 34, 32, compute="bf16", quant=dict(quantized=True, quantization_dtype="f8e4m3", quantization_type="per_channel_symmetric"))
    model = NativeModel(**shape, rms_norm_eps=cfg.rms_norm_eps, rope_theta=cfg.rope_theta, rope_type=0, rope_factor=1.0, num_blocks=34, block_size=32, max_num_seqs=32,
                        max_model_len=32, weight_dtype=MI_W["f8e4m3"], quant_type=MI_Q["per_channel_symmetric"], quantize_lm_head=1, tp_degree=1, tp_rank=0, device_id=0,
                        use_graphs=1, ctx_buckets=[32])
    model.load_state_dict(w)
    model.finalize()
    for at in range(2):
        inputs = decode_inputs([(31 * i + 7 * at) % 8208 for i in range(rows)], [at] * rows, [[1 + i] for i in range(rows)], 32, 32)
        want = oracle.forward(**inputs).float()
        for _ in range(2):             # eager pass, then the graph
            d = model.forward(**inputs).float() - want
            assert torch.isfinite(d).all() and d.pow(2).mean().sqrt() < 0.02 * want.std() and d.abs().max() < 0.1 * want.std()
    model.close()



# two row-tiles a work-group and more, of which the first has its epilogue's operands asked for ahead and the others do not: rotated queries and keys (384 row-tiles of 512), residual sums
# unsplit (272 of 256); one and two column groups, the last one with a single row
@pytest.mark.parametrize("wd", ["bf16", "f8e4m3", "int8"])
@pytest.mark.parametrize("rows", [5, 16, 17, 32])
@pytest.mark.parametrize("hidden,heads,kv,dim,inter", [(512, 32, 8, 128, 256), (4352, 4, 2, 64, 256)])
def test_epilogues_of_several_row_tiles(wd, rows, hidden, heads, kv, dim, inter):
    from oracle import DecoderConfig, PagedDecoderOracle
    from oracle.synth import make_weights
    from tests.helpers import decode_inputs
    from vllm_neuron_amd._native import MI_Q, MI_W, NativeModel
    shape = dict(num_layers=1, hidden_size=hidden, num_heads=heads, num_kv_heads=kv, head_dim=dim, intermediate_size=inter, vocab_size=512)
    cfg = DecoderConfig(**shape)
    w = make_weights(cfg, seed=4)
    oracle = PagedDecoderOracle(cfg, w, 34, 32, compute="bf16", quant=_quant(wd))
    model = NativeModel(**shape, rms_norm_eps=cfg.rms_norm_eps, rope_theta=cfg.rope_theta, rope_type=0, rope_factor=1.0, num_blocks=34, block_size=32, max_num_seqs=32,
                        max_model_len=32, weight_dtype=MI_W[wd], quant_type=MI_Q["per_channel_symmetric"], quantize_lm_head=1, tp_degree=1, tp_rank=0, device_id=0,
                        use_graphs=1, ctx_buckets=[32])
    model.load_state_dict(w)
    model.finalize()
    for at in range(3):                # (positions that turn)
        inputs = decode_inputs([(31 * i + 7 * at) % 512 for i in range(rows)], [at] * rows, [[1 + i] for i in range(rows)], 32, 32)
        want = oracle.forward(**inputs).float()
        d = model.forward(**inputs).float() - want
        assert torch.isfinite(d).all() and d.pow(2).mean().sqrt() < 0.02 * want.std() and d.abs().max() < 0.1 * want.std()
    model.close()


_oracle = []


# norms that a residual projection hands on to the next one: 3, 32, 33 and 64 requests of 4 parts for a row (the second 32 are a thread's second request), down projections that
# keep K in one piece (their norm is handed on too, the last one's to the head) and some that do not (up to 4 rows every kernel hands it on), a width whose next projection splits K; the rows on
# both sides of each kernel
@pytest.mark.parametrize("wd", ["bf16", "f8e4m3", "int8"])
@pytest.mark.parametrize("hidden,inter", [(192, 320), (2048, 4096), (2112, 4160), (4096, 1024), (4160, 512), (1024, 19008)])
def test_norms_handed_on(wd, hidden, inter):
    from oracle import DecoderConfig, PagedDecoderOracle
    from oracle.synth import make_weights
    from tests.helpers import decode_inputs
    from vllm_neuron_amd._native import MI_Q, MI_W, NativeModel
    shape = dict(num_layers=2, hidden_size=hidden, num_heads=4, num_kv_heads=2, head_dim=64, intermediate_size=inter, vocab_size=528)
    cfg = DecoderConfig(**shape)
    w = make_weights(cfg, seed=5)
    model = NativeModel(**shape, rms_norm_eps=cfg.rms_norm_eps, rope_theta=cfg.rope_theta, rope_type=0, rope_factor=1.0, num_blocks=34, block_size=32, max_num_seqs=32,
                        max_model_len=32, weight_dtype=MI_W[wd], quant_type=MI_Q["per_channel_symmetric"], quantize_lm_head=1, tp_degree=1, tp_rank=0, device_id=0,
                        use_graphs=1, ctx_buckets=[32])
    model.load_state_dict(w)
    model.finalize()
    for rows in (1, 2, 4, 5, 16, 17):
        oracle = PagedDecoderOracle(cfg, w, 34, 32, compute="bf16", quant=_quant(wd))
        for at in range(3):                # the call that is captured, and two replays
            inputs = decode_inputs([(31 * i + 7 * at) % 528 for i in range(rows)], [at] * rows, [[1 + i] for i in range(rows)], 32, 32)
            want = oracle.forward(**inputs).float()
            d = model.forward(**inputs).float() - want
            assert torch.isfinite(d).all() and d.pow(2).mean().sqrt() < 0.02 * want.std() and d.abs().max() < 0.1 * want.std()       # as above
    model.close()

"""The wide context-encoding GEMM (gemm_wide_kernel, gemm_wide16_kernel) at the edges of its tiles, K-steps and K-slices, for every weight type;
and, with the epilogues of the layer stacks, against the 128 x 128 kernel.  Products of bf16 activations with bf16, e4m3 or int8 weights are
exact in fp32, so two runs differ by their summation order alone."""
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


# one, two and three K-steps (fewer than the ring has stages); a ring's length and one more; slices of uneven length (5 and 11 K-steps over 2 .. 10
# slices); rows and columns one tile more than a block, one row short of it, a single 16-row tile behind the last block
@pytest.mark.parametrize("wd", ["bf16", "f8e4m3", "int8"])
@pytest.mark.parametrize("M,N,K", [(129, 32, 64), (255, 272, 128), (257, 528, 192), (300, 272, 320), (385, 256, 704), (130, 8208, 2112),
                                   (33, 4112, 4224), (100, 2064, 8640), (513, 1040, 1088), (1100, 6160, 576), (2031, 1296, 1984)])
def test_edges_of_the_wide_gemm(lib, wd, M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    w = torch.randn(N, K, generator=g) * 0.05
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    bias = torch.randn(N, generator=g) * 0.1
    tiled, scale = quantize_on_device(lib, w, wd, "per_channel_symmetric")
    wq = w.to(torch.bfloat16).float() if wd == "bf16" else dequantize_weight(*quantize_weight(w, wd, "per_channel_symmetric"))
    ref = (x.float() @ wq.t()).double() if M * N * K > 1 << 31 else x.double() @ wq.double().t()
    ref += bias.double()
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    xd, bd = dev(x), dev(bias)
    lib.check(lib.load_library().mi_op_qlinear(xd.data_ptr(), M, tiled.data_ptr(), scale.data_ptr(), bd.data_ptr(), N, K, WD[wd], y.data_ptr(), 8, None))
    torch.cuda.synchronize()
    err = (y.cpu().double() - ref).abs().max().item()
    tol = 2e-5 * ref.abs().max().item() + 1e-5 * (K ** 0.5)     # as the other linear tests: fp32 sums in another order
    assert err < tol, (err, tol)


# every tile, at shapes that leave none of its edges whole: a token and a 16-row weight tile past a block, K-steps fewer, as many and more than its stages,
# three uneven slices
@pytest.mark.parametrize("wd", ["bf16", "f8e4m3", "int8"])
@pytest.mark.parametrize("bm", [64, 128, 192, 256])
@pytest.mark.parametrize("ntw", [2, 3, 4])
def test_every_tile_of_the_wide_gemm(lib, wd, bm, ntw):
    check_tile(lib, wd, bm, ntw, ((bm + 1, 64 * ntw + 16, 64, 1), (bm - 1, 80, 320, 1), (2 * bm, 128 * ntw, 704, 1), (33, 8 * 64 * ntw + 32, 576, 1),
                                  (bm + 17, 64 * ntw + 16, 704, 3)))


def check_tile(lib, wd, bm, ntw, shapes):
    for M, N, K, ks in shapes:
        g = torch.Generator().manual_seed(M + N + K)
        w = torch.randn(N, K, generator=g) * 0.05
        x = torch.randn(M, K, generator=g).to(torch.bfloat16)
        bias = torch.randn(N, generator=g) * 0.1
        tiled, scale = quantize_on_device(lib, w, wd, "per_channel_symmetric")
        wq = w.to(torch.bfloat16).float() if wd == "bf16" else dequantize_weight(*quantize_weight(w, wd, "per_channel_symmetric"))
        ref = x.double() @ wq.double().t() + bias.double()
        y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
        xd, bd = dev(x), dev(bias)
        lib.check(lib.load_library().mi_op_qlinear(xd.data_ptr(), M, tiled.data_ptr(), scale.data_ptr(), bd.data_ptr(), N, K, WD[wd], y.data_ptr(),
                                                   100 * bm + 10 * ntw + ks, None))
        torch.cuda.synchronize()
        err = (y.cpu().double() - ref).abs().max().item()
        tol = 2e-5 * ref.abs().max().item() + 1e-5 * (K ** 0.5)
        assert err < tol, (M, N, K, ks, err, tol)


# blocks of 32, 96 and 160 tokens, whose activation pieces the two wave groups do not share evenly (32: the second has none)
@pytest.mark.parametrize("wd", ["bf16", "f8e4m3", "int8"])
@pytest.mark.parametrize("bm", [32, 96, 160])
@pytest.mark.parametrize("ntw", [2, 3, 4])
def test_tiles_of_uneven_pieces(lib, wd, bm, ntw):
    test_every_tile_of_the_wide_gemm(lib, wd, bm, ntw)


# 128-deep K-steps (weights of a byte, tiles that fit the LDS three times by them, K a multiple of 128): one, two and three of them, as many as the ring of
# three to six stages has, fewer and more; three uneven slices (4, 4 and 3 steps); four slices of 64-deep steps (3, 3, 3 and 1), whose last would be empty by
# 128-deep ones; rows that fill a token block but for one, and the least of the calls that take blocks of 32
@pytest.mark.parametrize("wd", ["f8e4m3", "int8"])
@pytest.mark.parametrize("bm,ntw", [(32, 2), (32, 3), (32, 4), (64, 2), (64, 3), (64, 4), (96, 2), (96, 3), (128, 2)])
def test_tiles_by_128_deep_steps(lib, wd, bm, ntw):
    rows = (17, 31, 32) if bm == 32 else (bm - 1, bm, bm + 17)
    steps = [(rows[i % 3], 64 * ntw * (1 + i % 2) + 16, 128 * n, 1) for i, n in enumerate((1, 2, 3, 4, 5, 6, 7, 8, 11))]
    check_tile(lib, wd, bm, ntw, steps + [(m, 64 * ntw + 16, 1408, 3) for m in rows] + [(rows[0], 64 * ntw + 16, 640, 4), (rows[1], 208, 256, 2)])


# bf16 tiles by 32-deep K-steps: one pair of them, as many pairs as the ring of activations has, fewer and more; slices of two and of uneven length
@pytest.mark.parametrize("bm,ntw", [(192, 4), (256, 3), (256, 4)])
@pytest.mark.parametrize("M,N,K,ks", [(1, 16, 64, 1), (193, 208, 128, 1), (257, 272, 192, 1), (191, 400, 256, 1), (640, 560, 1088, 1), (300, 272, 128, 2), (255, 784, 704, 3)])
def test_tiles_by_32_deep_steps(lib, bm, ntw, M, N, K, ks):
    g = torch.Generator().manual_seed(M + N + K)
    w = (torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16)
    x, bias = torch.randn(M, K, generator=g).to(torch.bfloat16), torch.randn(N, generator=g) * 0.1
    tiled, scale = quantize_on_device(lib, w.float(), "bf16", "per_channel_symmetric")
    ref = x.double() @ w.double().t() + bias.double()
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    xd, bd = dev(x), dev(bias)
    lib.check(lib.load_library().mi_op_qlinear(xd.data_ptr(), M, tiled.data_ptr(), scale.data_ptr(), bd.data_ptr(), N, K, WD["bf16"], y.data_ptr(),
                                               100 * bm + 10 * ntw + ks, None))
    torch.cuda.synchronize()
    err = (y.cpu().double() - ref).abs().max().item()
    assert err < 2e-5 * ref.abs().max().item() + 1e-5 * (K ** 0.5), err      # as above


_CHILD = r"""
import sys, torch
sys.path.insert(0, %(root)r)
from vllm_neuron_amd._native import NativeModel
from vllm_neuron_amd.models import config_from_dict, fill_sizes
from tests.helpers import prefill_inputs
out = sys.argv[1]
dense = {"kind": "dense", "ff": 1200}
att = {"heads": 8, "kv_heads": 2, "dim": 64, "vdim": 64, "mask": {"size": 256}, "scale": 0.125}
common = {"width": 500, "vocab": 1010, "norm": {"eps": 1e-5}}
designs = {
    "vimesun": {"architecture": "Vimesun", **common, "layers": [{"type": "attention", "mixer": att, "mlp": dense}] * 2, "residual_mult": 0.5,
                "max_positions": 1024},
    "rapodra": {"architecture": "Rapodra", **common, "norm": {"eps": 1e-5, "groups": 4}, "canon": {"taps": 4}, "logit_softcap": 30.0, "layers": [
        {"type": "latent_attention", "mixer": {"heads": 4, "dim": 64, "vdim": 64, "kv_rank": 192, "mask": {"size": 256}, "scale": 0.125},
         "mlp": dict(dense, limit=7.0)}] * 2},
    "nusovik": {"architecture": "Nusovik", **common, "embedding": {"scale": 1.0}, "logit_scale": 1.0, "layers": [{"type": "parallel", "mixer": {
        "left": dict(att, bias_max=128), "right": {"heads": 8, "vdim": 64, "state": 64, "groups": 1, "norm_groups": 1, "conv": 4},
        "left_scale": 1.0, "right_scale": 1.0}, "mlp": dense}] * 2},
}
g, res = torch.Generator().manual_seed(5), {}
for name, config in designs.items():
    c = config_from_dict(config)
    fill_sizes(c, lambda n: (32, 500))
    m = NativeModel(stack=dict(c.stack, compute_dtype=1), num_blocks=65, block_size=16, max_num_seqs=4, max_model_len=1024, device_id=0,
                    use_graphs=1, ctx_buckets=[1024])
    m.init_synthetic_weights(1, 0.05)
    m.finalize()
    for n in (40, 150, 300, 777):
        prompt = torch.randint(0, 1010, (n,), generator=g).tolist()
        inp = prefill_inputs(prompt, list(range(1, 2 + n // 16)), 16, 1024)
        res[name + str(n)] = m.forward(**inp).float().clone()
        print(name, n, flush=True)
    m.close()
torch.save(res, out)
print("CHILD_OK", flush=True)
"""


def test_stack_epilogues_agree_with_the_128x128_kernel(tmp_path):
    """Squared relu, clipped gate, soft cap, keys and values by head; widths that are no multiple of a tile.  The switch is read once per process."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    got = {}
    for wide in ("0", "1"):
        out = str(tmp_path / f"logits_{wide}.pt")
        r = subprocess.run([sys.executable, "-c", _CHILD % {"root": root}, out], env=dict(os.environ, MI355X_GEMM_WIDE=wide), capture_output=True,
                           text=True, timeout=300)
        assert r.returncode == 0 and "CHILD_OK" in r.stdout, (r.stdout[-1500:], r.stderr[-1500:])
        got[wide] = torch.load(out, weights_only=True)
    for k, want in got["0"].items():
        d = got["1"][k] - want
        assert torch.isfinite(d).all() and d.pow(2).mean().sqrt() < 0.02 * want.std(), k    # the bar of the other dispatch test


_LLAMAS = r"""
import sys, torch
sys.path.insert(0, %(root)r)
from vllm_neuron_amd._native import NativeModel, MI_W, MI_Q
from tests.helpers import prefill_inputs
out, hd, heads, kv, wd = sys.argv[1], *map(int, sys.argv[2:5]), sys.argv[5]
m = NativeModel(num_layers=2, hidden_size=320, num_heads=heads, num_kv_heads=kv, head_dim=hd, intermediate_size=448, vocab_size=1008, rms_norm_eps=1e-5,
                rope_theta=1e4, rope_type=0, qkv_bias=int(wd == "int8"), tie_word_embeddings=0, num_blocks=65, block_size=16, max_num_seqs=4,
                max_model_len=1024, weight_dtype=MI_W[wd], quant_type=MI_Q["per_channel_symmetric"], quantize_lm_head=0, tp_degree=1, tp_rank=0, device_id=0,
                use_graphs=1, prefill_fp8_activations=0)
m.init_synthetic_weights(1, 0.05)
m.finalize()
g, res = torch.Generator().manual_seed(5), {}
for n, cached in ((33, 0), (150, 0), (257, 0), (300, 112), (777, 0)):
    prompt = torch.randint(0, 1000, (n,), generator=g).tolist()
    blocks = list(range(1, 2 + n // 16))
    if cached:
        m.forward(**prefill_inputs(prompt[:cached], blocks, 16, 1024))
    res[n] = m.forward(**prefill_inputs(prompt, blocks, 16, 1024, cached)).float().cpu().clone()
    print(n, flush=True)
m.close()
torch.save(res, out)
print("CHILD_OK", flush=True)
"""


# a wave's tiles that hold q and k, k and v; one and three heads a kv head; every row block with a remainder; planned tiles, and 128 and 256 tokens x 256 rows
@pytest.mark.parametrize("hd,heads,kv,wd", [(64, 6, 2, "bf16"), (128, 1, 1, "int8"), (64, 3, 1, "f8e4m3")])
def test_llama_epilogues_agree_with_the_128x128_kernel(tmp_path, hd, heads, kv, wd):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    got = []
    for i, env in enumerate((dict(MI355X_GEMM_WIDE="0"), dict(MI355X_GEMM_WIDE="1"), dict(MI355X_GEMM_WIDE="1", MI355X_GEMM_WIDE_BM="128"),
                             dict(MI355X_GEMM_WIDE="1", MI355X_GEMM_WIDE_BM="256"))):
        out = str(tmp_path / f"{i}.pt")
        r = subprocess.run([sys.executable, "-c", _LLAMAS % {"root": root}, out, str(hd), str(heads), str(kv), wd], env=dict(os.environ, **env),
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0 and "CHILD_OK" in r.stdout, (r.stdout[-1500:], r.stderr[-1500:])
        got.append(torch.load(out, weights_only=True))
    for n, want in got[0].items():
        for other in got[1:]:
            d = other[n] - want
            assert torch.isfinite(d).all() and d.pow(2).mean().sqrt() < 0.02 * want.std(), n    # the bar of the other dispatch test


# Small whole numbers: the slices' sum is exact in fp32 in any order, so scale and bias are all that rounds, and the launch that adds slices makes one fused multiply-add of them.
# (Two roundings, half a unit each of numbers twice the result's size, would be off by more than half a unit of the result in a part of the rows.)
@pytest.mark.parametrize("M,N,K,ks", [(33, 272, 704, 3), (100, 1040, 1984, 8), (188, 528, 320, 2)])
def test_sums_of_slices_round_once(lib, M, N, K, ks):
    g = torch.Generator().manual_seed(M + N + K)
    q = torch.randint(-20, 21, (N, K), generator=g).float()
    q[:, 0] = 127                                                     # int8 codes are these numbers
    x = torch.randint(-3, 4, (M, K), generator=g).to(torch.bfloat16)
    bias = torch.randn(N, generator=g) * 20
    tiled, scale = quantize_on_device(lib, q * (0.3 + torch.rand(N, 1, generator=g)) / 127, "int8", "per_channel_symmetric")
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    xd, bd = dev(x), dev(bias)
    lib.check(lib.load_library().mi_op_qlinear(xd.data_ptr(), M, tiled.data_ptr(), scale.data_ptr(), bd.data_ptr(), N, K, WD["int8"], y.data_ptr(), 6420 + ks, None))
    torch.cuda.synchronize()
    ref = (x.double() @ q.double().t()) * scale.cpu().double() + bias.double()      # 48 bits and a sum: 64-bit rounding is 2^-29 of a unit here
    unit = 2.0 ** (torch.frexp(ref.abs())[1].double() - 24)
    assert ((y.cpu().double() - ref).abs() <= 0.50001 * unit).all()


# slabs of 24 MiB (written through) and one row more than that, in two and three slices; twice as much; whole token blocks and a short last one.  Weights of four times the slabs (through) and 64 of K more,
# in bf16 and in a byte
@pytest.mark.parametrize("wd", ["bf16", "f8e4m3", "int8"])
@pytest.mark.parametrize("M,N,K,bm,ntw,ks", [(1024, 2048, 192, 128, 2, 3), (1025, 2048, 192, 128, 3, 3), (1024, 3072, 128, 256, 4, 2), (1025, 3072, 128, 192, 4, 2), (2048, 2064, 192, 256, 4, 3),
                                             (32, 528, 512, 64, 2, 2), (32, 528, 576, 64, 3, 2), (32, 528, 1024, 64, 4, 2), (32, 528, 1088, 96, 2, 2), (48, 272, 1152, 64, 2, 3), (48, 272, 1216, 64, 2, 3),
                                             (48, 272, 2304, 64, 3, 3), (48, 272, 2368, 64, 3, 3)])
def test_slabs_left_in_l2_and_written_through(lib, wd, M, N, K, bm, ntw, ks):
    check_tile(lib, wd, bm, ntw, ((M, N, K, ks),))

"""Token generation over contexts of more 32-token tiles a wave than one look at the block table holds (32): the last of a look, the first of the next, a third look."""
import pytest
import torch

from oracle.nusovik import bucket
from tests.helpers import pool_to_native
from tests.test_ops_gpu import _make_pool, dev, lib, ref_attention  # noqa: F401  (lib: the fixture)
from tests.test_vimesun_gpu import spec_of

pytestmark = pytest.mark.gpu


def _tables(ctx, bs, MB, pad):
    g = torch.Generator().manual_seed(7)
    need = [-(-n // bs) for n in ctx]
    perm = (torch.randperm(sum(need), generator=g) + 1).int()
    bt = torch.full((len(ctx), MB), pad, dtype=torch.int32)
    for b, n in enumerate(need):
        bt[b, :n], perm = perm[:n], perm[n:]
    return bt, 1 + sum(need)


# 32 sequences of 8 kv heads: eight waves of one work-group take a sequence, 256 tokens to each of their tiles
@pytest.mark.parametrize("bs", [16, 48])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("tiles", [29, 30, 31, 32, 33, 63])
def test_long_contexts(lib, hd, bs, tiles):  # noqa: F811
    _long_contexts(lib, hd, bs, tiles, 32)


# 16 sequences: two slices of four waves to each, 256 tokens to each of a wave's tiles again, and a launch that puts the slices together
@pytest.mark.parametrize("hd,bs", [(64, 48), (128, 16)])
@pytest.mark.parametrize("tiles", [30, 31, 32, 33, 63])
def test_long_contexts_in_slices(lib, hd, bs, tiles):  # noqa: F811
    _long_contexts(lib, hd, bs, tiles, 16)


def _long_contexts(lib, hd, bs, tiles, rows):  # noqa: F811
    ctx = [3 + i for i in range(rows)]
    ctx[5], ctx[-2] = 256 * tiles + 1, 256 * tiles - 20
    MB = -(-max(ctx) // bs) + 3
    bt, nb = _tables(ctx, bs, MB, -1)                      # pad -1: must never be read
    k, v = _make_pool(nb, bs, 8, hd, 4)
    q = torch.randn(rows, 16, hd, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16)
    out = torch.empty(rows, 16 * hd, dtype=torch.bfloat16, device="cuda")
    L = lib.load_library()
    scratch = torch.empty(L.mi_op_attn_scratch_bytes(rows, 16, hd), dtype=torch.uint8, device="cuda")
    d = [dev(t) for t in (q, pool_to_native(k, v, nb, bs), bt, torch.tensor(ctx, dtype=torch.int32))]
    lib.check(L.mi_op_paged_attn_decode(d[0].data_ptr(), d[1].data_ptr(), nb, bs, d[2].data_ptr(), MB, d[3].data_ptr(), rows, 16, 8, hd, out.data_ptr(),
                                        scratch.data_ptr(), None))
    torch.cuda.synchronize()
    kk, vv = k.float().reshape(nb, bs, 8, hd), v.float().reshape(nb, bs, 8, hd)
    for b in (0, 5, rows - 2, rows - 1):
        idx = torch.arange(ctx[b])
        blk = bt[b, idx // bs].long()
        ref = ref_attention(q[b:b + 1].float(), kk[blk, idx % bs], vv[blk, idx % bs], torch.tensor([ctx[b] - 1]))
        assert (out[b].cpu().float() - ref[0]).abs().max().item() < 0.02, (b, ctx[b])      # bf16 output rounding of O(1) values


# the windowed kernel's, a launch a sequence here: 16 slices of four waves to each of 8 kv heads, one tile a wave to four; a window that starts inside a tile
@pytest.mark.parametrize("d,bs", [(64, 32), (100, 16)])
@pytest.mark.parametrize("tiles,window", [(30, 0), (31, 0), (32, 0), (33, 4000), (63, 0)])
def test_long_windows(lib, d, bs, tiles, window):  # noqa: F811
    ctx = [3 + i for i in range(32)]
    ctx[5], ctx[30] = 128 * tiles + 1, 128 * tiles - 20
    _long_windows(lib, 16, 8, d, bs, ctx, window, tiles, (0, 5, 30, 31))


# ... and with 130 kv heads, where the four waves of one work-group take a whole context, 128 tokens to each of their tiles: more of them than a look holds
@pytest.mark.parametrize("d,bs", [(32, 32), (20, 16)])
@pytest.mark.parametrize("tiles,window", [(30, 0), (31, 0), (32, 0), (33, 4000), (63, 0)])
def test_long_windows_of_one_work_group(lib, d, bs, tiles, window):  # noqa: F811
    _long_windows(lib, 130, 130, d, bs, [128 * tiles + 1, 128 * tiles - 20, 7], window, tiles, (0, 1, 2))


def _long_windows(lib, H, G, d, bs, ctx, window, seed, checked):  # noqa: F811
    dp, B = -(-d // 16) * 16, len(ctx)
    MB = -(-max(ctx) // bs) + 1
    bt, nb = _tables(ctx, bs, MB, 0)
    g = torch.Generator().manual_seed(seed)
    k, v = (torch.zeros(nb, G, bs, dp, dtype=torch.bfloat16) for _ in range(2))
    k[..., :d], v[..., :d] = torch.randn(nb, G, bs, d, generator=g), torch.randn(nb, G, bs, d, generator=g)
    q = torch.zeros(B, H, dp, dtype=torch.bfloat16)
    q[..., :d] = torch.randn(B, H, d, generator=g)
    ldo = (H * d + 63) // 64 * 64
    out = torch.zeros(B, ldo, dtype=torch.bfloat16, device="cuda")
    pos = torch.tensor([n - 1 for n in ctx], dtype=torch.int32)
    x = [dev(t) for t in (torch.zeros(H), q, k, v, bt, pos, pos + 1)]
    segs = torch.tensor([(i, 1, n - 1, i) for i, n in enumerate(ctx)], dtype=torch.int32).contiguous()
    spec = spec_of(lib, H, G, d, d, window, d ** -0.5, bias=0, sink=0, unit=0)
    lib.check(lib.load_library().mi_op_window_attn(spec, x[0].data_ptr(), x[1].data_ptr(), x[2].data_ptr(), x[3].data_ptr(), bs, x[4].data_ptr(), MB, x[5].data_ptr(),
                                                   x[6].data_ptr(), segs.data_ptr(), B, B, max(ctx), out.data_ptr(), ldo, 0, 0, None))
    torch.cuda.synchronize()
    for b in checked:
        idx = torch.arange(max(0, ctx[b] - window) if window else 0, ctx[b])
        blk = bt[b, idx // bs].long()
        K, W = (t[blk, :, idx % bs, :d].double() for t in (k, v))
        s = torch.einsum("hd,nhd->hn", q[b, :, :d].double(), K.repeat_interleave(H // G, 1)) * d ** -0.5
        ref = torch.einsum("hn,nhd->hd", torch.softmax(s, -1), W.repeat_interleave(H // G, 1)).flatten()
        assert (out[b, :H * d].cpu().double() - ref).abs().max().item() < 0.02, (b, ctx[b])      # as above


# chunked attention with its distance table and sinks, so many kv heads that one work-group's four waves take a whole context (128 tokens to each of their tiles): no tile, one, two and three for a wave, the last of a look, the first of the next, a third look
@pytest.mark.parametrize("n", [1, 33, 128, 129, 257, 300, 400, 128 * 31 + 5, 128 * 32, 128 * 32 + 1, 128 * 33, 128 * 63 + 20])
def test_tables_and_tiles(lib, n):  # noqa: F811
    H, G, d, bs, mult = 130, 130, 32, 32, 0.7
    MB = -(-n // bs) + 1
    bt, nb = _tables([n], bs, MB, 0)
    g = torch.Generator().manual_seed(n)
    k, v = (torch.randn(nb, G, bs, d, generator=g).to(torch.bfloat16) for _ in range(2))
    k[0], v[0] = 50., 50.                                  # (nobody's block)
    q = torch.randn(1, H, d, generator=g).to(torch.bfloat16)
    rel, sink, gate = torch.randn(16, H, generator=g) * 2, torch.randn(H, generator=g) + 1, torch.randn(1, H, generator=g)
    out = torch.zeros(1, H * d, dtype=torch.bfloat16, device="cuda")
    spec = lib.layer_spec(dict(num_heads=H, num_kv_heads=G, qk_dim=d, v_dim=d, chunk=8200, scale=0.1, rel_rows=16, rel_far=200, softmax_sink=2))
    pos = torch.tensor([n - 1], dtype=torch.int32)
    x = [dev(t) for t in (sink, rel, gate, q, k, v, bt, pos, pos + 1)]
    segs = torch.tensor([(0, 1, n - 1, 0)], dtype=torch.int32).contiguous()
    lib.check(lib.load_library().mi_op_chunk_attn(spec, x[0].data_ptr(), x[1].data_ptr(), x[2].data_ptr(), H, mult, x[3].data_ptr(), x[4].data_ptr(), x[5].data_ptr(), bs,
                                                  x[6].data_ptr(), MB, x[7].data_ptr(), x[8].data_ptr(), segs.data_ptr(), 1, 1, n, out.data_ptr(), H * d, 0, 0, None))
    torch.cuda.synchronize()
    idx = torch.arange(n)
    blk = bt[0, idx // bs].long()
    K, V = (t[blk, :, idx % bs].double().repeat_interleave(H // G, 1) for t in (k, v))
    rows = torch.tensor([bucket(n - 1 - i, 16, 200) for i in range(n)])
    s = torch.cat([torch.einsum("hd,nhd->hn", q[0].double(), K) * 0.1 + rel.double()[rows].t(), sink.double()[:, None]], 1)
    ref = torch.einsum("hn,nhd->hd", torch.softmax(s, -1)[:, :n], V) * mult * torch.sigmoid(gate[0].double())[:, None]
    assert ((out.cpu().double().reshape(H, d) - ref).abs() <= 1.5e-2 * (1 + ref.abs())).all()      # as the tests of chunked attention

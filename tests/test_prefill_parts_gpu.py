"""Context-encoding attention of 3 to 8 query heads on a kv head, where two waves share a head's keys tile by tile (5 heads and more: over two work-groups): against
fp32 attention, at counts of tiles (64 keys) that leave the second wave without one, with one that is partly or wholly ahead of the query, and at grids that put two
blocks on a work-group; 96 keys (one wave) and 97; and grids where one wave a head takes less time."""
import pytest
import torch

from tests.test_ops_gpu import _make_pool, dev, lib, pool_to_native, ref_attention  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,hd,T,pos0", [
    (4, 1, 64, 1, 0), (4, 1, 128, 1, 63), (4, 1, 128, 1, 64), (3, 1, 64, 33, 95), (3, 1, 128, 64, 64), (4, 1, 64, 65, 127), (8, 2, 128, 31, 321), (3, 1, 64, 129, 256),
    (5, 1, 128, 33, 40), (6, 1, 64, 70, 0), (7, 1, 128, 129, 130), (8, 1, 64, 65, 63), (14, 2, 64, 200, 300), (28, 4, 128, 1061, 0), (32, 4, 64, 1030, 31), (20, 4, 128, 1025, 0),
    (32, 8, 128, 1023, 0), (32, 8, 64, 1030, 0), (24, 8, 128, 1057, 70), (4, 1, 128, 33, 64), (3, 1, 64, 32, 64), (4, 1, 64, 33, 63),
    (40, 8, 64, 1200, 0), (32, 8, 128, 1057, 2000),       # (these two: one wave a head, where two would be a second round, and behind a long prefix)
    (32, 8, 128, 512, 0), (32, 8, 64, 513, 0), (24, 4, 128, 512, 5), (20, 4, 64, 513, 0), (5, 1, 64, 97, 0)])      # two heads to a work-group up to 512 tokens here; a third (two) of the groups empty
def test_two_waves_a_head(lib, nh, nkv, hd, T, pos0):  # noqa: F811
    bs, kv_len = 16, pos0 + T
    MB = -(-kv_len // bs) + 1
    nb = 1 + MB
    k, v = _make_pool(nb, bs, nkv, hd, 3)
    pool = dev(pool_to_native(k, v, nb, bs))
    bt = torch.zeros(MB, dtype=torch.int32)
    bt[:MB - 1] = (torch.randperm(nb - 1, generator=torch.Generator().manual_seed(4)) + 1)[:MB - 1].int()
    q = torch.randn(T, nh, hd, generator=torch.Generator().manual_seed(5)).to(torch.bfloat16)
    out, qd, btd = torch.empty(T, nh * hd, dtype=torch.bfloat16, device="cuda"), dev(q), dev(bt)
    lib.check(lib.load_library().mi_op_paged_attn_prefill(qd.data_ptr(), T, pos0, pool.data_ptr(), nb, bs, btd.data_ptr(), MB, nh, nkv, hd, out.data_ptr(), None))
    torch.cuda.synchronize()
    idx = torch.arange(kv_len)
    blk = bt[idx // bs].long()
    kk, vv = k.float().reshape(nb, bs, nkv, hd), v.float().reshape(nb, bs, nkv, hd)
    ref = ref_attention(q.float(), kk[blk, idx % bs], vv[blk, idx % bs], pos0 + torch.arange(T))
    assert (out.cpu().float() - ref).abs().max().item() < 0.03     # P is rounded to bf16 in front of its product with V

"""The row norms on both sides of their rules: a float4 per thread with every request in front (up to 512 rows of up to 4096), and the loops beyond."""
import pytest
import torch

from oracle import vimesun as V
from tests.test_ops_gpu import dev, lib  # noqa: F401  (lib: the fixture)
from tests.test_vimesun_gpu import pad16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H", [(1, 4), (3, 260), (512, 4096), (513, 4096), (2, 4100), (40, 8192)])
def test_rmsnorm(lib, T, H):  # noqa: F811
    g = torch.Generator().manual_seed(T + H)
    x, w = torch.randn(T, H, generator=g) * 3, 1 + 0.1 * torch.randn(H, generator=g)
    y = torch.empty(T, H, dtype=torch.bfloat16, device="cuda")
    xd, wd = dev(x), dev(w)
    lib.check(lib.load_library().mi_op_rmsnorm(xd.data_ptr(), wd.data_ptr(), T, H, 1e-5, y.data_ptr(), None))
    torch.cuda.synchronize()
    x, w = x.double(), w.double()
    ref = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * w
    assert ((y.cpu().double() - ref).abs() <= 2.0 ** -8 * 1.01 * ref.abs() + 1e-6).all()      # one bf16 rounding of an fp32 result


@pytest.mark.parametrize("T,D", [(512, 2048), (513, 2048), (2, 4096), (3, 4099)])
def test_layernorm(lib, T, D):  # noqa: F811
    g = torch.Generator().manual_seed(T + D)
    ld, ldy = pad16(D), (D + 63) // 64 * 64
    x, w, b = torch.zeros(T, ld), torch.zeros(ld), torch.zeros(ld)
    x[:, :D] = torch.randn(T, D, generator=g) + 5.0
    w[:D], b[:D] = torch.randn(D, generator=g), torch.randn(D, generator=g)
    y = torch.zeros(T, ldy, device="cuda")
    xd, wd, bd = dev(x), dev(w), dev(b)
    lib.check(lib.load_library().mi_op_layernorm2(xd.data_ptr(), T, D, ld, 1e-3, wd.data_ptr(), bd.data_ptr(), y.data_ptr(), None, None, None, ldy, 1, None))
    torch.cuda.synchronize()
    ref = V.layer_norm(x[:, :D].double(), w[:D].double(), b[:D].double(), 1e-3)
    got = y.cpu().double()
    assert (got[:, D:] == 0).all() and ((got[:, :D] - ref).abs() <= 1e-5 * (1 + ref.abs())).all()


# slabs: one, all of a batch of requests (5), the first of a second batch, two batches; rows: a float4 per thread, the loop of a long row, the loop of many rows
@pytest.mark.parametrize("T,H", [(1, 128), (7, 4096), (5, 4224), (513, 256)])
@pytest.mark.parametrize("KS", [1, 2, 5, 6, 8, 10])
@pytest.mark.parametrize("form", ["bf16", "rinv", "fp8"])
@pytest.mark.parametrize("bias,row_scale", [(False, False), (True, True)])
def test_sums_of_k_slices(lib, T, H, KS, form, bias, row_scale):  # noqa: F811
    g = torch.Generator().manual_seed(T + H + KS)
    x, slab, sc = torch.randn(T, H, generator=g) * 3, torch.randn(KS, T, H, generator=g), 0.5 + torch.rand(H, generator=g)
    w, b, rs = 1 + 0.1 * torch.randn(H, generator=g), torch.randn(H, generator=g), 0.5 + torch.rand(T, generator=g)
    d = [dev(t) for t in (x, slab, sc, b, rs, w)]
    out, y = torch.full((T, H), float("nan"), device="cuda"), torch.empty(T, H, dtype=torch.bfloat16, device="cuda")
    rinv, x8 = torch.full((T,), float("nan"), device="cuda"), torch.zeros(H // 128, T, 128, dtype=torch.uint8, device="cuda")
    scale8 = d[4] if row_scale else torch.empty(T, device="cuda")      # (the models read and write the same array)
    lib.check(lib.load_library().mi_op_rmsnorm_slabs(
        d[0].data_ptr(), d[1].data_ptr(), KS, d[2].data_ptr(), d[3].data_ptr() if bias else None, d[4].data_ptr() if row_scale else None, d[5].data_ptr(), T, H, 1e-5,
        out.data_ptr(), None if form == "fp8" else y.data_ptr(), rinv.data_ptr() if form == "rinv" else None, x8.data_ptr() if form == "fp8" else None,
        scale8.data_ptr() if form == "fp8" else None, None))
    torch.cuda.synchronize()
    x, slab, sc, b, rs, w = (t.double() for t in (x, slab, sc, b, rs, w))
    if not bias:
        b = torch.zeros_like(b)
    if not row_scale:
        rs = torch.ones_like(rs)
    factor = sc * rs[:, None]
    h, size = x + slab.sum(0) * factor + b, x.abs() + slab.abs().sum(0) * factor + b.abs()
    got = out.cpu().double()
    assert ((got - h).abs() <= (KS + 4) * 2.0 ** -24 * size).all()      # KS - 1 additions and four more operations, half a place of fp32 each
    r = torch.rsqrt(got.pow(2).mean(-1, keepdim=True) + 1e-5)
    if form == "rinv":
        assert ((rinv.cpu().double() - r[:, 0]).abs() <= 1e-6 * r[:, 0]).all()
        assert torch.equal(y.cpu(), (out.cpu() * w.float()).to(torch.bfloat16))
        return
    ref = got * r * w
    if form == "bf16":
        assert ((y.cpu().double() - ref).abs() <= 2.0 ** -8 * 1.01 * ref.abs()).all()      # one bf16 rounding of an fp32 result
        return
    s8 = scale8.cpu().double()
    assert ((s8 - ref.abs().amax(-1) / 448).abs() <= 2.0 ** -8 * 1.01 * s8).all()
    got8 = x8.cpu().view(torch.float8_e4m3fn).double().permute(1, 0, 2).reshape(T, H) * s8[:, None]
    assert ((got8 - ref).abs() <= (2.0 ** -4 + 2.0 ** -8) * 1.01 * ref.abs() + 2.0 ** -10 * s8[:, None]).all()      # e4m3 of a bf16; half its least step below 2^-6


# the row over four work-groups: one wave and one number a thread of it, the last wave partly idle, sixteen waves; one batch of slabs and two
@pytest.mark.parametrize("T,H", [(1, 16), (5, 3584), (32, 4096), (3, 4112), (2, 16384)])
@pytest.mark.parametrize("KS,bias,partial", [(0, False, False), (0, False, True), (1, True, False), (5, False, False), (8, True, False)])
def test_row_parts(lib, T, H, KS, bias, partial):  # noqa: F811
    g = torch.Generator().manual_seed(T + H + KS)
    x, slab, sc = torch.randn(T, H, generator=g) * 3, torch.randn(max(KS, 1), T, H, generator=g), 0.5 + torch.rand(H, generator=g)
    w, b, p = 1 + 0.1 * torch.randn(H, generator=g), torch.randn(H, generator=g), torch.randn(T, H, generator=g)
    d = [dev(t) for t in (x, p, slab, sc, b, w)]
    out, y, ss = torch.full((T, H), float("nan"), device="cuda"), torch.empty(T, H, dtype=torch.bfloat16, device="cuda"), torch.full((T, 4), float("nan"), device="cuda")
    lib.check(lib.load_library().mi_op_rmsnorm_parts(
        d[0].data_ptr(), d[1].data_ptr() if partial else None, d[2].data_ptr() if KS else None, KS, d[3].data_ptr(), d[4].data_ptr() if bias else None, d[5].data_ptr(), T, H,
        out.data_ptr(), y.data_ptr(), ss.data_ptr(), None))
    torch.cuda.synchronize()
    h = x.double() + (p.double() if partial else 0) + (slab.double().sum(0) * sc.double() + (b.double() if bias else 0) if KS else 0)
    assert ((out.cpu().double() - h).abs() <= 2e-6 * (1 + h.abs()) * max(KS, 1)).all()              # KS + 2 fp32 roundings of sums of this size
    ref = h * w.double()
    assert ((y.cpu().double() - ref).abs() <= 2.0 ** -8 * 1.01 * ref.abs() + 1e-5 * max(KS, 1)).all()
    sq = h.reshape(T, 4, H // 4).pow(2).sum(-1)
    assert ((ss.cpu().double() - sq).abs() <= 1e-5 * sq).all()

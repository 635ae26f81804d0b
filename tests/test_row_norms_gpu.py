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

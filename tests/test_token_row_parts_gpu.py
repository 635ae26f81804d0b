"""The row kernel of the sandwich blocks with a work-group to each part of a norm: one wave a part, several, one part of a whole row, the most columns it takes and the most rows with
a convolution's state, whose pages the parts share; and without one, rows of prompts on both sides of where the general kernel takes over."""
import pytest
import torch

from tests import test_rapodra_gpu as T
from tests.rapodra_cases import config, dense, latent
from tests.test_rapodra_gpu import R, lib, sandwich, test_convolution_over_portions_pages_and_sequences as convolutions, test_norms_around_the_residual_sum as norms  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("T,D,groups", [(1, 256, 1), (4, 2048, 4), (3, 3072, 2), (32, 4096, 16), (32, 4096, 1)])
def test_norms(lib, T, D, groups, f32):  # noqa: F811
    norms(lib, T, D, groups, f32)


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("D,taps,bs", [(512, 4, 16), (1536, 2, 32), (512, 1, 16)])
def test_convolutions(lib, D, taps, bs, f32):  # noqa: F811
    convolutions(lib, D, taps, bs, f32)


# prompts: up to 512 rows, up to 2048 columns and parts of 256 columns this kernel, else the general one (256 threads a row with four float4 each, three, and a third that a quarter of them has)
@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("T,D,groups", [(300, 768, 1), (512, 4096, 1), (513, 4096, 1), (513, 4096, 16), (513, 4096, 8), (700, 2048, 1), (700, 2304, 1), (700, 2304, 9), (600, 3072, 3)])
def test_norms_of_prompts(lib, T, D, groups, f32):  # noqa: F811
    norms(lib, T, D, groups, f32)


# ... their sources experts' rows
@pytest.mark.parametrize("T,D,top", [(300, 512, 3), (512, 2560, 5), (513, 2560, 5)])
def test_experts_rows_of_prompts(lib, T, D, top):  # noqa: F811
    torch.manual_seed(T)
    x, y, p = torch.randn(T, D), torch.randn(T * top, D), torch.softmax(torch.randn(T, top), -1)
    w, wn = torch.randn(D), torch.randn(D)
    got_x, got = sandwich(lib, x, T, D, 1, 1e-3, 1, y=y, pair_w=p, w_post=w, w_pre=wn)
    ref_x = x.double() + R.group_rms((p[:, :, None] * y.view(T, top, D)).sum(1).double(), w.double(), 1, 1e-3)
    assert ((got_x - ref_x).abs() <= 2e-5 * (1 + ref_x.abs())).all()
    ref = R.group_rms(ref_x, wn.double(), 1, 1e-3)
    assert ((got - ref).abs() <= 2e-5 * (1 + ref.abs())).all()


# ... and the slices of a deep feed-forward's sum
def test_slices_left_to_the_norms_of_prompts():
    cfg = config(256, 160, [latent(4, 32, 32, 64, 40, dense(6144)), latent(4, 32, 32, 64, 48, dense(6144), kv_from=0)], groups=1)
    w = T.weights(cfg, 9)
    r = T.replay(cfg, w, "bfloat16", max_tokens=512, max_live=1)
    toks = T.tokens(cfg, w, 200, 7100)
    worst = T.error(T.score(r, toks, [130, 70]), T.reference("deep prompts", cfg, w, toks, "bfloat16"))
    assert worst <= T.LIMIT["bfloat16"], worst
    r.engine.close()

"""Token generation's row kernel of the sandwich blocks with a work-group to each part of a norm: one wave a part, several, one part of a whole row, and the most rows and
columns it takes; with convolutions whose state the parts share pages of."""
import pytest

from tests.test_rapodra_gpu import lib, test_convolution_over_portions_pages_and_sequences as convolutions, test_norms_around_the_residual_sum as norms  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("T,D,groups", [(1, 256, 1), (4, 2048, 4), (3, 3072, 2), (32, 4096, 16), (32, 4096, 1)])
def test_norms(lib, T, D, groups, f32):  # noqa: F811
    norms(lib, T, D, groups, f32)


@pytest.mark.parametrize("f32", [0, 1])
@pytest.mark.parametrize("D,taps,bs", [(512, 4, 16), (1536, 2, 32), (512, 1, 16)])
def test_convolutions(lib, D, taps, bs, f32):  # noqa: F811
    convolutions(lib, D, taps, bs, f32)

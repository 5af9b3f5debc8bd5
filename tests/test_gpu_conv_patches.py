"""The network's layers at the edges of the 16 x 8 patches their kernels stage:
one pixel, less than, exactly and just over a patch, several patches and slices,
more patches than the weight gradient has blocks."""
import pytest

from tests import test_gpu_learned as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin", [8, 32])
@pytest.mark.parametrize("shape", [(1, 1, 1), (15, 7, 1), (16, 8, 1), (17, 9, 2), (48, 33, 3)])
def test_layer_matches_oracle_at_patch_edges(cin, shape):
    T.test_conv_forward_backward_match_oracle(cin, shape)

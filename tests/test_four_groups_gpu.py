"""NVFP4 tile kernels whose workgroups multiply quarters of K in four groups of two waves (K a multiple of 1024): the
oracle's values, bias and residual included, and the same bits on every repetition, at two, three and more 256-K blocks
per group, 64 x 128 and 128 x 128 workgroup tiles, ragged edges, and from the first row past the weight-streaming kernel."""
import pytest

from test_tile_split_gpu import test_two_groups_per_workgroup_match_the_oracle as _matches_the_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(129, 8192, 2048), (161, 4616, 3072), (257, 136, 2048), (333, 1000, 5120), (512, 4096, 4096),
                                   (511, 200, 14336), (600, 4100, 2048), (1025, 3072, 3072), (512, 8192, 6144)])
def test_four_groups_match_the_oracle(m, n, k):
    _matches_the_oracle(m, n, k)

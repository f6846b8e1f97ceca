"""The fused prefill kernel (csrc/prefill.hip): K ranges of one to a few
32-row stages, and the partial sums of a split product, whose rows and columns
past the output are dropped by the buffer's bounds, against the float64 oracle
at the tolerance of the other products."""
import pytest

from tests.test_decode_tiles_gpu import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["union", "dense"])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 160, 192, 224])
def test_few_stages(K, mode):
    _check(70, K, 400, 8, 32, "float16", mode)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("mode", ["union", "dense"])
@pytest.mark.parametrize("M,N", [(65, 16), (127, 272), (129, 400), (200, 1040)])
def test_split_partials(M, N, mode, dtype):
    """Two to four K ranges (K = 1056: whole stages, unequal), the last row and
    column blocks partial."""
    _check(M, 1056, N, 8, 32, dtype, mode)

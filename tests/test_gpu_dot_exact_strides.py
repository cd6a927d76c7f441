"""GPU: the EXACT dot on both sides of the rule that gives a strided dot one launch or two (strides of 8 and more count as 8
lines an element, at most 49152 of both vectors and 6144 elements), against the oracle's correctly rounded sum."""
import pytest

from test_gpu_dot_exact_small import test_dot_exact_small as dot_exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ("uniform", "cancel", "far"))
@pytest.mark.parametrize("n,incx,incy", [(6144, 2, 2), (6145, 2, 2), (6144, 1, 7), (6144, 1, 8), (6144, 4, 4), (6143, 5, 4),
                                         (3072, 64, 8), (3073, 8, 64), (5461, 1, 65), (5462, 65, 1), (8192, 2, 1)])
def test_dot_exact_either_side_of_the_rule(O, Q, cuda, n, incx, incy, kind):
    dot_exact(O, Q, cuda, n, incx, incy, kind)

"""The adjoint's reverse pass at the widths of its wavefront rows: 64, 32, 16
or 4 cells of x a row, several rows j a wavefront with a remainder, and more
than one wavefront along x -- the dot-product check of test_gpu_adjoint.py
(1e-6 relative, central differences of the GPU step)."""
import pytest

from tests import test_gpu_adjoint as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,split", [((4, 5, 4), 0), ((8, 6, 8), 0), ((32, 7, 4), 1), ((64, 5, 8), 1),
                                         ((128, 9, 8), 1)])
def test_rows_of_a_wavefront(shape, split):
    A.test_step_adjoint_dot_product(shape, split)

"""Contiguous single-rank lines in planes of few lines, which go through the
solver as one plane, and in planes that leave part of a workgroup idle: bit
for bit against the oracle, at line lengths around its 16-row chunks."""
import pytest

from tests.test_gpu_tdma_exact_edges import test_contiguous_lines as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(17, 1, 70), (16, 2, 32), (31, 5, 30), (32, 32, 3), (33, 33, 3), (47, 63, 2), (2, 7, 10),
                                   (100, 1, 1)])
@pytest.mark.parametrize("cyclic", [False, True])
def test_planes_of_few_lines(shape, cyclic):
    check(shape, cyclic)

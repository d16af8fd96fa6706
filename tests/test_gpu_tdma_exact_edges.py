"""The single-rank line solves at the edges of their layout, bit for bit
against the oracle (the same operations in the same order): line lengths
around the 8-row chunks of strided lines, the 16-row chunks of contiguous
ones and the rows kept in LDS (104, 52, 26 for 1, 2, 4 wavefronts a CU), and
line counts around a wavefront."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_tdma import _torch, dominant

pytestmark = pytest.mark.gpu


def _check(got, exp):
    for g, e, name in zip(got, exp, "ACD"):
        assert np.array_equal(g, e), f"{name} differs: {np.abs(g - e).max()}"


@pytest.mark.parametrize("n_sys,n_row", [(2, 2), (63, 4), (64, 9), (65, 10), (64, 11), (100, 18), (130, 103),
                                         (64, 104), (65, 105), (64, 106), (16385, 54), (33000, 27), (70000, 30)])
@pytest.mark.parametrize("cyclic", [False, True])
def test_strided_lines(n_sys, n_row, cyclic):
    import torch
    from pascal_tcs_amd import ptdma
    a, b, c, d = dominant(np.random.default_rng(n_sys + n_row), (n_row, n_sys))
    A, B, C, D = _torch((a, b, c, d))
    f = ptdma.PaScaL_TDMA_many_solve_cycle if cyclic else ptdma.PaScaL_TDMA_many_solve
    f(None, A, B, C, D, n_sys, n_row)
    torch.cuda.synchronize()
    O.ptdma_many_solve(a, b, c, d, cyclic=cyclic)
    _check((A.cpu().numpy(), C.cpu().numpy(), D.cpu().numpy()), (a, c, d))


@pytest.mark.parametrize("shape", [(2, 63, 2), (3, 64, 2), (16, 65, 3), (17, 64, 2), (18, 7, 3), (33, 130, 2), (48, 64, 1),
                                   (1030, 3, 2)])
@pytest.mark.parametrize("cyclic", [False, True])
def test_contiguous_lines(shape, cyclic):
    import torch
    from pascal_tcs_amd import ptdma
    n1, n2, n3 = shape
    arrs = dominant(np.random.default_rng(sum(shape)), (n3, n2, n1))
    A, B, C, D = _torch(arrs)
    ptdma.axis_solve(A, B, C, D, 0, cyclic)
    torch.cuda.synchronize()
    flat = [np.ascontiguousarray(x.transpose(2, 0, 1)).reshape(n1, -1) for x in arrs]
    O.ptdma_many_solve(*flat, cyclic=cyclic)
    exp = [f.reshape(n1, n3, n2).transpose(1, 2, 0) for f in flat]
    _check((A.cpu().numpy(), C.cpu().numpy(), D.cpu().numpy()), (exp[0], exp[2], exp[3]))

"""tcs_step, whose kernels write the periodic ghosts and carry the wall rows
over, against the routines called one by one with their ghost-cell updates:
whole arrays, ghosts and wall rows included, over steps in a row, after
fields (wall rows and ghosts of no periodic kind among them) were written
in between, and after reads.  The exact form gives the same bits; the fast
form 1e-12 of a field's size a step (its bound against the oracle), the mixed
form the 2e-6 of FP32 rows."""
import numpy as np
import pytest

from tests.cases import max_rel, small_config

pytestmark = pytest.mark.gpu
NAMES = ("T", "U", "V", "W", "P", "dU", "dV", "dW", "dP", "dPhat", "dP0")


def _noise(s, names, seed):
    rng = np.random.default_rng(seed)
    for n in names:
        a = s.get(n)
        s.set(n, a + 1e-3 * max(1.0, float(np.max(np.abs(a)))) * rng.standard_normal(a.shape))


@pytest.mark.parametrize("form,split,bound", [(0, 0, 0.0), (0, 1, 0.0), (1, 1, 3e-12), (2, 1, 6e-6)])
@pytest.mark.parametrize("shape", [(4, 3, 4), (16, 33, 8), (128, 18, 16), (64, 40, 64),
                                   (256, 129, 256)])  # the last past 2^23 cells
def test_steps_against_routines(shape, form, split, bound):
    from pascal_tcs_amd.solver import TCSSolver
    cfg = small_config(*shape, DeltaT=0.2)
    a, b = (TCSSolver(cfg, tdma_split=split, precision=form) for _ in range(2))
    for s in (a, b):
        s.setup_seeded(amp=0.05, seed=31)
    dt = cfg.dtStart
    edits = [NAMES, (), ("U", "dW"), ("T",), ()]  # written before each group of two steps
    for g, names in enumerate(edits):
        for s in (a, b):
            _noise(s, names, 100 + g)
        for _ in range(2):
            a.step(dt)
            b.step_routines(dt)
        errs = {n: max_rel(a.get(n), b.get(n)) for n in NAMES}
        print(shape, form, split, g, {n: f"{e:.1e}" for n, e in errs.items()}, flush=True)
        assert max(errs.values()) <= bound * 2 * (g + 1), errs
        for s in (a, b):
            s.set("U", b.get("U"))  # a read and a write between steps
    a.close()
    b.close()

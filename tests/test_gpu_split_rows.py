"""y lines split in parts of every size from 8 to 16 rows (of one size, and of
two with the longer ones first), one step against the oracle.  The bounds are
those of test_gpu_split_plans.py for long y lines (1e-10 of a field's size in
FP64) and, for the mixed form, 2e-4 (the FP32 rounding of its increments, of which the projection
cancels all but a thousandth)."""
import pytest

from tests.cases import FIELDS, WALLS, make_oracle, max_rel, small_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,bound", [(1, 1e-10), (2, 2e-4)])
@pytest.mark.parametrize("n2", [257, 288, 300, 331, 352, 383, 400, 431, 449, 480, 511, 512])
def test_step_of_every_part_size(n2, precision, bound):
    from pascal_tcs_amd.solver import TCSSolver
    cfg = small_config(8, n2, 8, DeltaT=0.2)
    s = TCSSolver(cfg, tdma_split=1, precision=precision)
    s.setup_seeded(amp=0.05, seed=31)
    o = make_oracle(cfg)
    for n in FIELDS:
        o.f[n][...] = s.get(n)
    for w in WALLS:
        o.bc[w][...] = s.get_wall(w)
    o.step(cfg.dtStart)
    s.step(cfg.dtStart)
    errs = {n: max_rel(s.get(n), o.f[n]) for n in ("T", "U", "V", "W", "P")}
    s.close()
    print(n2, precision, {n: f"{e:.1e}" for n, e in errs.items()}, flush=True)
    assert max(errs.values()) <= bound, errs

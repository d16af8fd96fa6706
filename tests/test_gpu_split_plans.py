"""The fast form's splits of its ADI lines: 4- and 8-row parts (few lines, with
remainders), 64 and 128 parts (lines of more than 512 rows, along x, y and z)
and lines past the split range, one step against the oracle.  The bound is
the fast form's: 1e-12 of each field's size a step at these sizes; the
oracle's V and P of the long y lines are themselves only good to about 1e-11
(their Poisson systems), hence 1e-10 there."""
import numpy as np
import pytest

from tests.cases import FIELDS, WALLS, make_oracle, max_rel, small_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,bound", [((64, 12, 8), 1e-12), ((16, 31, 64), 1e-12), ((128, 49, 16), 1e-12),
                                         ((8, 65, 256), 1e-12), ((1024, 9, 8), 1e-12), ((2048, 5, 4), 1e-12),
                                         ((4096, 4, 4), 1e-12), ((8, 6, 1024), 1e-12), ((8, 530, 8), 1e-10)])
def test_step_of_every_plan(shape, bound):
    from pascal_tcs_amd.solver import TCSSolver
    cfg = small_config(*shape, DeltaT=0.2)
    s = TCSSolver(cfg, tdma_split=1, precision=1)
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
    print(shape, {n: f"{e:.1e}" for n, e in errs.items()}, flush=True)
    assert max(errs.values()) <= bound, errs

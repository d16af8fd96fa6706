"""x lines of 4096 points, the longest the forward transform takes: one step in
every form of the arithmetic against the oracle (1e-12 of each field's size)."""
import pytest

from tests.cases import FIELDS, WALLS, make_oracle, max_rel, small_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
def test_step_with_4096_points_along_x(precision):
    from pascal_tcs_amd.solver import TCSSolver
    cfg = small_config(4096, 4, 4, DeltaT=0.2)
    s = TCSSolver(cfg, precision=precision)
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
    assert max(errs.values()) <= 1e-12, errs

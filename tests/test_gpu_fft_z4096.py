"""z lines of 4096 points, the longest the transforms take (67.6 KB of LDS a
line), over few x lines: one step in both FP64 forms against the
oracle, 1e-12 of each field's size as for x lines of that length.  (The
exact form is not bit for bit the oracle's at 4096 points: one of the 2048
twiddles comes out one unit in the last place apart from libm's sin and cos
and from its sincos, which the two compilers choose between.)"""
import pytest

from tests.cases import FIELDS, WALLS, make_oracle, max_rel, small_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(4, 4, 4096), (8, 5, 4096)])
def test_step_with_4096_points_along_z(shape, precision):
    from pascal_tcs_amd.solver import TCSSolver
    cfg = small_config(*shape, DeltaT=0.2)
    s = TCSSolver(cfg, tdma_split=0, precision=precision)
    s.setup_seeded(amp=0.05, seed=37)
    o = make_oracle(cfg)
    for n in FIELDS:
        o.f[n][...] = s.get(n)
    for w in WALLS:
        o.bc[w][...] = s.get_wall(w)
    o.step(cfg.dtStart)
    s.step(cfg.dtStart)
    errs = {n: max_rel(s.get(n), o.f[n]) for n in ("T", "U", "V", "W", "P")}
    s.close()
    print(shape, precision, {n: f"{e:.1e}" for n, e in errs.items()}, flush=True)
    assert max(errs.values()) <= 1e-12, errs

"""Every length of the x and z transforms, with line counts that leave a
remainder in the workgroups that take several lines: one step against the
oracle, bit for bit in the exact form, within the fast form's 1e-12 of a
field's size otherwise."""
import pytest

from tests.cases import FIELDS, WALLS, make_oracle, max_rel, small_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,bound", [(0, 0.0), (1, 1e-12)])
@pytest.mark.parametrize("shape", [(4, 5, 64), (32, 4, 128), (64, 4, 256), (128, 4, 512), (256, 4, 1024), (512, 4, 4),
                                   (1024, 4, 8), (2048, 4, 4), (16, 4, 2048)])
def test_step_at_every_length(shape, precision, bound):
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
    assert max(errs.values()) <= bound, errs

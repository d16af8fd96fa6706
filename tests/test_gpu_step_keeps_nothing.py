"""What a step writes does not depend on the steps before it: dV's wall rows,
written through a device pointer taken before an earlier step, are zero after
the next one (dV is not exchanged, so the pointer stays valid), and dP0's
ghosts survive a step taken after others were captured into a graph and not
yet run."""
import numpy as np
import pytest

from tests.cases import small_config

pytestmark = pytest.mark.gpu
FORMS = [(0, 0), (0, 1), (1, 1), (2, 1)]


def _solver(precision, split, shape=(16, 12, 8)):
    from pascal_tcs_amd.solver import TCSSolver
    cfg = small_config(*shape, DeltaT=0.2)
    s = TCSSolver(cfg, tdma_split=split, precision=precision)
    s.setup_seeded(amp=0.05, seed=31)
    return s, cfg


@pytest.mark.parametrize("precision,split", FORMS[:3])  # the mixed form's dV is an FP32 array behind the entries
@pytest.mark.parametrize("shape", [(16, 12, 8), (4, 3, 4), (8, 530, 8)])
def test_wall_rows_written_through_an_earlier_pointer(precision, split, shape):
    import torch
    s, cfg = _solver(precision, split, shape)
    p, pitch = s.device_ptr("dV"), s.device_pitch()
    s.step(cfg.dtStart)
    s.sync()

    class View:
        __cuda_array_interface__ = {"shape": (s.shape[0] * s.shape[1] * pitch,), "typestr": "<f8", "data": (p, False),
                                    "version": 2}
    dV = torch.as_tensor(View(), device="cuda").view(s.shape[0], s.shape[1], pitch)
    dV[:, 0, :s.shape[2]] = 7.0
    dV[:, -1, :s.shape[2]] = -5.0
    torch.cuda.synchronize()
    s.step(cfg.dtStart)
    got = s.get("dV")
    s.close()
    assert not got[:, 0].any() and not got[:, -1].any()


@pytest.mark.parametrize("precision,split", FORMS)
def test_step_after_a_capture(precision, split):
    import torch
    pair = [_solver(precision, split)[0] for _ in range(2)]
    dt = 1e-3
    rng = np.random.default_rng(5)
    ghosts = 1e-2 * rng.standard_normal(pair[0].shape)
    for s in pair:
        s.step(dt)
        s.set("dP0", ghosts)
        s.sync()
    a, b = pair
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(torch.cuda.ExternalStream(b.stream())):
        graph.capture_begin()
        b.step(dt)
        b.step(dt)
        graph.capture_end()
    for _ in range(3):  # two steps of its own, which give back the captured ones' buffers, and a replay
        for s in pair:
            s.step(dt)
        assert np.array_equal(a.get("dP0"), b.get("dP0"))
        for s in pair:
            s.step(dt)
        a.step(dt)
        a.step(dt)
        b.sync()
        with torch.cuda.stream(torch.cuda.ExternalStream(b.stream())):
            graph.replay()
        b.sync()
        for n in ("T", "U", "V", "W", "P", "dU", "dV", "dW", "dPhat", "dP0"):
            assert np.array_equal(a.get(n), b.get(n)), n
    for s in pair:
        s.close()

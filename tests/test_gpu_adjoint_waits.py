"""tcs_adjoint_step returns with its work done: the context's stream is idle
when it does, and a buffer that a copy before it reads may be written again."""
import pytest

from tests.cases import small_config

pytestmark = pytest.mark.gpu


def test_stream_is_idle_after_the_adjoint_step():
    import torch
    from pascal_tcs_amd.adjoint import StepAdjoint
    from pascal_tcs_amd.solver import TCSSolver
    cfg = small_config(128, 64, 128, DeltaT=0.2)
    s = TCSSolver(cfg)
    s.setup_seeded(amp=0.05, seed=3)
    adj, stream = StepAdjoint(s), torch.cuda.ExternalStream(s.stream())
    for _ in range(3):
        adj.add_nusselt(1.0)
        adj.step(1e-4)
        assert stream.query()
    s.close()

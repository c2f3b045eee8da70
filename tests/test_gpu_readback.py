"""Field reads: below and at the size from which chunks go through pinned
memory, at the sizes where the chunk grows, and lengths that leave a short last
chunk or fewer chunks than ring slots.  What was written comes back bit for
bit, into pageable and into pinned memory, right after steps and on a second
read through the same ring."""
import numpy as np
import pytest
import torch

from dtmaxwell4_amd import abi, configs

pytestmark = pytest.mark.gpu

MB = 1 << 18  # floats of a megabyte


@pytest.mark.parametrize("shape", [(4, 4, 4), (1, 1, MB - 1), (1, 1, MB), (1, 64, MB // 64 + 1), (2, 512, 1024),
                                   (1, 1031, 1019), (2, 2, MB), (4, 1024, 1024), (4, 1024, 1025), (37, 331, 1013)])
def test_field_read_returns_what_was_written(shape):
    from dtmaxwell4_amd.solver import Solver
    cfg = abi.default_config(*shape, 0.05, 0.05, 0.05, configs.dt_for(0.05, 0.05, 0.05))
    s = Solver(cfg)
    s.step(1)
    rng = np.random.default_rng(3)
    for comp in (abi.EX, abi.HZ):
        a = rng.standard_normal(shape).astype(np.float32)
        s.set_field(comp, a)
        assert np.array_equal(s.field(comp), a)
        pin = torch.zeros(shape, pin_memory=True)
        abi.check(s.L.dtm_field_read(s.h, comp, pin.data_ptr()), "dtm_field_read")
        assert np.array_equal(pin.numpy(), a)
        assert np.array_equal(s.field(comp), a)
    s.close()

"""A solver's first reads of a mid-size field are plain copies, later ones go
through the pinned ring, larger fields take it at once and smaller ones follow
when it is there: each read returns what was written, in any order of sizes'
turns (FP16 reads go through a converted copy)."""
import numpy as np
import pytest

from dtmaxwell4_amd import abi, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(100, 100, 110), (128, 128, 128), (163, 155, 157), (160, 160, 163)])
@pytest.mark.parametrize("storage", [abi.STORE_FP32, abi.STORE_FP16])
def test_reads_in_a_row(shape, storage):
    from dtmaxwell4_amd.solver import Solver
    cfg = abi.default_config(*shape, 0.05, 0.05, 0.05, configs.dt_for(0.05, 0.05, 0.05))
    cfg.storage = storage
    s = Solver(cfg)
    rng = np.random.default_rng(4)
    a = [rng.standard_normal(shape, dtype=np.float32).astype(np.float16).astype(np.float32) for _ in range(3)]
    for turn in range(4):
        for c in range(3):
            s.set_field(c, a[(c + turn) % 3])
        for c in range(3):
            assert np.array_equal(s.field(c), a[(c + turn) % 3])
    s.close()

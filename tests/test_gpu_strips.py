"""Planes larger than what an XCD's waves hold at once (384 blocks of 64 chunks in
FP32, 512 in FP16) run in strips.  Random fields in every cell, a few steps
against the FP64 oracle: two and three strips, the last one smaller, ragged z
extents, a periodic grid, the split layer, and FP16 with the hole that an FP32 zone
leaves in the plain launch.  1e-5 in relative L2 (the bound of the FP32 path);
FP16 2e-2 (that of FP16 against FP32).  Slab by slab, one call equals single steps."""
import numpy as np
import pytest

from conftest import rel_l2
from dtmaxwell4_amd import abi, configs
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

D = 0.05


def start(make, n, storage, periodic=0, split=0, zone=None):
    cfg = abi.default_config(*n, D, D, D, configs.dt_for(D, D, D))
    if periodic:
        cfg.bc[:] = [abi.BC_PERIODIC] * 3
    else:
        cfg.npml[:] = [3, 4, 5, 4, 6, 3]
    cfg.pml_kind = abi.PML_SPLIT if split else abi.PML_CPML
    cfg.storage = storage
    if storage:
        cfg.scale_e_log2[:] = cfg.scale_h_log2[:] = [10] * 3
    s = make(cfg)
    if zone:
        s.set_fp32_zone(*zone)
    rng = np.random.default_rng(5)
    for c in range(6):
        s.set_field(c, rng.standard_normal(n, dtype=np.float32))
    return s


@pytest.mark.parametrize("n,storage,periodic,split,zone", [
    ((50, 400, 420), abi.STORE_FP32, 0, 0, None),
    ((50, 257, 387), abi.STORE_FP32, 0, 0, None),
    ((20, 1000, 301), abi.STORE_FP32, 0, 0, None),
    ((40, 512, 256), abi.STORE_FP32, 1, 0, None),
    ((41, 300, 350), abi.STORE_FP32, 0, 1, None),
    ((60, 400, 420), abi.STORE_FP16, 0, 0, None),
    ((60, 400, 420), abi.STORE_FP16, 0, 0, (20, 41, 150, 171, 200, 221)),
    ((60, 400, 420), abi.STORE_FP16, 0, 0, (50, 60, 380, 400, 1, 22)),
])
def test_strips_against_the_oracle(n, storage, periodic, split, zone):
    from dtmaxwell4_amd.solver import Solver
    g, o = start(Solver, n, storage, periodic, split, zone), start(Oracle, n, 0, periodic, split)
    g.step(6)
    o.step(6)
    err = rel_l2(g.fields(), o.fields())
    g.close()
    o.close()
    print("rel-L2", err)
    assert err <= (1e-5 if storage == abi.STORE_FP32 else 2e-2)


@pytest.mark.parametrize("n,storage", [((70, 384, 420), abi.STORE_FP32), ((150, 401, 403), abi.STORE_FP16)])
def test_strips_slab_by_slab(n, storage):
    from dtmaxwell4_amd.solver import Solver
    out = []
    for calls in ([1] * 13, [13]):
        s = start(Solver, n, storage)
        for m in calls:
            s.step(m)
        out.append(s.fields())
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)

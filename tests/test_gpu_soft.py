"""Soft sources, subtracted inside the E sweep (FP32, at most four, no folded
plane wave, CPML) or by a launch after it, against the FP64 oracle: every cell
of a chunk, all components, several sources in one chunk and plane, next to the
boundaries and in the layer, odd z extents, more sources than the sweep takes,
and the configurations that keep the launch.  1e-5 in relative L2 (the bound of
the FP32 path); FP16: 2e-2 (test_gpu_parity's bound of FP16 against FP32)."""
import math

import numpy as np
import pytest

from conftest import rel_l2
from dtmaxwell4_amd import abi, configs
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

D = 0.05


def build(make, n, sources, storage, split, wave):
    cfg = abi.default_config(*n, D, D, D, configs.dt_for(D, D, D))
    cfg.npml[:] = [4] * 6
    cfg.storage = storage
    cfg.pml_kind = abi.PML_SPLIT if split else abi.PML_CPML
    cfg.nsoft = len(sources)
    for q, (comp, i, j, k) in enumerate(sources):
        so = cfg.soft[q]
        so.comp, so.i, so.j, so.k = comp, i, j, k
        so.waveform, so.amp, so.w, so.tw, so.t0 = abi.WAVE_GAUSS_SINE, 5.0 + q, 2 * math.pi, 0.3, 0.2
    if wave:
        t = cfg.tfsf
        t.kind, t.waveform, t.sf_inside = abi.TFSF_PLANE, abi.WAVE_GAUSS_SINE, 0
        t.box[:] = [6 * D, (n[0] - 6) * D, 6 * D, (n[1] - 6) * D, 6 * D, (n[2] - 6) * D]
        t.w, t.cSrc, t.Imp, t.amp = 2 * math.pi, 1.0, 1.0, 1.0
        t.theta, t.phi, t.psi = math.pi / 2, (math.pi if wave == 1 else math.pi / 2), 0.3
        t.tw, t.t0, t.tStop = 0.3, 0.2, 1e30
        t.pos[:] = [v * D / 2 for v in n]
    s = make(cfg)
    s.step(25)
    out = s.fields()
    s.close()
    return out


FOUR = [(0, 9, 10, 8), (1, 9, 10, 9), (2, 9, 10, 10), (2, 9, 10, 11)]


@pytest.mark.parametrize("n,sources,storage,split,wave", [
    ((20, 21, 16), FOUR, abi.STORE_FP32, 0, 0),
    ((20, 21, 19), [(2, 0, 0, 0), (0, 19, 20, 18), (1, 2, 18, 17), (2, 12, 3, 16)], abi.STORE_FP32, 0, 0),
    ((20, 21, 19), FOUR + [(1, 5, 6, 7)], abi.STORE_FP32, 0, 0),
    ((20, 21, 64), [(1, 9, 10, 63)], abi.STORE_FP32, 0, 0),
    ((20, 21, 19), FOUR, abi.STORE_FP32, 1, 0),
    ((20, 21, 19), FOUR, abi.STORE_FP32, 0, 1),
    ((20, 21, 19), FOUR, abi.STORE_FP32, 0, 2),
    ((20, 21, 19), FOUR, abi.STORE_FP16, 0, 0),
])
def test_soft_sources_against_the_oracle(n, sources, storage, split, wave):
    from dtmaxwell4_amd.solver import Solver
    ref = build(Oracle, n, sources, abi.STORE_FP32, split, wave)
    assert max(np.abs(r).max() for r in ref) > 1e-3
    err = rel_l2(build(Solver, n, sources, storage, split, wave), ref)
    print("rel-L2", err)
    assert err <= (1e-5 if storage == abi.STORE_FP32 else 2e-2)

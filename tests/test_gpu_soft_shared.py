"""Soft sources that share a component of a cell add up, whether the E sweep
subtracts them or a launch after it: FP32 with at most and more than four
sources, the split layer, a folded plane wave, FP16, three on one value and two
in one chunk, against the FP64 oracle (1e-5 in relative L2, the bound of the
FP32 path; FP16 2e-2, that of FP16 against FP32).  Alone, each of the sources
that share a value makes a field that is off by more than that.  On a grid that
advances slab by slab one call equals single steps."""
import math

import numpy as np
import pytest

from conftest import rel_l2
from dtmaxwell4_amd import abi, configs
from oracle.oracle import Oracle

D = 0.05
THREE = [(2, 9, 10, 8), (2, 9, 10, 8), (0, 9, 10, 9), (2, 9, 10, 8)]
SIX = [(1, 9, 10, 9), (2, 12, 10, 8), (1, 9, 10, 9), (0, 9, 10, 9), (1, 9, 11, 9), (1, 9, 10, 8)]
# (0, 1 at the layer; 2, 3 in one chunk, each twice; one alone)
SEVEN = [(0, 4, 4, 4), (0, 4, 4, 4), (2, 9, 10, 8), (2, 9, 10, 9), (2, 9, 10, 8), (2, 9, 10, 9), (1, 12, 9, 11)]


def config(n, sources, storage=abi.STORE_FP32, split=0, wave=0):
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
        t.theta, t.phi, t.psi = math.pi / 2, math.pi, 0.3
        t.tw, t.t0, t.tStop = 0.3, 0.2, 1e30
        t.pos[:] = [v * D / 2 for v in n]
    return cfg


def fields(make, cfg, steps=25):
    s = make(cfg)
    s.step(steps)
    out = s.fields()
    s.close()
    return out


@pytest.mark.parametrize("sources", [THREE, SIX, SEVEN])
def test_each_source_counts(sources):
    n = (20, 21, 19)
    ref = fields(Oracle, config(n, sources))
    for q, at in enumerate(sources):
        if sources.count(at) > 1:
            assert rel_l2(fields(Oracle, config(n, sources[:q] + sources[q + 1:])), ref) > 4e-2


@pytest.mark.gpu
@pytest.mark.parametrize("n,sources,storage,split,wave", [
    ((20, 21, 16), THREE, abi.STORE_FP32, 0, 0),
    ((20, 21, 19), THREE, abi.STORE_FP32, 0, 0),
    ((20, 21, 16), SIX, abi.STORE_FP32, 0, 0),
    ((20, 21, 19), SEVEN, abi.STORE_FP32, 0, 0),
    ((20, 21, 19), THREE, abi.STORE_FP32, 1, 0),
    ((20, 21, 19), THREE, abi.STORE_FP32, 0, 1),
    ((20, 21, 19), SEVEN, abi.STORE_FP16, 0, 0),
])
def test_shared_cells_against_the_oracle(n, sources, storage, split, wave):
    from dtmaxwell4_amd.solver import Solver
    ref = fields(Oracle, config(n, sources, abi.STORE_FP32, split, wave))
    err = rel_l2(fields(Solver, config(n, sources, storage, split, wave)), ref)
    print("rel-L2", err)
    assert err <= (1e-5 if storage == abi.STORE_FP32 else 2e-2)


@pytest.mark.gpu
def test_shared_cells_slab_by_slab():
    """More sources than a sweep takes, but not in every slab."""
    from dtmaxwell4_amd.solver import Solver
    n = (240, 208, 212)
    sources = [(2, 20, 100, 101), (2, 20, 100, 101), (1, 70, 104, 100), (0, 120, 99, 98), (2, 170, 100, 99),
               (2, 200, 101, 103)]
    out = []
    for calls in ([1] * 19, [19]):
        s = Solver(config(n, sources))
        for m in calls:
            s.step(m)
        out.append(s.fields())
        s.close()
    assert max(np.abs(x).max() for x in out[0]) > 1e-3
    for x, y in zip(*out):
        assert np.array_equal(x, y)

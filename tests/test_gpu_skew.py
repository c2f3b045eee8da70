"""Grids larger than the Infinity Cache advance several steps slab by slab in
one call; a call of one step takes that step over the whole grid.  Both give
the same fields, probes and DFT bins bit for bit: FP32 and FP16, a folded plane
wave that ends in the middle, soft sources and the split-field layer, probes and
sensors on slab bounds, numbers of steps that leave a short last group, a series
that fills up, grids just above the size from which it applies and of no round
number."""
import math

import numpy as np
import pytest

from dtmaxwell4_amd import abi, configs

pytestmark = pytest.mark.gpu

D = 0.05


def build(n, storage, split, wave, soft, probes, calls):
    from dtmaxwell4_amd.solver import Solver
    nx, ny, nz = n
    cfg = abi.default_config(*n, D, D, D, configs.dt_for(D, D, D))
    cfg.storage = storage
    cfg.npml[:] = [7, 6, 5, 8, 9, 4]
    cfg.pml_kind = abi.PML_SPLIT if split else abi.PML_CPML
    if wave:
        t = cfg.tfsf
        t.kind, t.waveform, t.sf_inside = abi.TFSF_PLANE, abi.WAVE_GAUSS_SINE, 0
        t.box[:] = [12 * D, (nx - 12) * D, 12 * D, (ny - 12) * D, 12 * D, (nz - 12) * D]
        t.w, t.cSrc, t.Imp, t.amp = 2 * math.pi, 1.0, 1.0, 1.0
        t.theta, t.phi, t.psi = math.pi / 2, math.pi, 0.3
        t.tw, t.t0, t.tStop = 0.3, 0.2, 30.5 * cfg.dt
        t.pos[:] = [(nx - 12) * D, 0.0, 0.0]
    cfg.nsoft = soft
    for q in range(soft):
        so = cfg.soft[q]
        so.comp, so.i, so.j, so.k = q % 3, (nx // 2 + 11 * q) % nx, ny // 2, nz // 2 + q
        so.waveform, so.amp, so.w, so.tw, so.t0 = abi.WAVE_GAUSS_SINE, 5.0, 2 * math.pi, 0.3, 0.2
    s = Solver(cfg)
    for c in range(6):
        for i in range(nx - 1, 0, -probes):
            s.add_probe(c, i, ny // 2 + 1, nz // 2 + 2)
            s.add_sensor(("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")[c], i, ny // 2, nz // 2)
    s.set_dft(np.array([3.0, 6.0]))
    for m in calls:
        s.step(m)
    out = s.fields() + [s.probes().copy(), s.dft().copy()]
    s.close()
    return out


@pytest.mark.parametrize("n,storage,split,wave,soft,probes", [
    ((163, 251, 255), abi.STORE_FP32, 0, 1, 0, 1),
    ((211, 208, 212), abi.STORE_FP32, 0, 0, 3, 7),
    ((150, 210, 211), abi.STORE_FP32, 1, 1, 1, 5),
    ((256, 256, 256), abi.STORE_FP16, 0, 1, 5, 3),
    ((301, 241, 237), abi.STORE_FP16, 0, 0, 1, 11),
])
def test_one_call_equals_single_steps(n, storage, split, wave, soft, probes):
    a = build(n, storage, split, wave, soft, probes, [1] * 43)
    b = build(n, storage, split, wave, soft, probes, [43])
    assert max(np.abs(x).max() for x in a[:6]) > 1e-4
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("every,inside", [(0, False), (13, False), (13, True)])
def test_adjoint_slab_by_slab_equals_whole_steps(every, inside):
    """Both passes of the adjoint on a large grid; with event timing on, every
    step runs over the whole grid.  Monitors beside and inside the design box,
    with the history kept and rebuilt from checkpoints."""
    from dtmaxwell4_amd.solver import Solver
    n = (300, 190, 207)
    out = []
    for timing in (False, True):
        cfg = abi.default_config(*n, D, D, D, configs.dt_for(D, D, D))
        cfg.npml[:] = [8] * 6
        cfg.nsoft = 1
        so = cfg.soft[0]
        so.comp, so.i, so.j, so.k = abi.EZ, 130, 95, 103
        so.waveform, so.amp, so.w, so.tw, so.t0 = abi.WAVE_GAUSS_SINE, 5.0, 2 * math.pi, 0.3, 0.2
        s = Solver(cfg)
        s.set_design_eps(144, 90, 98, 1 + 2 * np.random.default_rng(2).random((25, 11, 10)))
        if every:
            s.set_adjoint_checkpoints(every)
        s.set_kernel_timing(timing)
        mon = [(150, 95, 100), (160, 92, 103)] if inside else [(175, 95, 100), (138, 93, 103), (180, 96, 105)]
        out.append(s.design_gradient(47, 6.0, mon))
        s.close()
    assert out[0][0] > 0 and np.abs(out[0][1]).max() > 0
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])

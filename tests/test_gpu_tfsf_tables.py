"""The tabulated TF/SF corrections against the FP64 oracle: a dipole whose box
is the smallest allowed, ragged, next to a grid face, inside the layer, or just
small or too large for the point tables, and plane waves along y and z.  Steps
are taken one by one and several at once: a call fills the tables of its own
half-steps only.  FP32 storage, 1e-5 in relative L2 (the bound of the FP32
path)."""
import math

import numpy as np
import pytest

from conftest import rel_l2
from dtmaxwell4_amd import abi, configs
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

D = 0.05
N = (40, 44, 47)


def build(make, kind, box, axis, split):
    cfg = abi.default_config(*N, D, D, D, configs.dt_for(D, D, D))
    cfg.npml[:] = [6] * 6
    cfg.pml_kind = abi.PML_SPLIT if split else abi.PML_CPML
    t = cfg.tfsf
    t.kind, t.waveform = kind, abi.WAVE_GAUSS_SINE
    t.sf_inside = int(kind == abi.TFSF_DIPOLE)
    t.box[:] = [v * D for p in box for v in p]
    t.w, t.cSrc, t.Imp, t.amp = 2 * math.pi, 1.0, 1.0, 1.0
    t.theta, t.phi, t.psi = (math.pi / 2, math.pi / 2, 0.4) if axis == 1 else (0.0, 0.0, 0.4)
    t.tw, t.t0, t.tStop = 0.3, 0.2, 1e30
    t.pos[:] = [0.5 * (p[0] + p[1]) * D for p in box]
    s = make(cfg)
    for n in (1, 1, 20, 1, 7):
        s.step(n)
    out = s.fields()
    s.close()
    return out


@pytest.mark.parametrize("kind,box,axis,split", [
    (abi.TFSF_DIPOLE, [(18.0, 22.0), (20.0, 24.0), (21.0, 25.0)], 0, 0),
    (abi.TFSF_DIPOLE, [(17.2, 22.3), (19.1, 26.4), (14.3, 27.7)], 0, 1),
    (abi.TFSF_DIPOLE, [(2.1, 12.2), (1.3, 10.4), (33.3, 45.6)], 0, 0),
    (abi.TFSF_DIPOLE, [(2.1, 12.2), (1.3, 10.4), (33.3, 45.6)], 0, 1),
    (abi.TFSF_DIPOLE, [(8.2, 32.1), (10.3, 34.4), (11.2, 35.3)], 0, 0),
    (abi.TFSF_DIPOLE, [(7.2, 33.1), (9.3, 35.4), (10.2, 37.3)], 0, 0),
    (abi.TFSF_PLANE, [(9.3, 30.2), (8.1, 33.3), (9.2, 37.4)], 1, 0),
    (abi.TFSF_PLANE, [(3.3, 36.2), (2.1, 40.3), (4.2, 43.4)], 2, 1),
])
def test_tables_against_the_oracle(kind, box, axis, split):
    from dtmaxwell4_amd.solver import Solver
    ref = build(Oracle, kind, box, axis, split)
    assert max(np.abs(r).max() for r in ref) > 1e-3
    err = rel_l2(build(Solver, kind, box, axis, split), ref)
    print("rel-L2", err)
    assert err <= 1e-5

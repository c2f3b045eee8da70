"""The update of dispersive, conductive and gyrotropic cells, against the FP64
oracle from random fields: every number of poles its variants hold (none with
a conductivity, one, two, more, and a mix), more than 32 classes, a box that
is no multiple of a block or a wave, cells of other classes in between.  FP32,
60 steps, 1e-5 in relative L2 (the bound of the FP32 path)."""
import numpy as np
import pytest

from conftest import rel_l2
from dtmaxwell4_amd import abi, configs
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

D = 0.05


def material(m, kind):
    m.eps_inf = 2.0
    if kind == "sigma":
        m.sigma = 1.5
    elif kind == "gyro":
        m.gyro, m.gyro_wp, m.gyro_nu = 1, 3.0, 0.4
        m.gyro_wc[:] = [0.6, -0.9, 1.7]
    elif kind != "plain":
        m.npoles = int(kind)
        for p in range(m.npoles):
            if p == 0:
                m.pole[p].setDrude(Deps=1.0, wp=4.0, gp=0.3)
            else:
                m.pole[p].set(Deps=0.7 / p, wp=5.0 + 2 * p, gp=0.2 * p)


def build(make, kinds, mixed):
    n = (15, 14, 37)
    cfg = abi.default_config(*n, D, D, D, configs.dt_for(D, D, D))
    cfg.nmat = len(kinds)
    for q, kind in enumerate(kinds):
        material(cfg.mat[q], kind)
    rng = np.random.default_rng(5)
    ids = [rng.integers(0, len(kinds), n).astype(np.uint8) for _ in range(3)]
    for m in ids:  # the box of special cells is inside the grid
        m[:2], m[:, :1], m[:, :, :3], m[:, :, -2:] = 0, 0, 0, 0
    s = make(cfg)
    s.set_materials(*(ids if mixed else [ids[0]] * 3))
    for c in range(6):
        s.set_field(c, rng.standard_normal(n).astype(np.float32))
    s.step(60)
    out = s.fields()
    s.close()
    return out


@pytest.mark.parametrize("kinds,mixed", [
    (("plain", "sigma"), True), (("plain", "1"), True), (("plain", "2"), False), (("plain", "3"), True),
    (("plain", "4", "sigma", "1"), True), (("plain", "gyro"), False), (("plain", "gyro", "2", "sigma"), False),
    (("plain", "gyro", "4"), False),
])
def test_special_cells_against_the_oracle(kinds, mixed):
    from dtmaxwell4_amd.solver import Solver
    ref = build(Oracle, kinds, mixed)
    assert all(np.isfinite(r).all() for r in ref) and max(np.abs(r).max() for r in ref) < 100
    err = rel_l2(build(Solver, kinds, mixed), ref)
    print(kinds, "rel-L2", err)
    assert err <= 1e-5

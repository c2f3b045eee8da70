"""Conductive, dispersive and gyrotropic cells along a whole grid of 2^24 + 100
planes of one cell: with a block per plane the correction of its cells was a
launch of more than 2^32 lanes, of which the device ran the first 100 blocks and
reported nothing.  Fields that start the same in every plane stay so away from the
ends: equal, bit for bit, to those of the middle of a short grid."""
import numpy as np
import pytest

from dtmaxwell4_amd import abi, configs

pytestmark = pytest.mark.gpu

D, STEPS = 0.05, 4


def middle(nx, storage, poles, gyro):
    """Fields away from the ends."""
    from dtmaxwell4_amd.solver import Solver
    cfg = abi.default_config(nx, 1, 1, D, D, D, configs.dt_for(D, D, D))
    cfg.storage = storage
    m = cfg.mat[0]
    m.eps_inf, m.npoles, m.gyro = 2.0, poles, gyro
    if poles:
        m.pole[0].setDrude(1.0, 9.0, 1.5, 0.0)
        m.pole[1].set(0.5, 9.0, 0.9, 0.0)
    else:
        m.sigma = 3.0
    if gyro:
        m.gyro_wp, m.gyro_nu = 8.0, 0.1
        m.gyro_wc[:] = [0.3, 0.1, 1.6]
    s = Solver(cfg)
    for c in range(6):
        s.set_field(c, np.full((nx, 1, 1), 0.5 + 0.25 * c, np.float32))
    s.step(STEPS)
    out = [f[4 * STEPS:-4 * STEPS] for f in s.fields()]
    s.close()
    return out


@pytest.mark.parametrize("storage,poles,gyro", [(abi.STORE_FP32, 0, 0), (abi.STORE_FP16, 0, 0),
                                                (abi.STORE_FP32, 2, 0), (abi.STORE_FP32, 0, 1)])
def test_box_of_more_than_2_24_planes(storage, poles, gyro):
    short = middle(100, storage, poles, gyro)
    long = middle((1 << 24) + 100, storage, poles, gyro)
    for a, b in zip(short, long):
        assert np.abs(a).max() > 1e-3
        assert (a == a[0]).all() and (b == a[0]).all()

"""Probes that ride with the sweeps: a call of many steps records each step's E
probes with the next H sweep and its H probes with its E sweep, a call of one
step with a launch of its own.  Series, last values and DFT bins of both are
the same bit for bit, for cells and sensors of every component on and beside
the boundaries, in FP32, FP16, FP16 with an FP32 zone over part or all of the
grid, and where the series is emptied in the middle of a call."""
import numpy as np
import pytest

from dtmaxwell4_amd import abi, configs

pytestmark = pytest.mark.gpu

D = 0.05


def build(storage, zone, periodic, many, calls):
    from dtmaxwell4_amd.solver import Solver
    n = (9, 10, 11)
    cfg = abi.default_config(*n, D, D, D, configs.dt_for(D, D, D))
    cfg.storage = storage
    if periodic:
        cfg.bc[:] = [abi.BC_PERIODIC] * 3
    s = Solver(cfg)
    if zone:
        s.set_fp32_zone(*zone)
    rng = np.random.default_rng(8)
    for c in range(6):
        s.set_field(c, (0.1 * rng.standard_normal(n)).astype(np.float32))
    for c in range(6):
        for at in ((0, 0, 0), (8, 9, 10), (4, 5, 6)):
            s.add_probe(c, *at)
    for name in ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz"):
        for at in ((0, 0, 0), (8, 9, 10), (5, 1, 0)):
            s.add_sensor(name, *at)
    for q in range(many):
        s.add_probe(q % 6, q % 9, q % 10, q % 11)
    s.set_dft(np.array([1.0, 2.5, 7.0]))
    last = []
    for m in calls:
        s.step(m)
        last.append(s.probe_last().copy())
    out = s.probes().copy(), s.dft().copy(), last[-1]
    s.close()
    return out


@pytest.mark.parametrize("storage,zone,periodic,many,steps", [
    (abi.STORE_FP32, None, False, 0, 21), (abi.STORE_FP32, None, True, 0, 21), (abi.STORE_FP16, None, False, 0, 21),
    (abi.STORE_FP16, (2, 6, 3, 7, 1, 8), False, 0, 21), (abi.STORE_FP16, (0, 9, 0, 10, 0, 11), True, 0, 21),
    (abi.STORE_FP32, None, False, 4000, 1100),  # 1038 rows of the series at a time
])
def test_one_call_records_what_single_steps_record(storage, zone, periodic, many, steps):
    a = build(storage, zone, periodic, many, [1] * steps)
    b = build(storage, zone, periodic, many, [steps])
    assert a[0].shape == b[0].shape and np.abs(a[0]).max() > 0 and np.abs(a[1]).max() > 0
    for x, y in zip(a, b):
        assert np.array_equal(x, y)

"""The half-step sweeps where a lane's chunk of four z cells, a wave of 64
chunks, a slab or the addressing of a plane can go wrong.

- Against the FP64 oracle, from random fields, per z plane: z extents below a
  chunk, around it, and around a wave's 256 cells, ragged rows, layers that end
  inside a chunk or leave one or two cells between them, a periodic z axis,
  materials, the folded plane wave.  After 12 steps FP32 is held to 1e-5 (the
  bound of the FP32 path); FP16 to 24 roundings of 2^-11, 1.2e-2: one of each
  component in each of 24 half-steps.  A neighbour or weight that is missed in
  one plane is an error of order one there.
- Planes of 4 GiB and more, and a field set of 4 GiB with the FP32 zone, which
  are addressed in other ways: near the far corner of the grid the fields of a
  source next to it are those of a small grid with the same corner, to 1e-6 of
  the peak."""
import math

import numpy as np
import pytest

from dtmaxwell4_amd import abi, configs
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

D = 0.05
CASES = [  # nz, z layer (low, high), periodic z
    (1, (0, 0), False), (2, (0, 0), False), (3, (0, 0), False), (4, (0, 0), True), (5, (2, 2), False),
    (9, (5, 3), False), (13, (6, 5), False), (16, (8, 8), False), (23, (0, 0), True), (31, (3, 9), False),
    (64, (10, 10), False), (66, (6, 7), False), (128, (0, 0), True), (255, (10, 9), False), (256, (10, 10), False),
    (257, (4, 4), False), (258, (0, 0), True),
]


def build(make, nz, npml, perz, storage, split, wave):
    nx, ny = 19, 22
    cfg = abi.default_config(nx, ny, nz, D, D, D, configs.dt_for(D, D, D))
    cfg.storage = storage
    cfg.npml[:] = [4, 5, 3, 6, *npml]
    if perz:
        cfg.bc[2] = abi.BC_PERIODIC
    cfg.pml_kind = abi.PML_SPLIT if split else abi.PML_CPML
    cfg.nmat = 2
    cfg.mat[0].eps_inf, cfg.mat[1].eps_inf = 1.5, 3.0
    if wave:
        t = cfg.tfsf
        t.kind, t.waveform, t.sf_inside = abi.TFSF_PLANE, abi.WAVE_GAUSS_SINE, 0
        t.box[:] = [6.3 * D, 13.2 * D, 6.1 * D, 13.4 * D, 0.23 * nz * D, 0.71 * nz * D]
        t.w, t.cSrc, t.Imp, t.amp = 2 * math.pi, 1.0, 1.0, 2.0
        t.theta, t.phi, t.psi = math.pi / 2, math.pi, -math.pi / 3
        t.tw, t.t0, t.tStop = 1.0, 0.2, 1e30
    s = make(cfg)
    rng = np.random.default_rng(100 * nz + split)
    s.set_materials(*[(rng.random((nx, ny, nz)) < 0.3).astype(np.uint8) for _ in range(3)])
    for c in range(6):
        f = np.clip(rng.standard_normal((nx, ny, nz)), -4, 4)
        s.set_field(c, f.astype(np.float16).astype(np.float32))
    s.step(12)
    out = s.fields()
    s.close()
    return out


@pytest.mark.parametrize("nz,npml,perz", CASES)
def test_edges_against_the_oracle(nz, npml, perz):
    from dtmaxwell4_amd.solver import Solver
    for split in (0, 1):
        wave = not perz
        ref = build(Oracle, nz, npml, perz, abi.STORE_FP32, split, wave)
        norm = math.sqrt(sum(float(np.sum(np.square(r))) for r in ref) / nz)
        for storage, tol in ((abi.STORE_FP32, 1e-5), (abi.STORE_FP16, 24 * 2.0 ** -11)):
            got = build(Solver, nz, npml, perz, storage, split, wave)
            err = sum(np.sum(np.square(g.astype(np.float64) - r), axis=(0, 1)) for g, r in zip(got, ref))
            worst = math.sqrt(err.max()) / norm
            print(f"nz {nz} split {split} storage {storage}: worst z plane {worst:.2e} (k = {int(err.argmax())})")
            assert worst <= tol


def corner(shape, storage, split, zone):
    from dtmaxwell4_amd.solver import Solver
    nx, ny, nz = shape
    cfg = abi.default_config(nx, ny, nz, D, D, D, configs.dt_for(D, D, D))
    cfg.storage = storage
    cfg.npml[:] = [0, 0, 0, 5, 0, 6]
    cfg.pml_kind = abi.PML_SPLIT if split else abi.PML_CPML
    cfg.nsoft = 1
    so = cfg.soft[0]
    so.comp, so.i, so.j, so.k = abi.EX, nx - 1, ny - 9, nz - 10
    so.waveform, so.amp, so.w, so.tw, so.t0 = abi.WAVE_GAUSS_SINE, 100.0, 20.0, 0.05, 0.02
    s = Solver(cfg)
    if zone:
        s.set_fp32_zone(0, nx, ny - 12, ny - 7, nz - 13, nz - 8)
    for c in range(6):
        for dj, dk in ((9, 10), (8, 11), (10, 9), (5, 6), (3, 4), (1, 1), (2, 12), (13, 3)):
            s.add_probe(c, nx - 1, ny - dj, nz - dk)
    s.step(6)  # 18 cells of reach
    p = s.probes()
    s.close()
    return p


@pytest.mark.parametrize("shape,storage,split,zone", [
    ((1, 32771, 32770), abi.STORE_FP32, 0, 0),
    ((1, 32771, 32770), abi.STORE_FP16, 0, 0),
    ((1, 32771, 32770), abi.STORE_FP32, 1, 0),
    ((1, 32771, 32770), abi.STORE_FP16, 0, 1),
    ((8, 8192, 5610), abi.STORE_FP16, 0, 1),
    ((8, 8192, 5610), abi.STORE_FP16, 1, 0),
    ((4, 8192, 5610), abi.STORE_FP32, 1, 0),
])
def test_large_planes_equal_a_small_grid(shape, storage, split, zone):
    big = corner(shape, storage, split, zone)
    small = corner((shape[0], 43, 46 - (46 - shape[2]) % 4), storage, split, zone)
    peak = np.abs(small).max()
    d = np.abs(big - small).max() / peak
    print("peak", peak, "max |big - small| / peak", d)
    assert peak > 1e-3
    assert d <= 1e-6

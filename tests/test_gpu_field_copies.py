"""Fields to and from the host in chunks: meshes whose field is one chunk, whole
rows of elements per chunk, and pieces of rows, with node and element counts
that end inside the 32 x 64 tiles. What is set comes back: exactly in FP64,
rounded once in FP32; the density sensitivity equals the numpy sum."""
import numpy as np
import pytest

from helpers import random_unique, small_grid, unique_to_local
from ses3d_amd import api

pytestmark = pytest.mark.gpu

# order, elements: chunks of 1 MB to 4 MB hold 131072 to 524288 values (a third
# of each of three fields): one chunk; rows of 64 nodes; pieces of rows of 27
# and of 64 nodes
MESHES = [(7, (3, 2, 2)), (3, (9, 5, 3)), (4, (17, 16, 16)), (2, (33, 32, 20)), (5, (23, 20, 19))]


def _sim(p, shape, **kw):
    nx, ny, nz = shape
    grid = small_grid(nx=nx, ny=ny, nz=nz, lpd=p)
    s = api.Simulation(grid, **kw)
    one = np.ones(s.shape)
    for par, x in ((api.RHOINV, 1 / 3000.0), (api.LAMBDA, 6e10), (api.MU, 5e10), (api.Q, 300.0)):
        s.set_model(par, x * one)
    s.init()
    return s, grid


@pytest.mark.parametrize("p,shape", MESHES)
def test_fp64_fields_come_back(p, shape):
    s, grid = _sim(p, shape, precision="fp64")
    rng = np.random.default_rng(p)
    for f in (api.VX, api.VZ):
        v = unique_to_local(random_unique(grid, rng), grid)
        s.set(f, v)
        assert np.array_equal(s.get(f), v), f
    for f in (api.SXY, api.SZZ, api.MXX, api.MXX + 17):
        x = rng.standard_normal(s.shape)
        s.set(f, x)
        assert np.array_equal(s.get(f), x), f
    assert not np.any(s.get(api.SXX))


@pytest.mark.parametrize("p,shape", MESHES)
@pytest.mark.parametrize("ks", [0, 1, 2])
def test_fp32_fields_come_back_rounded(p, shape, ks):
    s, grid = _sim(p, shape, precision="fp32", kahan_v=2 if ks == 2 else 1, kahan_sigma=ks,
                   memory_vars=5 if ks else 6)
    rng = np.random.default_rng(10 * p + ks)
    v = unique_to_local(random_unique(grid, rng), grid)
    s.set(api.VY, v)
    # 24 + 24 bits, or 24 + 8 bits with BF16 words
    assert np.all(np.abs(s.get(api.VY) - v) <= np.abs(v) * 2.0 ** (-33 if ks == 2 else -48))
    x = rng.standard_normal(s.shape)
    for f in (api.SXX, api.SXY, api.SYZ, api.MXX + 6, api.MXX + 9):
        s.set(f, x)
        assert np.array_equal(s.get(f), x.astype(np.float32).astype(np.float64)), f
    if ks:
        # zz of a deviatoric memory variable, from the two just set
        assert np.array_equal(s.get(api.MXX + 11), -2.0 * x.astype(np.float32).astype(np.float64))


@pytest.mark.parametrize("p,shape", MESHES)
def test_density_sensitivity_sum(p, shape):
    s, grid = _sim(p, shape, precision="fp64")
    rng = np.random.default_rng(p + 50)
    v = [unique_to_local(random_unique(grid, rng), grid) for _ in range(3)]
    for f, a in zip((api.VX, api.VY, api.VZ), v):
        s.set(f, a)
    fw = [rng.standard_normal(s.shape) for _ in range(3)]
    s.grad_add(*fw, -2)
    s.grad_add(*fw, 1)
    d = [np.radians(grid.lat_max - grid.lat_min) / grid.nx, np.radians(grid.lon_max - grid.lon_min) / grid.ny,
         (grid.rad_max - grid.rad_min) / grid.nz]
    want = -grid.dt * sum(a * b for a, b in zip(fw, v)) / (d[0] * d[1] * d[2] / 8.0)
    got = s.get(api.GRAD_RHO)
    # a dozen roundings of terms up to |f . v|
    scale = 2 * grid.dt * sum(np.abs(a * b) for a, b in zip(fw, v)) / (d[0] * d[1] * d[2] / 8.0)
    assert np.all(np.abs(got - want) <= 16 * 2.0 ** -53 * 2 * scale)

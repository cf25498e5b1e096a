"""Edge cases of the mesh and of the run against the FP64 oracle: a single
element, meshes one element thick along one or two axes (every node on a
domain face), tiles that overhang the last element, the plane-pair tile
order with an odd number of planes, and a run with neither sources nor
receivers."""
import numpy as np
import pytest

import oracle
from helpers import random_model, random_unique, rel_l2, small_grid, unique_to_local
from ses3d_amd import api
from test_gpu_parity import FIELDS, PARAMS, _pair, _random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 1, 1), (1, 3, 2), (3, 2, 1), (5, 1, 3)])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("fp32", 1e-5)])
def test_tiny_and_thin_meshes_match_oracle(shape, precision, tol):
    nx, ny, nz = shape
    grid = small_grid(nx=nx, ny=ny, nz=nz, lpd=4, taper_width=0)
    rng = np.random.default_rng(40 + nx + 3 * ny + 7 * nz)
    o, s = _pair(grid, random_model(grid, rng, visco=True), precision=precision)
    _random_state(o, s, grid, rng, visco=True)
    o.step(5)
    s.step(5)
    for f in FIELDS:
        assert rel_l2(s.get(f), o.get(f)) < tol, (shape, f)


@pytest.mark.parametrize("tile", [1, 2, 4])
def test_tiles_overhanging_the_last_element(tile):
    """7 x 3 x 1 elements: 21 elements, so tiles of 2 and 4 leave idle slots
    in the last workgroup; the results equal the oracle's."""
    grid = small_grid(nx=7, ny=3, nz=1, lpd=4, taper_width=0)
    rng = np.random.default_rng(77)
    o, s = _pair(grid, random_model(grid, rng, visco=True), precision="fp32")
    s.set_tile(tile)
    _random_state(o, s, grid, rng, visco=True)
    o.step(4)
    s.step(4)
    for f in FIELDS:
        assert rel_l2(s.get(f), o.get(f)) < 1e-5, (tile, f)


@pytest.mark.parametrize("tile", [1, 2, 4])
@pytest.mark.parametrize("nz", [3, 4])
def test_plane_pair_order_matches_oracle(tile, nz):
    """4 x 4 planes hold whole tiles of 1, 2 and 4 elements, so the element
    kernel runs the tiles of planes 2m and 2m+1 alternately; with 3 planes
    the last one runs alone. Every element is still advanced once: the
    fields equal the oracle's, FP64 and FP32."""
    grid = small_grid(nx=4, ny=4, nz=nz, lpd=4, taper_width=0)
    for precision, tol in (("fp64", 1e-11), ("fp32", 1e-5)):
        rng = np.random.default_rng(90 + nz)
        o, s = _pair(grid, random_model(grid, rng, visco=True), precision=precision)
        s.set_tile(tile)
        _random_state(o, s, grid, rng, visco=True)
        o.step(4)
        s.step(4)
        for f in FIELDS:
            assert rel_l2(s.get(f), o.get(f)) < tol, (precision, tile, f)
        s.close()


@pytest.mark.parametrize("shape", [(8, 16, 16), (13, 15, 11), (17, 11, 11), (16, 16, 9), (13, 14, 13)])
def test_workgroup_orders_match_oracle(shape):
    """One element per workgroup, so the shapes are 2048 and 2145 workgroups
    (8 x 256, and just past the resident limit), 2057 (a multiple of neither
    8 nor 128), 2304 (whole groups of 8 chunks) and 2366 (a tail): every
    element is advanced once in the XCD-aware order, as the oracle has it, and
    bit for bit as in the plain order."""
    nx, ny, nz = shape
    grid = small_grid(nx=nx, ny=ny, nz=nz, lpd=2)
    rng = np.random.default_rng(17)
    model = random_model(grid, rng)
    o, s = _pair(grid, model, precision="fp32")
    plain = api.Simulation(grid, "fp32", xcd_remap=False)
    for k, arr in model.items():
        plain.set_model(PARAMS[k][1], arr)
    plain.init()
    _random_state(o, s, grid, rng)
    for f in FIELDS:
        plain.set(f, o.get(f))
    for x in (s, plain):
        x.set_tile(1)
        x.step(3)
    o.step(3)
    for f in FIELDS:
        assert rel_l2(s.get(f), o.get(f)) < 1e-5, (shape, f)
        assert np.array_equal(s.get(f), plain.get(f)), (shape, f)


@pytest.mark.parametrize("lpd,tile", [(2, 0), (2, 1), (3, 1), (4, 0), (4, 1), (5, 1), (6, 0), (7, 0)])
@pytest.mark.parametrize("ks,words", [(0, 0), (1, 0), (2, 0), (0, 5), (1, 5), (2, 5), (0, 6), (1, 6)])
def test_tile_loads_at_every_alignment(lpd, tile, ks, words):
    """The FP32 element kernel loads a tile's contiguous words in 16-byte
    vectors, whatever word the tile starts at: tiles of 1 to 9 elements of 27
    to 512 nodes and 6 to 30 words per node start at every place modulo 4, and
    the last of 7 elements ends inside a tile of 2, 4 or 9. One state block
    for odd, two for even compensation modes."""
    grid = small_grid(nx=7, ny=1, nz=1, lpd=lpd, taper_width=0)
    rng = np.random.default_rng(10 * lpd + ks)
    model = random_model(grid, rng, visco=words > 0)
    o = oracle.Oracle(grid)
    s = api.Simulation(grid, "fp32", kahan_sigma=ks, memory_vars=words, state_buffers=1 if ks == 1 else 2)
    for k, arr in model.items():
        o.set_model(PARAMS[k][0], arr)
        s.set_model(PARAMS[k][1], arr)
    o.init()
    s.init()
    s.set_tile(tile)
    for f in (api.VX, api.VY, api.VZ):
        v = unique_to_local(random_unique(grid, rng, 1e-3), grid)
        o.set(f, v)
        s.set(f, v)
    shp = o.shape
    for f in range(api.SXX, api.SZZ + 1):
        x = 1e5 * rng.standard_normal(shp)
        o.set(f, x)
        s.set(f, x)
    for m in range(3 if words else 0):
        x = [1e-9 * rng.standard_normal(shp) for _ in range(6)]
        x[5] = -(x[0] + x[3])               # deviatoric: both forms hold it
        for c in range(6):
            o.set(api.MXX + 6 * m + c, x[c])
            if words == 6 or c < 5:
                s.set(api.MXX + 6 * m + c, x[c])
    o.step(3)
    s.step(3)
    for f in FIELDS:
        assert rel_l2(s.get(f), o.get(f)) < 1e-5, f


@pytest.mark.parametrize("lpd,precision,kahan_v,shape", [
    (2, "fp32", False, (127, 1, 127)), (2, "fp32", True, (31, 31, 31)), (2, "fp32", "bf16", (1, 127, 127)),
    (2, "fp64", False, (127, 127, 1)), (2, "fp32", True, (126, 127, 1)), (3, "fp32", False, (85, 1, 85)),
    (3, "fp64", False, (29, 28, 27)), (3, "fp32", True, (28, 27, 26)), (4, "fp64", False, (63, 63, 1)),
    (4, "fp32", False, (1, 62, 63)), (5, "fp32", False, (16, 17, 17))])
def test_assembly_by_rows_and_by_nodes(lpd, precision, kahan_v, shape):
    """The assembly takes one lane per row of nodes from 131072 rows on (order
    2, uncompensated up to order 5) and one per node elsewhere: the oracle's
    results at that line, at the last mesh before it, past it and, by nodes,
    in chunks of workgroups with a tail; on meshes one element thick along
    each axis; and the same values from a member of a batch."""
    nx, ny, nz = shape
    grid = small_grid(nx=nx, ny=ny, nz=nz, lpd=lpd, taper_width=0 if 1 in shape else 1, dt=0.02)
    rng = np.random.default_rng(300 + 10 * lpd + nx)
    model = random_model(grid, rng)
    o, s = _pair(grid, model, precision=precision, kahan_v=kahan_v)
    member = api.Simulation(grid, precision, kahan_v=kahan_v)
    other = small_grid(nx=3, ny=2, nz=2, lpd=lpd)
    small = api.Simulation(other, precision, kahan_v=kahan_v)
    for x, m in ((member, model), (small, random_model(other, rng))):
        for k, arr in m.items():
            x.set_model(PARAMS[k][1], arr)
        x.init()
    _random_state(o, s, grid, rng)
    for f in FIELDS:
        member.set(f, o.get(f))
    o.step(2)
    s.step(2)
    b = api.Batch([small, member])
    b.step(2)
    b.synchronize()
    for f in FIELDS:
        got = s.get(f)
        assert rel_l2(got, o.get(f)) < (1e-11 if precision == "fp64" else 1e-5), f
        assert np.array_equal(member.get(f), got), f
    b.close()


def test_run_without_sources_or_receivers():
    grid = small_grid(nx=3, ny=2, nz=2, nt=20)
    rng = np.random.default_rng(5)
    o, s = _pair(grid, random_model(grid, rng), precision="fp32")
    s.step(20)   # one graph chunk and four direct steps
    assert np.array_equal(s.vrange(), [0.0, 0.0])
    assert s.it == 20
    for f in FIELDS:
        assert not np.any(s.get(f)), f
    with pytest.raises(api.S3dError):
        s.trace(0, 0)
    with pytest.raises(api.S3dError, match="past nt"):
        s.step(1)

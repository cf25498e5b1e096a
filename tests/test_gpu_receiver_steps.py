"""Receivers of a step recorded by the next step's element kernel: the traces
of one call of many steps (captured chunks and direct steps) equal, bit for
bit, those of single steps, whose receivers are recorded by their own launch,
and the oracle's. With one and two state blocks, velocity channels only or
also pressure, source echo and curl channels, and receiver counts that do and
do not fill the recording workgroups."""
import numpy as np
import pytest

from helpers import random_model, rel_l2, small_grid
from ses3d_amd import api
from test_gpu_parity import PARAMS, _pair, _random_state

pytestmark = pytest.mark.gpu

V = ("vx", "vy", "vz")
SETS = [V, V + ("pressure",), ("n", "mxy", "fz", "pressure"), V + ("rot_vz",)]


def _stations(x, grid, nrec, channels):
    rng = np.random.default_rng(3)
    e, vm = x.locate(0.6, 14.1, 60e3)
    stf = 1e13 * rng.standard_normal((6, grid.nt))
    x.add_source_mt(e, vm, stf)
    x.add_source_sf(e, vm, 1e8 * rng.standard_normal((3, grid.nt)))
    x.add_receiver(e, vm, channels)
    for _ in range(nrec - 1):
        e, vm = x.locate(rng.uniform(-2, 3), rng.uniform(11, 17), 0.0)
        x.add_receiver(e, vm, channels)


@pytest.mark.parametrize("channels", SETS)
@pytest.mark.parametrize("lpd,buffers,nrec", [(4, 2, 1), (4, 1, 9), (2, 2, 33), (6, 1, 4), (7, 2, 17)])
def test_many_steps_record_as_single_steps(lpd, buffers, nrec, channels):
    grid = small_grid(lpd=lpd, nt=40)
    rng = np.random.default_rng(lpd + nrec)
    model = random_model(grid, rng)
    o, s = _pair(grid, model)
    runs = [s]
    for _ in range(2):
        x = api.Simulation(grid, "fp32", state_buffers=buffers)
        for k, arr in model.items():
            x.set_model(PARAMS[k][1], arr)
        x.init()
        runs.append(x)
    _random_state(o, s, grid, rng)
    for x in runs[1:]:
        for f in range(api.VX, api.SZZ + 1):
            x.set(f, o.get(f))
    for x in runs + ([o] if "rot_vz" not in channels else []):
        _stations(x, grid, nrec, channels)
    n = 37                                  # two chunks of 16 and 5 steps
    s.step(n)
    runs[1].step(n)
    for _ in range(n):
        runs[2].step(1)
    if "rot_vz" not in channels:
        o.step(n)
    for r in range(nrec):
        for c in range(len(channels)):
            a, b = runs[1].trace(r, c), runs[2].trace(r, c)
            assert np.array_equal(a, b), (r, c)
            assert not np.any(a[n:])
            if "rot_vz" not in channels:
                t = o.trace(r, c)
                assert rel_l2(s.trace(r, c), t) < 1e-10, (r, c)

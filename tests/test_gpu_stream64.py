"""The FP64 population kernel that advances two steps per launch, against the
oracle bit for bit (populations, fields, halo): column segments of 60 with the
remainder at their edges, strips of one row to more than the lattice has, both
rounding policies, the extensions, odd and even numbers of steps per call, and
the calls that leave the path (uploaded ghost velocities, single subroutines in
between).  BGK_POP_VARIANT=2 takes lattices below the size the rule would.
"""
import numpy as np
import pytest

from bgk_pcm_amd.lattice import Lattice
from bgk_pcm_amd.params import Params
from golden_io import compare_state
from oracle_py import Oracle
from test_gpu_parity import POPS, STATE, compare_interior, gpu_state

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (1, 9), (9, 1), (2, 2), (59, 3), (60, 7), (61, 4), (62, 5), (63, 33), (121, 6),
          (124, 40), (185, 21)]
EXT = dict(k_ratio=1.5, t_cold=273.0, noise_amp=1e-3, noise_seed=5)


@pytest.fixture(autouse=True)
def two_steps_per_launch(monkeypatch):
    monkeypatch.setenv("BGK_POP_VARIANT", "2")


def check(lat, o):
    got = gpu_state(lat, STATE + POPS)
    want = {f: o.field(f) for f in STATE + POPS}
    assert compare_state(got, want, STATE) == []
    assert compare_interior(got, want, POPS) == []


@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("rounding", [0, 1])
@pytest.mark.parametrize("ext", [{}, EXT])
@pytest.mark.parametrize("rows", [0, 1, 64])
def test_two_steps_per_launch_equal_the_oracle(monkeypatch, nx, ny, rounding, ext, rows):
    monkeypatch.setenv("BGK_MOM_ROWS", str(rows))
    p = Params(nx=nx, ny=ny, rounding=rounding, re=3.0, length=float(ny), grav=1e-3)
    o = Oracle(p, **ext)
    o.step(47)
    with Lattice(p, **ext) as lat:
        for n in (20, 1, 3, 23):
            lat.step(n)
        check(lat, o)


def test_uploaded_ghost_velocities_and_subroutines_between_calls():
    p = Params(nx=70, ny=20, re=3.0, length=20.0, grav=1e-3)
    o = Oracle(p)
    with Lattice(p) as lat:
        lat.step(6)
        o.step(6)
        for s in Lattice.STAGES:
            lat.stage(s)
        o.step(1)
        lat.step(4)
        o.step(4)
        check(lat, o)
        u = lat.download("u")
        u[:, 0] += 1e-4  # the west ghost column: enters the thermal ghosts
        lat.upload("u", u)
        o.field("u")[:] = u
        lat.step(4)
        o.step(4)
        check(lat, o)

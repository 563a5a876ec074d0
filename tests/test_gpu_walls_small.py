"""Every boundary type on lattices of a few rows or columns, where rows and columns of
the boundary launch's first workgroup coincide, and on long ones among them, against
the oracle bit for bit, halo included."""
import pytest

from bgk_pcm_amd.lattice import Lattice
from bgk_pcm_amd.params import Params
from golden_io import compare_state
from oracle_py import Oracle
from test_gpu_parity import POPS, STATE, compare_interior, gpu_state
from test_gpu_walls import WALLS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(1, 1), (1, 2), (2, 1), (2, 2), (3, 3), (3, 4), (4, 3), (4, 4),
                                   (1, 40), (40, 1), (2, 300), (3, 700), (700, 2), (600, 4)])
def test_every_wall_equals_the_oracle(nx, ny):
    for k, (w, e, n, s) in enumerate(WALLS):
        p = Params(nx=nx, ny=ny, re=2.0, length=float(ny), west_bc=w, east_bc=e, north_bc=n,
                   south_bc=s, rounding=k % 2)
        o = Oracle(p)
        o.step(7)
        with Lattice(p) as lat:
            lat.step(3)
            for st in Lattice.STAGES:
                lat.stage(st)
            lat.step(3)
            got = gpu_state(lat, STATE + POPS)
        want = {f: o.field(f) for f in STATE + POPS}
        assert compare_state(got, want, STATE) == [], (w, e, n, s)
        assert compare_interior(got, want, POPS) == [], (w, e, n, s)

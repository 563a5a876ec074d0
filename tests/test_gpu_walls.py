"""bgk_step with every boundary type of the reference (one launch for BC_f and
BC_g, one for the rest) against the oracle, bit for bit, halo included: lattices
on either side of the sizes at which the boundary launch spreads over several
workgroups, steps split over calls and mixed with single subroutines."""
import itertools

import pytest

from bgk_pcm_amd.lattice import Lattice
from bgk_pcm_amd.params import Params
from golden_io import compare_state
from oracle_py import Oracle
from test_gpu_parity import POPS, STATE, compare_interior, gpu_state

pytestmark = pytest.mark.gpu

WALLS = [w for w in itertools.product((0, 1, 2, 3, 4), (0, 3, 4), (0, 1, 4, 5, 6), (0, 4, 6))
         if w != (4, 4, 4, 4)]
SIZES = [(7, 8), (8, 8), (8, 7), (9, 12), (270, 9), (11, 300)]


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("part", range(8))
def test_every_wall_equals_the_oracle(nx, ny, part):
    for k, (w, e, n, s) in enumerate(WALLS):
        if k % 8 != part:
            continue
        p = Params(nx=nx, ny=ny, re=2.0, length=float(ny), west_bc=w, east_bc=e, north_bc=n,
                   south_bc=s, rounding=k // 8 % 2)
        o = Oracle(p)
        o.step(9)
        with Lattice(p) as lat:
            lat.step(3)
            for st in Lattice.STAGES:
                lat.stage(st)
            lat.step(5)
            got = gpu_state(lat, STATE + POPS)
        want = {f: o.field(f) for f in STATE + POPS}
        assert compare_state(got, want, STATE) == [], (w, e, n, s)
        assert compare_interior(got, want, POPS) == [], (w, e, n, s)

"""FP32 populations: a step has the same bits alone and within a launch of two, and a
re-basing falls on the same step, so a run does not depend on how it is cut into
calls.  Exact, fields and stored populations, halo included.  Widths on either side
of the 60-column segments and the 256-column tiles (BGK_POP_VARIANT=2 takes lattices
below the size the rule would), sizes on either side of 2^19 nodes by the rule, and
ghost velocities that an upload changed in between, which take steps alone.
"""
import numpy as np
import pytest

from bgk_pcm_amd.lattice import Lattice
from bgk_pcm_amd.params import FP32_DEV, ROUND_CLEAN, Params

pytestmark = pytest.mark.gpu

FIELDS = ("rho", "u", "v", "T", "phi") + tuple(f"{p}{k}" for p in "fg" for k in range(9))
EXT = dict(k_ratio=1.5, noise_amp=1e-3, noise_seed=3)
SHAPES = [(1, 1), (1, 9), (9, 2), (59, 3), (61, 4), (121, 6), (256, 5), (257, 19), (600, 21)]


def params(nx, ny, tau_f):
    return Params(nx=nx, ny=ny, length=float(max(nx, ny)), grav=1e-3, re=1.0, tau_f=tau_f,
                  rounding=ROUND_CLEAN, precision=FP32_DEV)


def run(p, ext, split, between=None):
    with Lattice(p, **ext) as lat:
        for n in split:
            lat.step(n)
            if between:
                between(lat)
                between = None
        nx, ny = p.nx, p.ny
        # (of the halo of f and g only the two corners that no boundary routine
        # writes are defined)
        return {f: lat.download(f) if len(f) != 2 else lat.download(f)[1:-1, 1:-1]
                for f in FIELDS} | {"corners": (lat.gather("f6", [nx + 1], [0])[0],
                                                lat.gather("f7", [nx + 1], [ny + 1])[0])}


def differing(a, b):
    return [f for f in a if not np.array_equal(a[f], b[f])]


@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("tau_f", [1.0, 0.8])
@pytest.mark.parametrize("cold,rebase", [(False, 0), (True, 5), (False, 1)])
def test_every_split_gives_the_same_bits(monkeypatch, nx, ny, tau_f, cold, rebase):
    monkeypatch.setenv("BGK_POP_VARIANT", "2")
    monkeypatch.setenv("BGK_REBASE_EVERY", str(rebase))
    p = params(nx, ny, tau_f)
    ext = dict(EXT, t_cold=273.0) if cold else EXT
    want = run(p, ext, [14])
    for split in ([1] * 14, [3, 5, 6], [2, 1, 11], [7, 7]):
        assert differing(run(p, ext, split), want) == [], split


@pytest.mark.parametrize("nx,ny", [(700, 700), (1003, 777), (2100, 1500)])
def test_splits_on_either_side_of_the_rule(nx, ny):
    p = params(nx, ny, 0.8)
    want = run(p, EXT, [7])
    for split in ([1] * 7, [3, 4], [2, 5]):
        assert differing(run(p, EXT, split), want) == [], split


def test_uploaded_ghost_velocities(monkeypatch):
    def east_u(lat):
        u = lat.download("u")
        u[:, -1] += 1e-3
        lat.upload("u", u)

    out = []
    for variant in (1, 2):
        monkeypatch.setenv("BGK_POP_VARIANT", str(variant))
        out.append([run(params(97, 20, 0.8), dict(EXT, t_cold=272.0), split, east_u)
                    for split in ([3, 8], [3] + [1] * 8)])
    assert differing(out[1][0], out[1][1]) == []
    # against the other arithmetic: FP32 rounding of what 8 steps stored (2e-8 of 273)
    assert np.abs(out[0][0]["T"] - out[1][0]["T"]).max() <= 8 * 6e-8 * 273
    assert np.abs(out[1][0]["T"] - run(params(97, 20, 0.8), dict(EXT, t_cold=272.0),
                                       [11])["T"]).max() > 8 * 6e-8 * 273

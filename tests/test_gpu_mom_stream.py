"""The streaming moment kernel (several time steps per launch) at the places
where it can go wrong: lattices of one to three column segments with the
remainder at every edge of a segment (60 output columns for two steps per
launch, 62 for one, 58 for three), strips of one row and more rows than the
lattice has, and every split of a run into calls.

Bits: a step is the same arithmetic whichever launch it is part of (every
multiply-add written out, the stored precision applied between the steps of a
launch), so all splits give the same fields, halo included.  Against the
oracle: FP64 moments with the tolerance of test_gpu_mom.py (1e-11 after 60
steps, halo included); FP32 moments run the same code with a rounding on
store, and test_gpu_mom.py bounds that rounding.
"""
import numpy as np
import pytest

from bgk_pcm_amd.lattice import Lattice
from bgk_pcm_amd.params import FP32_MOM, FP64_MOM, ROUND_CLEAN, Params
from oracle_py import Oracle
from test_gpu_mom import FIELDS, rel_errors

pytestmark = pytest.mark.gpu

EXT = dict(k_ratio=1.5, noise_amp=1e-3, noise_seed=11)
SHAPES = [(1, 1), (1, 9), (9, 1), (2, 2), (59, 3), (60, 7), (61, 4), (62, 5), (63, 33), (121, 6),
          (124, 40), (175, 70)]


def params(nx, ny, precision, tau_f):
    return Params(nx=nx, ny=ny, length=float(max(nx, ny)), grav=1e-3, rounding=ROUND_CLEAN,
                  tau_f=tau_f, precision=precision)


@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("precision", [FP32_MOM, FP64_MOM])
@pytest.mark.parametrize("tau_f", [1.0, 0.8])
def test_every_split_gives_the_same_bits(monkeypatch, nx, ny, precision, tau_f):
    p = params(nx, ny, precision, tau_f)
    want = None
    for variant, split in [(0, [22]), (0, [1] * 22), (0, [1, 2, 3, 4, 5, 7]), (1, [22]),
                           (3, [22]), (3, [4, 1, 17])]:
        monkeypatch.setenv("BGK_MOM_VARIANT", str(variant))
        with Lattice(p, **EXT) as lat:
            for n in split:
                lat.step(n)
            got = {f: lat.download(f) for f in FIELDS}
        want = want or got
        for f in FIELDS:
            assert np.array_equal(got[f], want[f]), (variant, split, f)


@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("cold", [False, True])
@pytest.mark.parametrize("rows,variant", [(0, 0), (1, 2), (64, 3)])
def test_segments_and_strips_match_the_oracle(monkeypatch, nx, ny, cold, rows, variant):
    monkeypatch.setenv("BGK_MOM_ROWS", str(rows))
    monkeypatch.setenv("BGK_MOM_VARIANT", str(variant))
    p = params(nx, ny, FP64_MOM, 1.0 if variant == 3 else 0.8)
    ext = dict(EXT, t_cold=273.0) if cold else EXT
    o = Oracle(p, **ext)
    o.step(60)
    with Lattice(p, **ext) as lat:
        lat.step(60)
        err = rel_errors(lat, o, interior=False, speed_scale=True)
    assert max(err.values()) <= 1e-11, err

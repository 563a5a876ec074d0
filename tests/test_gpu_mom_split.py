"""Moment storage: a step has the same bits in whichever kernel and launch it runs,
one thread per node through the LDS ring (BGK_MOM_VARIANT=4), one wave per strip
(1: one step per launch, 2: two), mixed as the rule does on large lattices, and in a
gradient's forward run.  Exact, fields and halo: every one of them writes out the same
operations in the same order.  Widths on either side of the ring's 128, 256 and
512 columns, with segments and strips that touch no wall, and ring strips of 1 to 3 rows.
"""
import numpy as np
import pytest

from bgk_pcm_amd.lattice import Lattice
from bgk_pcm_amd.params import FP32_MOM, FP64_MOM, ROUND_CLEAN, Params

pytestmark = pytest.mark.gpu

FIELDS = ("rho", "u", "v", "T", "phi")
EXT = dict(k_ratio=1.5, noise_amp=1e-3, noise_seed=11)
SHAPES = [(1, 1), (1, 9), (9, 1), (2, 3), (61, 7), (130, 5), (256, 6), (513, 9), (300, 9), (700, 5),
          (1100, 9), (1537, 5)]


def params(nx, ny, precision, tau_f):
    return Params(nx=nx, ny=ny, length=float(max(nx, ny)), grav=1e-3, re=2.0, rounding=ROUND_CLEAN,
                  tau_f=tau_f, precision=precision)


def fields(lat):
    return {f: lat.download(f) for f in FIELDS}


@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("precision", [FP32_MOM, FP64_MOM])
@pytest.mark.parametrize("tau_f", [1.0, 0.8])
@pytest.mark.parametrize("cold,rows", [(False, 0), (True, 1), (False, 3)])
def test_ring_and_stream(monkeypatch, nx, ny, precision, tau_f, cold, rows):
    monkeypatch.setenv("BGK_MOM_ROWS", str(rows))
    ext = dict(EXT, t_cold=273.0) if cold else EXT
    want = None
    for variant, split in [(1, [13]), (4, [13]), (2, [13]), (4, [1, 5, 7])]:
        monkeypatch.setenv("BGK_MOM_VARIANT", str(variant))
        with Lattice(params(nx, ny, precision, tau_f), **ext) as lat:
            for n in split:
                lat.step(n)
            got = fields(lat)
        want = want or got
        for f in FIELDS:
            assert np.array_equal(got[f], want[f]), (variant, split, f)


@pytest.mark.parametrize("nx,ny", [(1, 300), (2, 300), (3, 50), (16, 16), (64, 2500), (64, 2600), (64, 4097),
                                   (65, 40), (97, 61), (144, 30), (145, 689), (145, 690), (145, 904),
                                   (160, 13200), (161, 13100)])
@pytest.mark.parametrize("precision", [FP32_MOM, FP64_MOM])
@pytest.mark.parametrize("tau_f", [1.0, 0.8])
def test_short_calls_on_small_and_narrow_lattices(monkeypatch, nx, ny, precision, tau_f):
    """The rule's own launches (ring launches alone, two at a call's end, and none),
    at its lines, against one strip launch per step of one call."""
    want = None
    for variant, split in [(1, [10]), (0, [10]), (0, [1] * 10), (0, [2, 3, 5]), (0, [4, 6])]:
        monkeypatch.setenv("BGK_MOM_VARIANT", str(variant))
        with Lattice(params(nx, ny, precision, tau_f), **EXT) as lat:
            for n in split:
                lat.step(n)
            got = fields(lat)
        want = want or got
        for f in FIELDS:
            assert np.array_equal(got[f], want[f]), (variant, split, f)


@pytest.mark.parametrize("nx,ny,precision", [(4100, 2050, FP32_MOM), (2900, 2899, FP64_MOM),
                                             (250, 2200, FP64_MOM), (130, 30000, FP32_MOM)])
@pytest.mark.parametrize("tau_f", [1.0, 0.8])
def test_splits_of_a_run_on_a_large_lattice(nx, ny, precision, tau_f):
    want = None
    for split in ([7], [1] * 7, [3, 4], [2, 5]):
        with Lattice(params(nx, ny, precision, tau_f), **EXT) as lat:
            for n in split:
                lat.step(n)
            got = fields(lat)
        want = want or got
        for f in FIELDS:
            assert np.array_equal(got[f], want[f]), (split, f)


@pytest.mark.parametrize("nx,ny,precision,tau_f", [(8200, 4100, FP32_MOM, 1.0),
                                                   (4100, 2050, FP32_MOM, 0.8),
                                                   (2900, 2899, FP64_MOM, 1.0)])
def test_recorded_forward_run_on_a_large_lattice(nx, ny, precision, tau_f):
    p = params(nx, ny, precision, tau_f)
    with Lattice(p, **EXT) as lat:
        lat.step(7)
        want = fields(lat)
    with Lattice(p, **EXT) as lat:
        lat.adj_setup_binomial(7, 3, [5, nx], [9, ny])
        lat.adj_forward()
        got = fields(lat)
    for f in FIELDS:
        assert np.array_equal(got[f], want[f]), f

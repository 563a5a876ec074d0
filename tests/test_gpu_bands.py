"""The one-step population kernels on either side of the sizes at which their rows
go to the XCDs in bands and their planes through the caches (more than 2^16
nodes; two states of at most 256 MB), heights that leave the last band short or
some XCDs without rows.

FP64: the oracle's fields bit for bit, halo included.  FP32: the FP64 run's within
1e-6 of each field's largest value (liquid fraction for phi; u and v against the
larger velocity) after 4 steps: the stored deviations, about 1e-2 of the
populations, are rounded to 6e-8 of themselves once a step, which leaves 2.4e-9
of w_k m and a hundred times that for the velocities; with FP32 collision
arithmetic 1e-4, the bound of tests/test_gpu_fp32.py."""
import numpy as np
import pytest

from bgk_pcm_amd.lattice import Lattice
from bgk_pcm_amd.params import FP32_DEV, FP32_MOM, FP64, FP64_MOM, ROUND_CLEAN, ROUND_STEP7, Params
from golden_io import compare_state
from oracle_py import Oracle
from test_gpu_parity import POPS, STATE, compare_interior, gpu_state

pytestmark = pytest.mark.gpu

SIZES = [(7, 1), (300, 7), (5, 9), (256, 256), (257, 256), (65, 1009), (1031, 66)]
FIELDS = ("rho", "u", "v", "T", "phi")


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("east", [4, 3], ids=["no_slip", "outlet"])
@pytest.mark.parametrize("rounding", [ROUND_CLEAN, ROUND_STEP7], ids=["clean", "step7"])
def test_fp64_step_equals_the_oracle(monkeypatch, nx, ny, east, rounding):
    monkeypatch.setenv("BGK_POP_VARIANT", "1")
    p = Params(nx=nx, ny=ny, re=2.0, length=float(ny), east_bc=east, rounding=rounding)
    o = Oracle(p)
    o.step(4)
    with Lattice(p) as lat:
        lat.step(4)
        got = gpu_state(lat, STATE + POPS)
    want = {f: o.field(f) for f in STATE + POPS}
    assert compare_state(got, want, STATE) == []
    assert compare_interior(got, want, POPS) == []


@pytest.mark.parametrize("nx,ny", SIZES + [(2048, 900)])
@pytest.mark.parametrize("single", [0, 1], ids=["fp64_collision", "fp32_collision"])
def test_fp32_step_follows_fp64(monkeypatch, nx, ny, single):
    monkeypatch.setenv("BGK_POP_VARIANT", "1")
    p = Params(nx=nx, ny=ny, length=float(max(nx, ny)), grav=1e-3, re=1.0, tau_f=0.8,
               rounding=ROUND_CLEAN)
    out = []
    for q in (p.replace(precision=FP64), p.replace(precision=FP32_DEV, fp32_collision=single)):
        with Lattice(q, k_ratio=1.5, noise_amp=1e-3, noise_seed=3) as lat:
            lat.step(4)
            out.append({f: lat.download(f) for f in FIELDS})
    want, got = out
    speed = max(np.abs(want["u"]).max(), np.abs(want["v"]).max())
    for f in FIELDS:
        scale = speed if f in "uv" else 1.0 if f == "phi" else np.abs(want[f]).max()
        err = np.abs(got[f] - want[f]).max() / scale
        print(nx, ny, f, err, flush=True)
        assert err <= (1e-4 if single else 1e-6), (f, err)


@pytest.mark.parametrize("precision,nx,ny", [(FP64_MOM, 645, 640), (FP32_MOM, 1003, 941),
                                             (FP32_MOM, 1290, 1003)])
@pytest.mark.parametrize("tau_f", [1.0, 0.8])
def test_moment_stores_through_the_caches(precision, nx, ny, tau_f):
    """Sizes whose plain launches store through the caches: the bits of single
    steps, each the last launch of its call, which stores past them."""
    p = Params(nx=nx, ny=ny, length=float(ny), grav=1e-3, rounding=ROUND_CLEAN, tau_f=tau_f,
               precision=precision)
    out = []
    for split in ([11], [1] * 11):
        with Lattice(p, k_ratio=1.5, noise_amp=1e-3, noise_seed=3) as lat:
            for n in split:
                lat.step(n)
            out.append({f: lat.download(f) for f in FIELDS})
    for f in FIELDS:
        assert np.array_equal(out[0][f], out[1][f]), f

"""FP32 populations with two steps per launch against one step per launch and
the clean FP64 oracle, at the edges of the 60-column segments and of the strips.

Every split of a run gives the fields of one-step launches to 1e-6 relative to
each field's largest value (liquid fraction for phi; u and v against the larger
velocity) after 40 steps: both round the stored deviations, about 1e-2 of the
populations at most here, to FP32 (6e-8) once per step, so each is within 40 x
6e-8 x 1e-2 = 2.4e-8 of w_k m of the FP64 run, and the velocities, about 1e-2
and more of the sums they come from, within 1e-6.  Re-basings every 7 steps
fall on the same steps whatever the split."""
import numpy as np
import pytest

from bgk_pcm_amd.lattice import Lattice
from bgk_pcm_amd.params import FP32_DEV, ROUND_CLEAN, Params

pytestmark = pytest.mark.gpu

FIELDS = ("rho", "u", "v", "T", "phi")
SHAPES = [(1, 1), (1, 9), (9, 2), (59, 3), (60, 7), (61, 4), (62, 5), (63, 33), (121, 6), (185, 21)]
EXT = dict(k_ratio=1.5, noise_amp=1e-3, noise_seed=3)


def run(monkeypatch, p, ext, variant, split):
    monkeypatch.setenv("BGK_POP_VARIANT", str(variant))
    with Lattice(p, **ext) as lat:
        for n in split:
            lat.step(n)
        return {f: lat.download(f) for f in FIELDS}


@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("tau_f", [1.0, 0.8])
@pytest.mark.parametrize("cold,rebase,rows", [(False, 0, 0), (True, 7, 1)])
def test_two_steps_per_launch(monkeypatch, nx, ny, tau_f, cold, rebase, rows):
    monkeypatch.setenv("BGK_REBASE_EVERY", str(rebase))
    monkeypatch.setenv("BGK_MOM_ROWS", str(rows))
    p = Params(nx=nx, ny=ny, length=float(max(nx, ny)), grav=1e-3, re=1.0, tau_f=tau_f,
               rounding=ROUND_CLEAN, precision=FP32_DEV)
    ext = dict(EXT, t_cold=273.0) if cold else EXT
    want = run(monkeypatch, p, ext, 1, [40])
    speed = max(np.abs(want["u"]).max(), np.abs(want["v"]).max())
    for split in ([40], [20, 1, 19], [4] * 10):
        got = run(monkeypatch, p, ext, 2, split)
        for f in FIELDS:
            a, b = got[f], want[f]
            scale = speed if f in "uv" else 1.0 if f == "phi" else np.abs(b).max()
            assert np.abs(a - b).max() <= 1e-6 * scale, (split, f, np.abs(a - b).max() / scale)

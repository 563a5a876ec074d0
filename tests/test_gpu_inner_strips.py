"""Strips and segments that touch no wall, in the instantiations that only large
lattices take by rule: launches of two steps that store the state between them, and
plain launches that store through the caches.  Exact: a step has the same bits in
either.
"""
import numpy as np
import pytest

from bgk_pcm_amd.lattice import Lattice
from bgk_pcm_amd.params import FP32_MOM, FP64_MOM, ROUND_CLEAN, Params

pytestmark = pytest.mark.gpu

FIELDS = ("rho", "u", "v", "T", "phi")


def params(nx, ny, precision, tau_f):
    return Params(nx=nx, ny=ny, length=float(max(nx, ny)), grav=2e-3, rounding=ROUND_CLEAN,
                  tau_f=tau_f, precision=precision, stefan_number=0.1)


@pytest.mark.parametrize("nx,ny", [(185, 40), (250, 23), (245, 70)])
@pytest.mark.parametrize("precision", [FP64_MOM, FP32_MOM])
@pytest.mark.parametrize("tau_f", [1.0, 0.8])
@pytest.mark.parametrize("rows", [0, 1, 3])
def test_schedules_that_keep_the_state_between_two_steps(monkeypatch, nx, ny, precision, tau_f,
                                                         rows):
    """Four column segments and up, of which two meet no wall, in strips of one row, of
    three and as the rule cuts them: record and fields have the bits of one step per
    launch; so has the gradient, with the strips that the adjoint kernel shares."""
    monkeypatch.setenv("BGK_MOM_ROWS", str(rows))
    p = params(nx, ny, precision, tau_f)
    pi = [1, nx // 2, 61, 122, nx]
    pj = [1, ny // 2, 7, 9, ny]
    for nsteps in (5, 12):
        want = None
        for variant, kind, n in [(1, "seg", nsteps), (2, "seg", nsteps), (2, "seg", 1),
                                 (2, "seg", 3), (2, "states", 2), (2, "states", 4),
                                 (2, "states", 9)]:
            monkeypatch.setenv("BGK_MOM_VARIANT", str(variant))
            with Lattice(p, initialize=False, t_hot=283.5, k_ratio=1.3, noise_amp=1e-2,
                         noise_seed=5) as lat:
                lat.initialization()
                if kind == "seg":
                    lat.adj_setup(nsteps, n, pi, pj)
                else:
                    lat.adj_setup_binomial(nsteps, n, pi, pj)
                rec = lat.adj_forward()
                got = {f: lat.download(f) for f in FIELDS}
                g = lat.adj_backward(2.0 * (rec - 280.0) / rec.size)
            want = want or (rec, g, got)
            case = (nsteps, variant, kind, n)
            assert np.array_equal(rec, want[0]), case
            assert np.array_equal(g, want[1]), case
            for f in FIELDS:
                assert np.array_equal(got[f], want[2][f]), (case, f)


# bytes per node of a stored state and the window in MiB of two of them
STATE_BYTES = {(FP32_MOM, 0.8): 56, (FP32_MOM, 1.0): 44, (FP64_MOM, 0.8): 88, (FP64_MOM, 1.0): 64}
WINDOW = {FP32_MOM: (96, 256), FP64_MOM: (64, 256)}


@pytest.mark.parametrize("precision,tau_f,nx,ny", [
    (FP64_MOM, 1.0, 1003, 777), (FP64_MOM, 1.0, 740, 735), (FP64_MOM, 0.8, 645, 640),
    (FP64_MOM, 0.8, 1203, 1200), (FP32_MOM, 1.0, 1203, 1003), (FP32_MOM, 0.8, 1003, 941),
    (FP32_MOM, 0.8, 1501, 1500)])
def test_stores_through_the_caches(precision, tau_f, nx, ny):
    """Sizes whose plain launches store through the caches, against single steps, each
    the last launch of its call, which stores past them."""
    mib = nx * ny * 2 * STATE_BYTES[precision, tau_f] / 2**20
    assert WINDOW[precision][0] + 1 <= mib <= WINDOW[precision][1] - 1, mib
    p = params(nx, ny, precision, tau_f)
    out = []
    for split in ([11], [1] * 11):
        with Lattice(p, k_ratio=1.5, noise_amp=1e-3, noise_seed=3) as lat:
            for n in split:
                lat.step(n)
            out.append({f: lat.download(f) for f in FIELDS})
    for f in FIELDS:
        assert np.array_equal(out[0][f], out[1][f]), f

"""Moment lattices so wide that a few rows, or one, are more elements than a 32-bit
byte offset reaches: fields near the east wall equal, bit for bit, those of a narrow
lattice of the same height (a node depends on the nodes within one column per step),
those near the west wall the narrow lattice's too, and the columns between are all
alike."""
import numpy as np
import pytest
import torch

from bgk_pcm_amd.lattice import Lattice
from bgk_pcm_amd.params import FP64_MOM, ROUND_CLEAN, Params

pytestmark = pytest.mark.gpu


def columns(lat, i):
    i = np.asarray(i)
    ii, jj = [a.ravel() for a in np.meshgrid(i, np.arange(lat.ny + 2), indexing="ij")]
    return {f: lat.gather(f, ii, jj).reshape(i.size, -1) for f in ("rho", "u", "v", "T", "phi")}


@pytest.mark.parametrize("nx,ny", [((1 << 27) + 100, 1), (46_000_000, 8)])
def test_far_columns(nx, ny):
    free, _ = torch.cuda.mem_get_info()
    if free < 232 * (nx + 2) * (ny + 2) + (4 << 30):
        pytest.skip("needs a device of 288 GB to itself")
    p = Params(nx=200, ny=ny, length=float(ny), tau_f=0.8, grav=1e-3, re=1.0,
               rounding=ROUND_CLEAN, precision=FP64_MOM)
    steps = (2, 1, 4)
    with Lattice(p) as lat:
        for n in steps:
            lat.step(n)
        east = columns(lat, np.arange(180, 202))
        plain = columns(lat, np.arange(100, 120))
    print(f"{nx} x {ny}", flush=True)
    with Lattice(p.replace(nx=nx)) as lat:
        for n in steps:
            lat.step(n)
        far = columns(lat, np.arange(nx - 20, nx + 2))
        half = columns(lat, np.arange(nx // 2, nx // 2 + 20))
        # the west of the lattice is liquid up to Nx/40: alike between the wall and there
        wet = columns(lat, np.arange(nx // 80, nx // 80 + 20))
    for f in far:
        assert np.array_equal(far[f], east[f]), f
        assert np.array_equal(half[f], plain[f]), f
        assert np.array_equal(wet[f], np.broadcast_to(wet[f][:1], wet[f].shape)), f


def test_gradient_at_the_far_wall():
    """The gradient of two steps' record beside the cold east wall (its dependence on
    the conductivity ratio; the others vanish in the solid): the narrow lattice's to
    1e-12, the order of the sums over workgroups apart."""
    nx, ny = (1 << 27) + 100, 1
    free, _ = torch.cuda.mem_get_info()
    if free < 620 * (nx + 2) * (ny + 2) + (4 << 30):
        pytest.skip("needs a device of 288 GB to itself")
    p = Params(nx=200, ny=ny, length=float(ny), tau_f=1.0, grav=1e-3, rounding=ROUND_CLEAN,
               precision=FP64_MOM)
    out = []
    for n in (200, nx):
        print(n, flush=True)
        with Lattice(p.replace(nx=n), initialize=False, k_ratio=1.5, t_cold=271.0) as lat:
            lat.initialization()
            lat.adj_setup(2, 2, [n - 1, n], [1, 1])
            rec = lat.adj_forward()
            out.append((rec, lat.adj_backward(2.0 * (rec - 270.0))))
    assert np.array_equal(out[0][0], out[1][0])
    assert abs(out[0][1][1]) > 1e-6
    np.testing.assert_allclose(out[1][1], out[0][1], rtol=1e-12, atol=0.0)

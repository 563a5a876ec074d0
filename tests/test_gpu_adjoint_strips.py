"""The adjoint kernel at the edges of its split: a wave stores 62 columns and a
strip a few rows, so widths on either side of one and two waves, lattices of one
and two columns or rows, and heights on either side of a strip, against autograd
of the CPU reference.

Tolerances, derived before the first run.  FP64: both evaluate the same chain
rule; temperatures are held to 1e-16 of 273 and differ by about 1, so a step's
adjoint carries 1e-13 at worst and the 24 steps 24 times that if nothing cancels;
a component of the gradient sums terms of either sign, none larger than the
largest component.  1e-9 of that one leaves a factor of 100, and 1e-7 of a
component is the bound of tests/test_gpu_adjoint.py.  FP32: 6e-8 of 273 over
differences of 1 is 2e-5 a step, 4e-4 over 24 if nothing cancels: 1e-3 of the
largest component.
"""
import numpy as np
import pytest
import torch

from bgk_pcm_amd.lattice import Lattice
from bgk_pcm_amd.params import FP32_MOM, FP64_MOM, ROUND_CLEAN, Params
from torch_ref import probe_record

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (1, 40), (2, 3), (61, 7), (62, 5), (63, 4), (64, 33), (124, 6), (125, 9),
         (187, 2), (40, 1), (300, 17)]


@pytest.mark.parametrize("tau_f", [1.0, 0.8])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_gradient_at_the_edges_of_the_split(nx, ny, tau_f):
    p = Params(nx=nx, ny=ny, length=float(max(nx, ny)), grav=2e-3, rounding=ROUND_CLEAN,
               tau_f=tau_f, re=2.0)
    nsteps, seg = 24, 5
    pi = sorted({1, min(nx, 2), min(nx, 62), min(nx, 63), nx})
    pj = [1 + (3 * k) % ny for k in range(len(pi))]
    theta0 = (0.1, 1.3, 283.5)
    th = torch.tensor(theta0, dtype=torch.float64, requires_grad=True)
    rec_ref = probe_record(p, th, pi, pj, nsteps)
    ((rec_ref - 280.0) ** 2).mean().backward()
    g_ref = th.grad.numpy()
    print(f"{nx}x{ny} tau_f {tau_f}: autograd {g_ref}", flush=True)
    largest = np.abs(g_ref).max()
    for prec, rtol, of_largest in ((FP64_MOM, 1e-7, 1e-9), (FP32_MOM, 0.0, 1e-3)):
        with Lattice(p.replace(precision=prec, stefan_number=theta0[0]), initialize=False,
                     t_hot=theta0[2], k_ratio=theta0[1]) as lat:
            lat.initialization()
            lat.adj_setup(nsteps, seg, pi, pj)
            rec = lat.adj_forward()
            g = lat.adj_backward(2.0 * (rec - 280.0) / rec.size)
        print("precision", prec, g, flush=True)
        np.testing.assert_allclose(g, g_ref, rtol=rtol, atol=of_largest * largest)


@pytest.mark.parametrize("precision", [FP64_MOM, FP32_MOM])
@pytest.mark.parametrize("tau_f", [1.0, 0.8])
@pytest.mark.parametrize("nx,ny", [(1, 3), (59, 4), (61, 9), (64, 33)])
def test_schedules_that_keep_the_state_between_two_steps(monkeypatch, nx, ny, precision, tau_f):
    """Launches of two steps that store the state between them: the record and the
    gradient have the bits of one step per launch, whatever is kept."""
    p = Params(nx=nx, ny=ny, length=float(max(nx, ny)), grav=2e-3, rounding=ROUND_CLEAN,
               tau_f=tau_f, precision=precision, stefan_number=0.1)
    pi = sorted({1, min(nx, 61), nx})
    pj = [1 + (3 * k) % ny for k in range(len(pi))]
    for nsteps in (1, 2, 3, 4, 5, 23):
        want = None
        for variant, kind, n in [(1, "seg", nsteps), (2, "seg", nsteps), (2, "seg", 1),
                                 (2, "seg", min(4, nsteps)), (2, "seg", min(7, nsteps)),
                                 (2, "states", 1), (2, "states", 2), (2, "states", 3),
                                 (2, "states", 5), (2, "states", 9)]:
            monkeypatch.setenv("BGK_MOM_VARIANT", str(variant))
            with Lattice(p, initialize=False, t_hot=283.5, k_ratio=1.3) as lat:
                lat.initialization()
                if kind == "seg":
                    lat.adj_setup(nsteps, n, pi, pj)
                else:
                    lat.adj_setup_binomial(nsteps, n, pi, pj)
                rec = lat.adj_forward()
                T = lat.download("T")
                g = lat.adj_backward(2.0 * (rec - 280.0) / rec.size)
            want = want or (rec, g, T)
            case = (nsteps, variant, kind, n)
            assert np.array_equal(rec, want[0]), case
            assert np.array_equal(T, want[2]), case
            assert np.array_equal(g, want[1]), case

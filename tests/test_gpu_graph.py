"""Steps recorded in a HIP graph: every replay gives the eager call's fields, bit for
bit, also after an initialization, an upload or eager calls since the recording, and
a recording that is not replayed leaves the handle as it was.  All storages, calls of an even
number of steps (each ends in the buffers it began in); walls other than no-slip and
the subroutines one by one, which exchange no buffers, for any number.
"""
import numpy as np
import pytest
import torch

from bgk_pcm_amd.lattice import Lattice
from bgk_pcm_amd.params import FP32_DEV, FP32_MOM, FP64, FP64_MOM, ROUND_CLEAN, Params

pytestmark = pytest.mark.gpu

FIELDS = ("rho", "u", "v", "T", "phi")
EXT = dict(k_ratio=1.5, noise_amp=1e-2, noise_seed=3)


def fields(lat):
    return {f: lat.download(f) for f in FIELDS}


def differing(a, b):
    return [f for f in FIELDS if not np.array_equal(a[f], b[f])]


def record(lat, stream, call):
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        call(lat)
    return graph


def replay(graph, stream):
    with torch.cuda.stream(stream):
        graph.replay()
    torch.cuda.synchronize()


def check(p, call, upload):
    with Lattice(p, **EXT) as lat:
        want = []
        for _ in range(5):
            call(lat)
            want.append(fields(lat))
    stream = torch.cuda.Stream()
    with Lattice(p, **EXT) as lat:
        lat.set_stream(stream.cuda_stream)
        call(lat)
        graph = record(lat, stream, call)
        assert differing(fields(lat), want[0]) == []
        lat.initialization()
        for n in range(3):
            replay(graph, stream)
            assert differing(fields(lat), want[n]) == [], n
        call(lat)  # eager, between replays
        assert differing(fields(lat), want[3]) == []
        replay(graph, stream)
        assert differing(fields(lat), want[4]) == []
        if upload:  # a T of the host's, then a replay, then an eager call
            T = want[1]["T"] + 0.25
            lat.upload("T", T)
            replay(graph, stream)
            call(lat)
            got = fields(lat)
            with Lattice(p, **EXT) as other:
                for _ in range(5):
                    call(other)
                other.upload("T", T)
                call(other)
                call(other)
                assert differing(got, fields(other)) == []
        # a recording that is never replayed
        lat.initialization()
        call(lat)
        record(lat, stream, call)
        call(lat)
        assert differing(fields(lat), want[1]) == []


@pytest.mark.parametrize("precision", [FP64, FP32_DEV, FP32_MOM, FP64_MOM])
@pytest.mark.parametrize("tau_f", [1.0, 0.8])
@pytest.mark.parametrize("nsteps", [2, 4, 6])
@pytest.mark.parametrize("variant", [0, 3])
def test_steps_of_the_cavity(monkeypatch, precision, tau_f, nsteps, variant):
    monkeypatch.setenv("BGK_MOM_VARIANT", str(variant))
    p = Params(nx=97, ny=61, length=61.0, tau_f=tau_f, grav=1e-3, rounding=ROUND_CLEAN,
               precision=precision)
    check(p, lambda lat: lat.step(nsteps), precision in (FP64, FP32_DEV))


@pytest.mark.parametrize("west,east", [(1, 3), (0, 0), (4, 3)])
@pytest.mark.parametrize("nsteps", [1, 2, 3])
def test_steps_with_other_walls(west, east, nsteps):
    p = Params(nx=70, ny=33, length=33.0, re=4.0, west_bc=west, east_bc=east, grav=1e-3,
               rounding=ROUND_CLEAN)
    check(p, lambda lat: lat.step(nsteps), True)


def test_adjoint_runs_between_replays():
    """A recorded gradient run of an even number of steps leaves the handle in the
    buffers that a recording of steps starts from."""
    p = Params(nx=97, ny=61, length=61.0, tau_f=1.0, grav=1e-3, rounding=ROUND_CLEAN,
               precision=FP64_MOM)

    def run(lat, replay_steps):
        lat.adj_setup(6, 3, [40], [30])
        replay_steps()
        lat.adj_forward()
        replay_steps()
        return fields(lat)

    with Lattice(p, **EXT) as lat:
        want = run(lat, lambda: lat.step(4))
    stream = torch.cuda.Stream()
    with Lattice(p, **EXT) as lat:
        lat.set_stream(stream.cuda_stream)
        lat.step(4)
        graph = record(lat, stream, lambda lat: lat.step(4))
        lat.initialization()
        assert differing(run(lat, lambda: replay(graph, stream)), want) == []


def test_subroutines():
    def call(lat):
        for s in Lattice.STAGES:
            lat.stage(s)

    check(Params(nx=70, ny=33, length=33.0, grav=1e-3), call, True)

"""Fields and gathers on their way to the host: one staging chunk and several,
the last one partial; a leading dimension larger than a row; a plane inside a
pair; more gathered nodes than one buffer holds; two threads with a handle each.
Exact: the values are copied."""
import ctypes
import threading

import numpy as np
import pytest

from bgk_pcm_amd.lattice import FIELD_ID, Lattice, load_library
from bgk_pcm_amd.params import FP32_DEV, Params
from oracle_py import Oracle

pytestmark = pytest.mark.gpu

EXT = dict(noise_amp=1e-2, noise_seed=9)


@pytest.mark.parametrize("nx,ny", [(1, 1), (722, 722), (723, 722), (1501, 903), (40000, 30)])
def test_download_equals_the_initial_fields(nx, ny):
    p = Params(nx=nx, ny=ny, re=3.0, length=float(ny))
    o = Oracle(p, **EXT)
    with Lattice(p, **EXT) as lat:
        for f in ("T", "rho", "phi", "g3", "f0"):
            assert np.array_equal(lat.download(f), o.field(f)), f
        wide = np.full((ny + 2, nx + 7), -1.0)
        rc = load_library().bgk_download(lat._h, FIELD_ID["T"],
                                         wide.ctypes.data_as(ctypes.POINTER(ctypes.c_double)),
                                         nx + 7)
        assert rc == 0
        assert np.array_equal(wide[:, :nx + 2], o.field("T")) and np.all(wide[:, nx + 2:] == -1.0)


def test_gather_of_more_nodes_than_a_buffer():
    p = Params(nx=300, ny=200)
    r = np.random.default_rng(1)
    i, j = r.integers(0, 302, 300001), r.integers(0, 202, 300001)
    for prec in (0, FP32_DEV):
        with Lattice(p.replace(precision=prec), **EXT) as lat:
            for f in ("T", "f5"):
                assert np.array_equal(lat.gather(f, i, j), lat.download(f)[j, i]), (prec, f)


def test_gather_of_several_fields():
    """More fields than a launch takes, FP32 deviations among them, and node
    counts on either side of what the launch's arguments hold."""
    names = ["T", "f5", "u", "phi", "g0", "v", "rho", "f1", "g8", "T", "phi_prec"]
    ids = np.array([FIELD_ID[f] for f in names], dtype=np.int32)
    r = np.random.default_rng(2)
    P32, PD = ctypes.POINTER(ctypes.c_int32), ctypes.POINTER(ctypes.c_double)
    for prec in (0, FP32_DEV):
        with Lattice(Params(nx=50, ny=40, precision=prec), **EXT) as lat:
            lat.step(3)
            for n in (0, 1, 32, 33, 400):
                i = r.integers(0, 52, n).astype(np.int32)
                j = r.integers(0, 42, n).astype(np.int32)
                out = np.empty((len(names), n))
                rc = lat._lib.bgk_gather_fields(lat._h, len(names), ids.ctypes.data_as(P32), n,
                                                i.ctypes.data_as(P32), j.ctypes.data_as(P32),
                                                out.ctypes.data_as(PD))
                assert rc == 0
                for k, f in enumerate(names):
                    assert np.array_equal(out[k], lat.download(f)[j, i]), (prec, n, f)
            assert np.array_equal(lat.prof_x()[24], np.array(lat.probe()))


def test_two_threads_with_a_handle_each():
    bad = []

    def work(seed):
        p = Params(nx=900, ny=800)
        ext = dict(EXT, noise_seed=seed)
        o = Oracle(p, **ext)  # (owns the memory its fields are views of)
        want = o.field("T").copy()
        with Lattice(p, **ext) as lat:
            for _ in range(5):
                if not np.array_equal(lat.download("T"), want) or \
                        not np.array_equal(lat.gather("T", [5, 9], [7, 3]), want[[7, 3], [5, 9]]):
                    bad.append(seed)

    ts = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert bad == []

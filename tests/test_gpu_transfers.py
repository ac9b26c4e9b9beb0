"""Copies between the caller's arrays and the device: one pass through the pinned buffer up to
4 MiB; above it chunks of 2 MiB on one to several threads, into the device from 8 MiB and the
runtime's copies up to there.  56 bytes a particle go in, 104 come out."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one particle; the last sizes of the small path and the first past it, out and in; chunk ends inside
# and between the arrays; the first size in chunks both ways; every thread busy
SIZES = [1, 40329, 40330, 74898, 74899, 87381, 87382, 149796, 149797, 1200001]


def pinned(a):
    """A copy of the array in pinned host memory, and its address."""
    import hip_mem as M
    p = C.c_void_p()
    assert M.runtime().hipHostMalloc(C.byref(p), C.c_size_t(a.nbytes), 0) == 0
    b = np.ctypeslib.as_array((C.c_double * a.size).from_address(p.value)).reshape(a.shape)
    b[:] = a
    return b, p


def cloud(n, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((n, 3)), rng.standard_normal((n, 4))


@pytest.mark.parametrize("n", SIZES)
def test_round_trip(vpmlib, n):
    """What goes in comes out, also into a buffer in use a moment ago and from pinned arrays."""
    with vpmlib.VPM(vpmlib.Params.make(0.125)) as c:
        for seed in (1, 2):
            x, q = cloud(n, seed)
            held = []
            if seed == 2:
                import hip_mem as M
                (x, px), (q, pq) = pinned(x), pinned(q)
                held = [px, pq]
            print("case: transfer", n, seed, flush=True)
            c.upload(x, q)
            xo, qo = c.download()[:2]
            assert np.array_equal(x, xo) and np.array_equal(q, qo)
            for p in held:
                M.runtime().hipHostFree(p)


def test_contexts_on_threads(vpmlib):
    """Two threads with a context each, small and large transfers in turn."""
    bad = []

    def run(seed):
        try:
            with vpmlib.VPM(vpmlib.Params.make(0.125)) as c:
                for n in (150000, 7, 90000, 400000):
                    x, q = cloud(n, seed + n)
                    c.upload(x, q)
                    xo, qo = c.download()[:2]
                    if not (np.array_equal(x, xo) and np.array_equal(q, qo)):
                        bad.append((seed, n))
        except Exception as e:  # shown by the main thread
            bad.append(repr(e))

    print("case: transfers on two threads", flush=True)
    th = [threading.Thread(target=run, args=(s,)) for s in (1, 2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad


@pytest.mark.parametrize("n", [5, 200000])
def test_missing_array_is_refused(vpmlib, n):
    """A null source is an error of the call, not a crash, and of that call alone."""
    with vpmlib.VPM(vpmlib.Params.make(0.125)) as c:
        x, q = cloud(n, 3)
        assert c._lib.vpmx_particles_upload(c._h, x.ctypes.data_as(C.POINTER(C.c_double)), None, n, 3) != 0
        c.upload(x, q)
        assert np.array_equal(c.download()[1], q)

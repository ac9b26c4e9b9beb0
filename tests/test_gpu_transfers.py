"""Copies between the caller's arrays and the device: one pass through the pinned buffer up to
4 MiB, chunks of 2 MiB on one to several threads above it.  56 bytes a particle go in."""
import ctypes as C
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# one particle; the last size of the small path and the first of the chunked one; chunk ends inside
# and between the arrays; every thread busy
SIZES = [1, 74898, 74899, 87381, 87382, 1200001]


def cloud(n, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((n, 3)), rng.standard_normal((n, 4))


@pytest.mark.parametrize("n", SIZES)
def test_round_trip(vpmlib, n):
    """What goes in comes out, also into a buffer in use a moment ago and from pinned arrays."""
    with vpmlib.VPM(vpmlib.Params.make(0.125)) as c:
        for seed in (1, 2):
            x, q = cloud(n, seed)
            if seed == 2:
                x, q = torch.from_numpy(x).pin_memory().numpy(), torch.from_numpy(q).pin_memory().numpy()
            print("case: transfer", n, seed, flush=True)
            c.upload(x, q)
            xo, qo = c.download()[:2]
            assert np.array_equal(x, xo) and np.array_equal(q, qo)


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
    """A null source is an error of the call, not a crash."""
    with vpmlib.VPM(vpmlib.Params.make(0.125)) as c:
        x, _ = cloud(n, 3)
        assert c._lib.vpmx_particles_upload(c._h, x.ctypes.data_as(C.POINTER(C.c_double)), None, n, 3) != 0

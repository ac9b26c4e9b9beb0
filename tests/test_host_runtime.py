"""Host-side handling of runtime calls that fail, on a stand-in for the HIP runtime (fake_hip.c: no GPU,
kernels do nothing): each test runs in a process of its own that loads the stand-in before libvpmx."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes, sys
import numpy as np
F = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
for f in (F.fake_calls, F.fake_done, F.fake_held):
    f.restype = ctypes.c_long
F.fake_fail.argtypes = [ctypes.c_int, ctypes.c_long]
MALLOC, MEMCPY, HOSTMALLOC, STREAM, EVENT, LAUNCH, RECORD, ASYNC = range(8)
sys.path.insert(0, %r)
from vpm_free_amd import vpm as V
rng = np.random.default_rng(1)
def fails(f, *a):
    try:
        f(*a)
    except V.VpmError:
        return True
    return False
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    cc = shutil.which("gcc")
    if not cc:
        pytest.skip("no host compiler")
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run([cc, "-shared", "-fPIC", "-O1", "-w", os.path.join(HERE, "fake_hip.c"), "-o", so], check=True)

    def go(code):
        r = subprocess.run([sys.executable, "-c", PRELUDE % (so, os.path.dirname(HERE)) + code], capture_output=True,
                           text=True, timeout=300)
        assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]

    return go


@pytest.mark.parametrize("itree", [0, 1])
def test_tables_after_a_failed_copy(run, itree):
    """A table whose upload failed is uploaded by the next call: whichever copy of a first pmesh call
    fails, that call is refused and the next one completes the set."""
    run("""
itree = %d
n = np.array([13, 15, 17], np.int32)
h = np.array([0.1, 0.11, 0.12])
xb = np.zeros(6)
a = rng.standard_normal((17, 15, 13, 3))
def call(c):
    c.stage_pmesh_inf(xb, h, n, a, np.zeros_like(a), itree=itree, levmax=2)
with V.VPM(V.Params.make(0.125)) as c:
    n0 = F.fake_done(MEMCPY)
    call(c)
    need = F.fake_done(MEMCPY) - n0
assert need > 4
for k in range(1, need + 1):
    with V.VPM(V.Params.make(0.125)) as c:
        n0 = F.fake_done(MEMCPY)
        F.fake_fail(MEMCPY, k)
        assert fails(call, c), k
        F.fake_fail(MEMCPY, 0)
        F.hipGetLastError()
        call(c)
        assert F.fake_done(MEMCPY) - n0 >= need, (k, F.fake_done(MEMCPY) - n0, need)
""" % itree)


TRANSFERS = """
def cloud(n):
    return rng.standard_normal((n, 3)), rng.standard_normal((n, 4))
def round_trip(c, n):
    x, q = cloud(n)
    c.upload(x, q)
    xo, qo = c.download()[:2]
    assert np.array_equal(x, xo) and np.array_equal(q, qo), n
LARGE, SMALL = 700000, 500  # 39 MB in chunks, 28 kB through the pinned buffer
"""


def test_transfer_slots_serve_every_context(run):
    """Contexts one after another: the pinned slots and the streams, four at most, of large transfers
    are set up once."""
    run(TRANSFERS + """
for turn in range(4):
    with V.VPM(V.Params.make(0.125)) as c:
        base = F.fake_done(STREAM), F.fake_done(HOSTMALLOC)
        round_trip(c, LARGE)
        new = F.fake_done(STREAM) - base[0], F.fake_done(HOSTMALLOC) - base[1]
        assert (0 < new[0] <= 4 and 0 < new[1] <= 8) if turn == 0 else new == (0, 0), (turn, new)
assert F.fake_held(1) <= 8
""")


@pytest.mark.parametrize("kind", ["HOSTMALLOC", "STREAM", "EVENT"])
def test_transfer_slots_that_cannot_grow(run, kind):
    """A refused allocation while the slots are set up leaves fewer of them, no error behind, and nothing
    allocated twice by the attempts that follow."""
    run(TRANSFERS + """
kind = %s
with V.VPM(V.Params.make(0.125)) as c:
    c.upload(*cloud(SMALL))  # (its buffer is there)
    for k in (1, 2, 3, 2, 1, 4):
        F.fake_fail(kind, k)
        round_trip(c, LARGE)
        assert F.fake_last_error() == 0, k
    F.fake_fail(kind, -1)
    for n in (LARGE, SMALL, LARGE):
        round_trip(c, n)
    assert F.fake_last_error() == 0
    F.fake_fail(kind, 0)
    round_trip(c, LARGE)
assert F.fake_held(1) <= 8, F.fake_held(1)
""" % kind)


def test_transfers_without_pinned_memory(run):
    """No pinned memory at all: every transfer goes through the runtime's own copies, and the evaluation
    after it finds no error."""
    run(TRANSFERS + """
F.fake_fail(HOSTMALLOC, -1)
with V.VPM(V.Params.make(0.125)) as c:
    for n in (SMALL, LARGE, SMALL):
        round_trip(c, n)
        assert F.fake_last_error() == 0, n
    x, q = cloud(SMALL)
    up, gp = np.zeros_like(x), np.zeros_like(x)
    c.vpm(x, q, up, gp, SMALL, 3, 0, 0)
    c.vpm(x, q, up, gp, SMALL, 3, 2, 1)
assert F.fake_held(1) == 0
""")


def test_large_transfers_go_in_chunks(run):
    """Into the device 8 MiB and more, out of it more than 4 MiB; the others are a copy per array."""
    run(TRANSFERS + """
def copies(f, *a):
    was = F.fake_done(ASYNC)
    f(*a)
    return F.fake_done(ASYNC) - was
with V.VPM(V.Params.make(0.125)) as c:
    # 56 bytes a particle go in (24 and 32 in two arrays), 104 come out (24, 32, 24 and 24 in four)
    chunks = lambda n, arrays: sum(-(-n * b // (2 << 20)) for b in arrays)
    for n, large_in, large_out in ((40329, 0, 0), (40330, 0, 1), (70000, 0, 1), (149796, 0, 1), (149797, 1, 1), (300000, 1, 1)):
        assert copies(c.upload, *cloud(n)) == (chunks(n, (24, 32)) if large_in else 2), n
        assert copies(c.download) == (chunks(n, (24, 32, 24, 24)) if large_out else 4), n
""")


def test_results_that_share_memory(run):
    """Two result arrays in one buffer: the later one's values stay, with one copy after the other."""
    run(TRANSFERS + """
P = ctypes.POINTER(ctypes.c_double)
for n in (SMALL, LARGE):
    with V.VPM(V.Params.make(0.125)) as c:
        x, q = cloud(n)
        c.upload(x, q)
        was = F.fake_done(ASYNC)
        buf = np.full(5 * n, 7.0)  # positions from 0, strengths from n
        xp, qp = buf.ctypes.data, buf.ctypes.data + 8 * n
        r = c._lib.vpmx_particles_download(c._h, ctypes.cast(xp, P), ctypes.cast(qp, P), None, None)
        assert r == 0 and F.fake_done(ASYNC) == was + 2
        assert np.array_equal(buf[n:], q.ravel()) and np.array_equal(buf[:n], x.ravel()[:n]), n
""")


def test_every_line_length_has_its_passes(run):
    """Solves with one axis of 1 to 420 points, in both precisions, find kernels for every length that
    the transform plans take (prime factors of m + 1 up to 64)."""
    run("""
def factor(n):
    p = 2
    while n > 1:
        while n % p == 0:
            n //= p
        if n > 1:
            p += 1
    return p
win = lambda nn: np.array([1, 1, 1, *nn], np.int32)
for prec in (0, 1):
    with V.VPM(V.Params.make(0.125)) as c:
        c.set_precision(prec)
        for m in range(1, 421):
            for axis in range(3):
                nn = np.array([9, 10, 11], np.int32)
                nn[axis] = m + 2
                a = np.zeros((nn[2], nn[1], nn[0], 3))
                args = (np.zeros(6), np.full(3, 0.1), nn, 3, win(nn), a)
                if factor(m + 1) > 64:
                    assert fails(c.stage_solve, *args), m
                else:
                    c.stage_solve(*args)
                    c.stage_solve(*args, None, True)
""")


def test_solve_uploads_the_tables_it_reads(run):
    """A first solve uploads, per axis, the eigenvalues and the sine matrix of the products, or the
    twiddles and sines of an FFT line; nothing for a second one."""
    run("""
def uploads(c, nn):
    nn = np.array(nn, np.int32)
    a = np.zeros((nn[2], nn[1], nn[0], 3))
    was = F.fake_done(MEMCPY)
    c.stage_solve(np.zeros(6), np.full(3, 0.1), nn, 3, np.array([1, 1, 1, *nn], np.int32), a, None, True)
    return F.fake_done(MEMCPY) - was
with V.VPM(V.Params.make(0.125)) as c:
    assert uploads(c, (13, 15, 17)) == 6
    assert uploads(c, (13, 15, 17)) == 0
    assert uploads(c, (13, 401, 17)) == 3  # 399 points: eigenvalues, twiddles, sines
    assert uploads(c, (13, 401, 17)) == 0
""")


def test_every_block_length_in_the_mixed_form(run):
    """Evaluations in the mixed form (its inner-box solves return in FP64) of boxes with one axis of up
    to 330 nodes."""
    run("""
h = 0.125
with V.VPM(V.Params.make(h)) as c:
    c.set_precision(1)
    for axis in range(3):
        for cells in range(6, 330, 8):
            ext = np.full(3, 3.0)
            ext[axis] = cells
            x = np.stack([np.zeros(3), ext * h])
            q = np.ones((2, 4))
            up, gp = np.zeros_like(x), np.zeros_like(x)
            c.vpm(x, q, up, gp, 2, 3, 0, 0)
            try:
                c.vpm(x, q, up, gp, 2, 3, 2, 1)
            except V.VpmError as e:
                assert "prime factor" in str(e) or "too long" in str(e), (axis, cells, str(e))
""")


def test_stage_interval_after_the_first_fill(run):
    """The stretching stage of a first mode-4 call begins after the fill of its new velocity grid: an
    event of its own, where later calls (no fill) share the projection's last one."""
    run("""
x, q = np.array([[0.0, 0, 0], [1, 2, 3]]), np.ones((2, 4))
up, gp = np.zeros_like(x), np.zeros_like(x)
with V.VPM(V.Params.make(0.125)) as c:
    c.vpm(x, q, up, gp, 2, 3, 0, 0)
    n = []
    for call in range(3):
        was = F.fake_done(RECORD)
        c.vpm(x, q, up, gp, 2, 3, 4, 1)
        n.append(F.fake_done(RECORD) - was)
assert n[0] == n[1] + 1 and n[1] == n[2], n
""")

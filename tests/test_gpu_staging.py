"""Ice and fields larger than the pinned staging buffer (16 MiB): a batch's
ice, one domain's ice and whole padded fields pass through it piece after piece,
exactly, and no update or read-back allocates pinned memory once the sizes in
use have been seen."""
import ctypes
import threading

import numpy as np
import pytest

from fastisostasy_amd import isostasy as G
from fastisostasy_amd import workloads as W
from fastisostasy_amd._lib import check, load

pytestmark = pytest.mark.gpu


def _pinned():
    n = ctypes.c_longlong()
    check(load().fi_prof_pinned(ctypes.byref(n)))
    return n.value


def _domain(nx, ny, seed=0):
    # no displacement: the update embeds the ice and nothing else moves
    z = np.random.default_rng(seed).uniform(100.0, 900.0, (ny, nx))
    b = G.bsl_init("const", 0.0)
    g = G.isos_init(W.params(min_pad=0.0, method=0), nx, ny, 16e3)
    G.isos_init_state(g, z, np.zeros_like(z), 0.0, b)
    return g, b, z


# MiB of ice per update: below the buffer's size; just above; many times; members that
# the pieces of 4 MiB cut in the middle (7.03 and 3.57 MiB each)
@pytest.mark.parametrize("nx,ny,members", [(512, 512, 7), (1024, 1024, 3), (1024, 1024, 9), (960, 960, 10),
                                           (700, 667, 6)])
def test_batch_ice_beyond_the_buffer(nx, ny, members):
    print(f"case: {members} domains, ice {nx} x {ny}", flush=True)
    rng = np.random.default_rng(nx + members)
    doms = [_domain(nx, ny, m) for m in range(members)]
    bat = G.Batch([d[0] for d in doms])
    made = None
    for k in range(1, 6):
        H = [rng.uniform(0.0, 3000.0, (ny, nx)) for _ in doms]
        bat.update(float(k), [d[1] for d in doms], H)
        for m, (g, _, _) in enumerate(doms):
            assert np.array_equal(g.out("Hice"), H[m]), (k, m)
        made = _pinned() if k == 1 else made
    assert _pinned() == made
    bat.close()


def test_two_batches_in_turn_keep_their_buffers():
    print("case: two batches of 34 and 42 MB of ice in turn", flush=True)
    sets = [[_domain(1024, 1024, m) for m in range(n)] for n in (4, 5)]
    bats = [G.Batch([d[0] for d in s]) for s in sets]
    for k in range(1, 5):
        for s, bat in zip(sets, bats):
            H = [np.full((1024, 1024), 100.0 * k + m) for m in range(len(s))]
            bat.update(float(k), [d[1] for d in s], H)
            assert all(np.array_equal(d[0].out("Hice"), h) for d, h in zip(s, H))
        if k == 1:
            made = _pinned()
    assert _pinned() == made
    for bat in bats:
        bat.close()


# the ice read in place by the first kernel, and in pieces: 15.4, 16.1 and 17.6 MiB
@pytest.mark.parametrize("nx,ny", [(1440, 1400), (1458, 1450), (1536, 1501)])
def test_one_domain_beyond_the_buffer(nx, ny):
    print(f"case: one domain, ice {nx} x {ny}", flush=True)
    n = G.padded_size(nx, ny, 16e3, 16e3, 0.0)
    assert n == nx
    g, b, z = _domain(nx, ny)
    rng = np.random.default_rng(7)
    for k in range(1, 4):
        H = rng.uniform(0.0, 3000.0, (ny, nx))
        G.isos_update(g, H, float(k), b)
        assert np.array_equal(g.out("Hice"), H) and np.array_equal(g.out("z_bed"), z)
        assert np.array_equal(g.out("maskgrounded"), H > 0)
        if k == 1:
            made = _pinned()
    assert _pinned() == made
    full = g.full("z_bed")
    jc = (n - ny + ny % 2) // 2
    assert np.array_equal(full[jc:jc + ny], z)


def test_threads_read_and_update_through_the_pool():
    """Each thread takes buffers of its own: fields of distinct domains read and
    ice of distinct domains brought in at the same time come out whole."""
    print("case: four host threads, 300 x 280 to 900 x 860", flush=True)
    doms = [_domain(nx, ny, nx) for nx, ny in ((300, 280), (512, 480), (640, 600), (900, 860))]
    errors = []

    def work(g, b, z):
        try:
            rng = np.random.default_rng(z.shape[1])
            for k in range(1, 9):
                H = rng.uniform(0.0, 3000.0, z.shape)
                G.isos_update(g, H, float(k), b)
                assert np.array_equal(g.out("Hice"), H) and np.array_equal(g.out("z_bed"), z)
                assert np.array_equal(g.out("maskgrounded"), H > 0)
        except BaseException as e:   # reported by the main thread
            errors.append(e)

    th = [threading.Thread(target=work, args=d) for d in doms]
    for t in th:
        t.start()
    for t in th:
        t.join(timeout=100)
    assert not any(t.is_alive() for t in th)
    assert not errors, errors

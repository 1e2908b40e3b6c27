"""The kernels a group runs are the ones it is meant to run: two-launch attempts
and grouped convolutions at every length they exist for (the comparisons of the
kernels with each other say nothing where both sides ran the same ones), their
concurrent sub-batches, and launch rounds with rejected steps."""
import ctypes

import numpy as np
import pytest

import oracle as O
from fastisostasy_amd import isostasy as G
from fastisostasy_amd import workloads as W
from fastisostasy_amd._lib import check, load
from test_gpu_turn import SHAPE_ENV
from test_gpu_turn import _make as make_domain
from test_gpu_turn import _run as run_domains
from test_lengths import lengths

pytestmark = pytest.mark.gpu

PROF_ALL = 99


def _clear(monkeypatch, **env):
    for k in SHAPE_ENV + ("FI_TURN_LO", "FI_TURN_C"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)


def _profiled(fn):
    """fn()'s result and fi_prof_path after it."""
    check(load().fi_prof_select(PROF_ALL))
    try:
        out = fn()
        path = (ctypes.c_int * 4)()
        check(load().fi_prof_path(path))
        return out, list(path)
    finally:
        check(load().fi_prof_select(-1))


def _update_once(n, prec):
    nx = n - 2 * (n // 8)
    p = W.params(min_pad=(n // 8) * 50e3, include_elastic=1, precision=prec)
    h, b = G.IsosClass(G.make_params(**p), nx, nx, 50e3), G.bsl_init("const", 0.0)
    h.init_state(np.full((nx, nx), 1e3), np.zeros((nx, nx)), 0.0, b)
    assert h.n == n
    h.update(W.disc_load(nx, 50e3), 1.0, b)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_every_length_runs_its_kernels(prec, monkeypatch):
    for n in lengths():
        print(f"case: paths N={n} {prec}", flush=True)
        _clear(monkeypatch)
        assert _profiled(lambda: _update_once(n, prec))[1] == [1, 1, 2, 1], n
        _clear(monkeypatch, FI_TURN="0")
        assert _profiled(lambda: _update_once(n, prec))[1][:3] == [0, 0, 0], n
        _clear(monkeypatch, FI_GENERIC_FFT="1")
        assert _profiled(lambda: _update_once(n, prec))[1] == [0, 0, 0, 0], n


@pytest.mark.parametrize("n,prec,distorted,members", [(486, "fp64", True, 1), (512, "mixed", True, 1),
                                                      (512, "fp64", True, 2), (384, "mixed", True, 3)])
def test_distorted_two_launch_attempts(n, prec, distorted, members, monkeypatch):
    """Non-uniform spacing beyond N = 320, where the strip's spacings and the
    largest LDS tiles meet: bit for bit the other kernels."""
    print(f"case: distorted N={n} {prec} members={members}", flush=True)
    _clear(monkeypatch, FI_SUBBATCHES="1", FI_TURN="0")
    ref, path = _profiled(lambda: run_domains(n, prec, distorted, members))
    assert path[0] == 0
    _clear(monkeypatch, FI_SUBBATCHES="1", FI_TURN="2")
    got, path = _profiled(lambda: run_domains(n, prec, distorted, members))
    assert path[0] == 1 and path[1] == 2
    for r, g in zip(ref, got):
        assert r["attempts"] == g["attempts"] > g["accepts"] == r["accepts"]
        for f in ("w", "dwdt", "z_bed"):
            assert np.array_equal(r[f], g[f]), f


# a general length, small groups at 2^k and 3 * 2^k, and one at the widest blocks
@pytest.mark.parametrize("n,prec,members", [(100, "mixed", 32), (64, "fp64", 6), (192, "mixed", 7), (500, "mixed", 4)])
def test_sub_batches_of_two_launch_attempts(n, prec, members, monkeypatch):
    """Concurrent sub-batches give the bits of one launch, over several updates
    with rejected steps and second rounds."""
    def run(k):
        _clear(monkeypatch, FI_SUBBATCHES=str(k))
        doms = [make_domain(n, prec, False, m) for m in range(members)]
        bat = G.Batch([d[0] for d in doms])
        for j, t in enumerate((2.0, 4.5, 4.6, 7.0)):
            bat.update(t, [d[1] for d in doms], [(1.0 + 0.5 * (j % 2)) * d[2] for d in doms])
        bat.close()
        return [([h.full(f) for f in ("w", "dwdt", "z_bed")], h.scalar("attempts"), h.scalar("accepts"))
                for h, _, _ in doms]

    print(f"case: sub-batches N={n} {prec} members={members}", flush=True)
    one, path = _profiled(lambda: run(1))
    assert path[0] == 1
    assert any(a > c for _, a, c in one)
    for k in (2, 3):
        got, path = _profiled(lambda: run(k))
        assert path[0] == 1
        for (f0, a0, c0), (f1, a1, c1) in zip(one, got):
            assert a0 == a1 and c0 == c1
            assert all(np.array_equal(x, y) for x, y in zip(f0, f1))


def test_split_that_depends_on_the_attempts_ahead(monkeypatch):
    """A double-precision group off 2^k of 1.6 million cells splits where the
    round is long and not where it is short: same bits as never split."""
    def run(env):
        _clear(monkeypatch, **env)
        doms = [make_domain(448, "fp64", False, m) for m in range(8)]
        bat = G.Batch([d[0] for d in doms])
        H = [d[2] for d in doms]
        # about 5, 80 and again 5 attempts
        for t in (0.5, 0.7, 0.9, 8.9, 16.9, 17.1, 17.3):
            bat.update(t, [d[1] for d in doms], H)
        bat.close()
        return [([h.full(f) for f in ("w", "dwdt")], h.scalar("attempts")) for h, _, _ in doms]

    print("case: 8 of 448^2 fp64, the built-in split and one launch", flush=True)
    for (f0, a0), (f1, a1) in zip(run({}), run({"FI_SUBBATCHES": "1"})):
        assert a0 == a1 > 80
        assert all(np.array_equal(x, y) for x, y in zip(f0, f1))


def test_sub_batches_have_their_own_limit(monkeypatch):
    """At FP64 384^2 one block of the two-launch attempts fills a CU's LDS: eight
    domains take them alone, not beside another sub-batch of eight."""
    def run(members):
        doms = [make_domain(384, "fp64", False, m) for m in range(members)]
        bat = G.Batch([d[0] for d in doms])
        for t in (0.5, 8.5):   # (the second update launches more than sixteen attempts ahead)
            bat.update(t, [d[1] for d in doms], [d[2] for d in doms])
        bat.close()

    print("case: 8 and 16 of 384^2 fp64", flush=True)
    _clear(monkeypatch)
    assert _profiled(lambda: run(8))[1][0] == 1
    assert _profiled(lambda: run(16))[1][0] == 0
    _clear(monkeypatch, FI_SUBBATCHES="2")
    assert _profiled(lambda: run(10))[1][0] == 1


@pytest.mark.parametrize("method", [1, 2])
def test_relaxation_rounds_with_rejected_steps(method, monkeypatch):
    """One-launch relaxation attempts over more than one launch round per
    update, with rejected steps, against the oracle's stepping."""
    _clear(monkeypatch)
    print(f"case: relaxation rounds, method {method}", flush=True)
    nx, dx = 32, 100e3
    par = dict(W.relax_disc(method)["params"], min_pad=800e3, rtol=1e-4, atol=1e-2, dt_init=40.0, dt_max=1e3)
    z, H = np.full((nx, nx), 1e6), W.disc_load(nx, dx)
    o, ob = O.OracleIsos(O.make_params(**par), nx, nx, dx), O.OracleBSL("const", 0.0)
    o.init_state(z, np.zeros_like(H), 0.0, ob)
    g, b = G.IsosClass(G.make_params(**par), nx, nx, dx), G.bsl_init("const", 0.0)
    g.init_state(z, np.zeros_like(H), 0.0, b)
    for k, scale in enumerate((1.0, 3.0, 0.5, 2.0)):
        t, before = 400.0 * (k + 1), g.scalar("attempts")
        o.update(scale * H, t, ob)
        g.update(scale * H, t, b)
        for s in ("attempts", "accepts", "t"):
            assert g.scalar(s) == o.scalar(s), (k, s)
        # (a first round never launches more than nine on the word of dt_init)
        assert k > 0 or g.scalar("attempts") - before > 9
        a = o.get_full("w")
        assert np.abs(g.full("w") - a).max() <= 1e-8 * max(1.0, np.abs(a).max() / 100)
    assert g.scalar("attempts") > g.scalar("accepts")

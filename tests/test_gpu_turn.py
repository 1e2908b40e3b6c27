"""Two-launch attempts (column pass; inverse rows, stencil and forward rows in
one kernel) against the other attempt kernels, bit for bit: every kind of
length (one to four exchange groups, line pairs that the blocks divide or not,
blocks wider than the domain, the register kernels' lengths), uniform and
distorted grids, both precisions, one domain and a batch, with rejected steps."""
import numpy as np
import pytest

from fastisostasy_amd import isostasy as G
from fastisostasy_amd import workloads as W

pytestmark = pytest.mark.gpu

SHAPE_ENV = ("FI_SROW_ROWS", "FI_INV_THREADS", "FI_COL_LINES", "FI_ROW_THREADS", "FI_GENERIC_FFT", "FI_GEN_LINES",
             "FI_NO_FUSED_STENCIL", "FI_ROW_TILES", "FI_TURN", "FI_SUBBATCHES")


def _make(n, prec, distorted, m):
    wl = W.ensemble_member(m, nx=n, seed=300 + m)
    # tight tolerances and a long first step: the first attempts are rejected
    p = dict(wl["params"], atol=1e-3, rtol=1e-5, dt_init=2.0)
    K = None
    if distorted:
        x = W.padded_coords(n, wl["dx"])
        K = 0.97 + 0.05 * (x[None, :] ** 2 + x[:, None] ** 2) / (x ** 2).max()
    h = G.IsosClass(G.make_params(precision=prec, **p), n, n, wl["dx"], K=K, he_field=wl["he_field"],
                    eta_field=wl["eta_field"])
    b = G.bsl_init("const", 0.0)
    h.init_state(wl["z_bed"], np.zeros_like(wl["H_ice"]), 0.0, b)
    return h, b, wl["H_ice"]


def _run(n, prec, distorted, members):
    doms = [_make(n, prec, distorted, m) for m in range(members)]
    if members == 1:
        h, b, H = doms[0]
        for t in (2.0, 4.5):
            h.update(H, t, b)
    else:
        bat = G.Batch([d[0] for d in doms])
        for t in (2.0, 4.5):
            bat.update(t, [d[1] for d in doms], [d[2] for d in doms])
        bat.close()
    return [dict({f: h.full(f) for f in ("w", "dwdt", "z_bed")}, t=h.scalar("t"), dt=h.scalar("dt"),
                 attempts=h.scalar("attempts"), accepts=h.scalar("accepts")) for h, _, _ in doms]


@pytest.mark.parametrize("n,prec,distorted,members", [
    (48, "fp64", False, 1), (50, "mixed", False, 1), (54, "fp64", True, 1), (64, "fp64", False, 1),
    (96, "mixed", True, 3), (126, "mixed", False, 1), (128, "mixed", True, 2), (162, "fp64", False, 1),
    (192, "mixed", False, 1), (192, "fp64", True, 1), (200, "mixed", False, 40), (240, "fp64", False, 2),
    (250, "mixed", False, 6), (256, "mixed", False, 1), (256, "fp64", True, 1), (320, "mixed", True, 1),
    (384, "mixed", False, 1), (486, "mixed", False, 1), (500, "fp64", False, 1), (512, "fp64", False, 1),
    # the register kernels' lengths in blocks of two line pairs, eight columns pairs
    (64, "fp64", False, 16), (192, "mixed", False, 5), (256, "mixed", False, 4), (384, "fp64", False, 2),
    (512, "mixed", False, 2),
    # the widest column blocks
    (500, "mixed", False, 2)])
def test_turn_bitwise(n, prec, distorted, members, monkeypatch):
    print(f"case: two-launch attempts N={n} {prec} distorted={distorted} members={members}", flush=True)
    for k in SHAPE_ENV:
        monkeypatch.delenv(k, raising=False)
    monkeypatch.setenv("FI_SUBBATCHES", "1")
    monkeypatch.setenv("FI_TURN", "0")
    ref = _run(n, prec, distorted, members)
    monkeypatch.setenv("FI_TURN", "2")
    got = _run(n, prec, distorted, members)
    for r, g in zip(ref, got):
        for k in ("t", "dt", "attempts", "accepts"):
            assert r[k] == g[k], (k, r[k], g[k])
        for f in ("w", "dwdt", "z_bed"):
            assert np.array_equal(r[f], g[f]), (f, np.abs(r[f] - g[f]).max())
    assert np.abs(got[0]["w"]).max() > 0 and got[0]["attempts"] > got[0]["accepts"] > 4


@pytest.mark.parametrize("n,prec,distorted", [(50, "mixed", False), (96, "fp64", True), (250, "mixed", True),
                                              (256, "fp64", False), (384, "mixed", False)])
def test_arena_and_descriptor_addresses(n, prec, distorted, monkeypatch):
    """A single domain's launches find its arrays by their offsets from its
    Member; a group's (here of one) by the descriptor's pointers."""
    print(f"case: addresses N={n} {prec} distorted={distorted}", flush=True)
    for k in SHAPE_ENV:
        monkeypatch.delenv(k, raising=False)
    ref = _run(n, prec, distorted, 1)[0]
    h, b, H = _make(n, prec, distorted, 0)
    bat = G.Batch([h])
    for t in (2.0, 4.5):
        bat.update(t, [b], [H])
    bat.close()
    assert h.scalar("t") == ref["t"] and h.scalar("attempts") == ref["attempts"] > 4
    for f in ("w", "dwdt", "z_bed"):
        assert np.array_equal(h.full(f), ref[f]), f

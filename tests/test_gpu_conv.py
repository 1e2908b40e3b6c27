"""The grouped register passes of the elastic and sea-surface convolutions
against the LDS Stockham passes (FI_GENERIC_FFT), at lengths of one to four
exchange groups, with last blocks of spare lines and columns, alone and in a
batch.  FP64 to rounding; FP32 bit for bit where both pair the same rows (2N
not a power of two), else to FP32 rounding of log2(2N) <= 10 stages."""
import numpy as np
import pytest

from fastisostasy_amd import isostasy as G
from fastisostasy_amd import workloads as W

pytestmark = pytest.mark.gpu


def _run(n, prec, members):
    pad = n // 8
    nx = n - 2 * pad
    wl = W.sealevel_cycle(nx=nx, dx=50e3, pad=pad * 50e3)
    p = G.make_params(precision=prec, **wl["params"])
    doms = []
    for m in range(members):
        g, b = G.IsosClass(p, nx, nx, 50e3), G.bsl_init("const", 0.0)
        g.init_state(wl["z_bed"], np.zeros((nx, nx)), 0.0, b)
        doms.append((g, b, (1.0 - 0.1 * m) * wl["H_max"]))
    assert doms[0][0].n == n
    # the first update's fields depend on the load alone, not on the stepping
    if members == 1:
        doms[0][0].update(doms[0][2], 10.0, doms[0][1])
    else:
        bat = G.Batch([d[0] for d in doms])
        bat.update(10.0, [d[1] for d in doms], [d[2] for d in doms])
        bat.close()
    return [{f: g.full(f) for f in ("we", "dz_ss")} for g, _, _ in doms]


@pytest.mark.parametrize("n,members", [(48, 1), (50, 3), (54, 1), (64, 2), (126, 1), (128, 1), (162, 1), (250, 2),
                                       (300, 1), (384, 1), (486, 1), (500, 1), (512, 1)])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_convolution_passes(n, members, prec, monkeypatch):
    print(f"case: convolution N={n} {prec} members={members}", flush=True)
    got = _run(n, prec, members)
    monkeypatch.setenv("FI_GENERIC_FFT", "1")
    ref = _run(n, prec, members)
    for r, g in zip(ref, got):
        for f in ("we", "dz_ss"):
            top, err = np.abs(r[f]).max(), np.abs(r[f] - g[f]).max()
            assert top > 1e-4
            if prec == "fp64":
                assert err <= 1e-13 * top, (f, err, top)
            elif n & (n - 1):
                assert err == 0.0, (f, err, top)
            else:
                assert err <= 10 * 2.0 ** -23 * top, (f, err, top)

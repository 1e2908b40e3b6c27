"""How many attempts the host launches ahead of an update (more than it needs are
idle launches of about 4 us each, fewer cost a second round of about 25 us):
after a jump of the load, and with a first step far too small."""
import ctypes

import numpy as np
import pytest

from fastisostasy_amd import isostasy as G
from fastisostasy_amd import workloads as W
from fastisostasy_amd._lib import check, load

pytestmark = pytest.mark.gpu

PROF_ALL = 99


def _count(kernel):
    ms, cnt = ctypes.c_double(), ctypes.c_longlong()
    check(load().fi_prof_collect_kernel(kernel, ctypes.byref(ms), ctypes.byref(cnt)))
    return cnt.value


def _update(h, H, t, b):
    """Launched attempts, needed attempts and rounds of one update."""
    a0 = h.scalar("attempts")
    check(load().fi_prof_select(PROF_ALL))
    try:
        h.update(H, t, b)
        return _count(2), int(h.scalar("attempts") - a0), _count(0)
    finally:
        check(load().fi_prof_select(-1))


def test_one_expensive_update_does_not_set_the_next_ones(monkeypatch):
    monkeypatch.delenv("FI_TURN", raising=False)   # (kernel 0 then starts each round)
    wl = W.ensemble_member(0)
    H = wl["H_ice"]
    h = G.IsosClass(G.make_params(precision="mixed", **wl["params"]), wl["nx"], wl["nx"], wl["dx"],
                    he_field=wl["he_field"], eta_field=wl["eta_field"])
    b = G.bsl_init("const", 0.0)
    h.init_state(wl["z_bed"], np.zeros_like(H), 0.0, b)
    t = 0.0
    for _ in range(6):
        t += 10.0
        h.update(H, t, b)
    t += 10.0
    jump = _update(h, 12.0 * H, t, b)
    after = []
    for _ in range(8):
        t += 10.0
        after.append(_update(h, 12.0 * H, t, b))
    print(f"jump {jump}, after {after}", flush=True)
    assert all(launched >= needed for launched, needed, _ in after) and jump[1] > 2 * after[-1][1]
    # at most what one saved and one unneeded round cost per update
    wasted = sum(4.0 * (launched - needed) + 25.0 * (rounds - 1) for launched, needed, rounds in after)
    assert wasted <= 50.0 * len(after), after


@pytest.mark.parametrize("dt_init", [1e-3, 1.0])
def test_first_step_far_too_small(dt_init):
    nx, dx = 128, 25e3
    h = G.IsosClass(G.make_params(**W.params(min_pad=1600e3, dt_init=dt_init)), nx, nx, dx)
    b = G.bsl_init("const", 0.0)
    h.init_state(np.full((nx, nx), 1e6), np.zeros((nx, nx)), 0.0, b)
    launched, needed, rounds = _update(h, W.disc_load(nx, dx), 10.0, b)
    print(f"dt_init {dt_init}: launched {launched}, needed {needed}, rounds {rounds}", flush=True)
    # the first round takes at most eight and one for a rejection, later ones follow the step as it is
    assert needed <= launched <= 2 * needed + 9

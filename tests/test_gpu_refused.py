"""A refused batch update leaves the batch as it was: the barystatic objects
of the call are taken by the next one that is accepted."""
import ctypes
import types

import numpy as np
import pytest

from fastisostasy_amd import isostasy as G
from fastisostasy_amd import workloads as W
from fastisostasy_amd._lib import FI_E_ARG, FiError

pytestmark = pytest.mark.gpu


def test_refused_batch_update_keeps_no_sea_level():
    print("case: a batch update refused for its second member's bsl, N = 64", flush=True)
    nx, dx = 48, 50e3
    doms = []
    for _ in range(2):
        h = G.IsosClass(G.make_params(**W.params(min_pad=400e3)), nx, nx, dx)
        b = G.bsl_init("const", 0.0)
        h.init_state(np.full((nx, nx), 500.0), np.zeros((nx, nx)), 0.0, b)
        doms.append((h, b))
    H = [W.disc_load(nx, dx)] * 2
    bat = G.Batch([h for h, _ in doms])
    bat.update(1.0, [b for _, b in doms], H)
    assert doms[0][0].scalar("bsl") == 0.0
    high = G.bsl_init("const", 40.0)
    with pytest.raises(FiError) as e:
        bat.update(2.0, [high, types.SimpleNamespace(h=ctypes.c_void_p())], H)
    assert e.value.code == FI_E_ARG and doms[0][0].scalar("t") == 1.0
    bat.update(2.0, [high, doms[1][1]], H)
    assert doms[0][0].scalar("bsl") == 40.0 and doms[1][0].scalar("bsl") == 0.0
    bat.close()

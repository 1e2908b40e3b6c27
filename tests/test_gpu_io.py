"""Fields crossing the bus through pinned memory: windows of the padded grid in
and out must be exact at every size (ragged grids, several chunks of 512 KiB,
a last chunk of one row), for values and for mask bits."""
import numpy as np
import pytest

from fastisostasy_amd import isostasy as G
from fastisostasy_amd import workloads as W

pytestmark = pytest.mark.gpu


# (nx, ny, pad cells): one row short of / past a chunk at 256 columns (256
# rows of 2 KiB), odd and non-square grids, no padding, the smallest
@pytest.mark.parametrize("nx,ny,pad", [(24, 24, 4), (31, 37, 6), (256, 256, 0), (256, 257, 31), (300, 255, 10),
                                       (511, 340, 0)])
def test_windows_are_exact(nx, ny, pad):
    n = max(nx + nx % 2, ny + ny % 2) + 2 * pad
    assert n == G.padded_size(nx, ny, 50e3, 50e3, pad * 50e3)
    print(f"case: window {nx} x {ny} of N = {n}", flush=True)
    rng = np.random.default_rng(nx * 1000 + ny)
    z = rng.uniform(-900.0, 900.0, (ny, nx))
    H = rng.uniform(0.0, 3000.0, (ny, nx)) * (rng.random((ny, nx)) < 0.7)
    b = G.bsl_init("const", 0.0)
    g = G.isos_init(W.params(min_pad=pad * 50e3, method=0), nx, ny, 50e3)
    G.isos_init_state(g, z, np.zeros_like(z), 0.0, b)
    assert np.array_equal(g.out("z_bed"), z)
    G.isos_update(g, H, 1.0, b)
    assert np.array_equal(g.out("Hice"), H)
    # the whole padded grid: the window embedded in ice-free cells
    full = g.full("z_bed")
    ic, jc = (n - nx + nx % 2) // 2, (n - ny + ny % 2) // 2
    assert full.shape == (n, n)
    assert np.array_equal(full[jc:jc + ny, ic:ic + nx], g.out("z_bed"))
    # flotation by hand (method 0 leaves the bed): bits of one byte per cell
    grounded = (H > 0) & (H - np.maximum(-z, 0.0) * (1028.0 / 910.0) > 0)
    assert np.array_equal(g.out("maskcontinent"), z > 0)
    assert np.array_equal(g.out("maskgrounded"), grounded)
    assert np.array_equal(g.out("maskocean"), ~((z > 0) | grounded))
    # an update without new ice keeps the ice the last one brought
    bat = G.Batch([g])
    bat.update(2.0, [b])
    assert np.array_equal(g.out("Hice"), H)
    bat.update(3.0, [b], [H[::-1].copy()])
    assert np.array_equal(g.out("Hice"), H[::-1])
    bat.close()

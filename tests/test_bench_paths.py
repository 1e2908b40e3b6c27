"""bench.py's account of a group that runs two-launch attempts (CPU only): the
kernels' names and bytes, and the roofline over one attempt."""
import types

import bench


def test_names_of_two_launch_attempts():
    # {N, fp64, fused, fast, ...}, {two-launch, row block, column block, convolution}
    shape = [256, 0, 1, 1, 256, 8, 1, 8, 64, 3, 2]
    assert bench.fast_kernel_names(shape, [1, 2, 2, -1]) == {
        0: "kt_turn<float, 256, 2, true>", 2: "kt_col<float, 256, 2>", 3: "kt_turn<float, 256, 2, true>"}
    general = [320, 1, 1, 0, 160, 4, 0, 0, 0, 3, 1]
    assert bench.fast_kernel_names(general, [1, 1, 8, -1])[2] == "kt_col<double, 320, 8>"
    # the other kernels keep theirs
    assert bench.fast_kernel_names(shape, [0, 0, 0, -1]) == bench.fast_kernel_names(shape)
    assert bench.fast_kernel_names(shape)[3] == "kf_row_inv<float, 256, 64, 1, 3>"


def test_bytes_of_two_launch_attempts():
    # column pass 3 s; the rest: g1, D, 1/(2 eta), canom_full in, g2 out (5 s), x in, x2 out (16)
    assert bench.kernel_bytes_per_cell(2, 4, True, turn=True) == 12
    assert bench.kernel_bytes_per_cell(3, 4, True, turn=True) == 36
    assert bench.kernel_bytes_per_cell(3, 8, True, turn=True) == 56
    assert bench.kernel_bytes_per_cell(0, 4, True, turn=True) == 24   # the launch that begins a round
    cells = 8 * 256 * 256
    r = bench.step_roofline(cells, 50.0, 1.0, turn=True)
    assert r["bytes_per_cell"]["attempt"] == 48
    assert r["bytes_per_step"] == cells * (230 + 48 * 50)


def test_roofline_of_two_launch_attempts(monkeypatch):
    monkeypatch.setattr(bench, "copy_bandwidth", lambda: 5150.0)
    cells = 8 * 256 * 256
    names = bench.fast_kernel_names([256, 0, 1, 1, 256, 8, 1, 8, 64, 3, 2], [1, 2, 2, -1])
    # 50 attempts in each of 10 rounds: 5.6 and 8.4 us, 6.0 us for the first launch of a round
    prof = {0: (10 * 6.0e-3, 10), 2: (500 * 5.6e-3, 500), 3: (500 * 8.4e-3, 500), "fused": True, "turn": True,
            "names": names}
    r = bench.roofline({"prof": prof}, types.SimpleNamespace(), cells, 256)
    assert r["kernel"] == "kt_turn" and r["template"] == names[3] and r["bytes_per_launch"] == 36 * cells
    assert [k["kernel"] for k in r["kernels"]] == ["kt_col", "kt_turn"]
    assert r["fft_passes"]["bytes_per_attempt"] == 48 * cells
    assert abs(r["fft_passes"]["us_per_attempt"] - 14.0) < 1e-9

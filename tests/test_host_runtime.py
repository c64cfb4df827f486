"""The host code of the library without a GPU: over a stand-in of the HIP
runtime (tests/cpp/fake_hip.cc) that logs the launches and runs none, each
scenario in a process of its own."""
import os
import subprocess
import sys

import pytest

import host_runtime


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("fake_hip") / "libamdhip64.so.7")
    host_runtime.build(path)
    return path


def _run(fake, scenario, *args):
    code = (f"import sys; sys.path.insert(0, {os.path.dirname(__file__)!r})\n"
            "import test_host_runtime as t, host_runtime as h\n"
            f"t.{scenario}(h.FakeHip({fake!r}), *{args!r})\nprint('scenario ok')\n")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "scenario ok" in r.stdout, r.stdout + r.stderr




def failed_launch(hip, kernel, call):
    """A launch that fails inside a call: the call reports it and waits for
    what it has queued; the next call clears the accumulators before any
    kernel counts into them; the one after it clears nothing."""
    import numpy as np
    from phaser_amd.capi import Context, PhaserError
    cloud = np.ones((40, 4), np.float32)

    def go(ctx):
        if call == "register":
            ctx.register(cloud, cloud)
        elif call == "graph":
            ctx.set_graphs(True)
            ctx.register(cloud, cloud)
        elif call == "pairs":
            ctx.register_pairs([cloud, cloud], [cloud, cloud])
        elif call == "device":
            a = [ctx.device_array(cloud) for _ in range(2)]
            ctx.register_pairs_device([a[0].ptr], [40], [a[1].ptr], [40])
        elif call == "sample":
            ctx.sample_s2(cloud)
        elif call == "voxelize":
            ctx.voxelize(cloud)
        else:
            ctx.spatial_correlate(np.ones((2, 8 ** 3)), np.ones((2, 8 ** 3)))

    def counts(log):
        return host_runtime.launches(log, "k_project", "k_voxel_scatter", "k_spat_r2c", "graph")

    with Context(bandwidth=8, n_voxels=8, max_points=64, max_batch=2, channels=4) as ctx:
        hip.reset()
        go(ctx)
        usual = hip.log()
        assert host_runtime.launches(usual, kernel), usual
        hip.reset()
        if call == "graph":
            ctx.set_graphs(False)  # captured before: capture again
        hip.fail(kernel)
        with pytest.raises(PhaserError, match="an error"):
            go(ctx)
        log = hip.log()
        at = [i for i, l in enumerate(log) if l == "failed"]
        assert at and "wait" in log[at[0]:], log
        fills = len(host_runtime.launches(usual, "k_fill_u32"))
        for cleared in (8, 0):  # the accumulators of four channels
            hip.reset()
            go(ctx)
            log = hip.log()
            first = counts(log)[0]
            fill = host_runtime.launches(log, "k_fill_u32")
            assert len(fill) == fills + cleared, log
            assert len([i for i in fill if i < first]) >= cleared, log


@pytest.mark.parametrize("kernel,call", [
    ("k_cell_bands", "register"), ("k_cell_scatter", "register"), ("k_voxel_scatter", "register"),
    ("k_trans_pose", "pairs"), ("k_cell_bands", "pairs"), ("k_cell_scatter", "device"),
    ("k_cell_bands", "graph"), ("k_cell_scatter", "sample"), ("k_voxel_scatter", "voxelize"),
    ("k_spat_cross_z", "spatial")])
def test_accumulators_are_cleared_after_a_failed_call(fake, kernel, call):
    _run(fake, "failed_launch", kernel, call)


def zero_tuning(hip, B, N):
    """phz_set_tuning with every field 0, or one set, leaves the others as a new
    context has them; -1 is off."""
    from phaser_amd.capi import Context
    with Context(bandwidth=B, n_voxels=N, max_points=16) as ctx:
        new = ctx.tuning()
        ctx.set_tuning()
        assert ctx.tuning() == new
        ctx.set_tuning(nn_lanes=4)
        assert ctx.tuning() == dict(new, nn_lanes=4)
        ctx.set_tuning(fused_reg=-1, so3_reg=-1)
        assert ctx.tuning() == dict(new, fused_reg=-1, so3_reg=-1)


@pytest.mark.parametrize("B,N", [(64, 128), (50, 100), (31, 49), (8, 200)])
def test_zero_tuning_fields_are_the_defaults(fake, B, N):
    _run(fake, "zero_tuning", B, N)


def tiles_of_a_call(hip, N, tile, fused):
    """The tiles a caller sets are those of the kernels a call launches, in the
    LDS passes that skip empty rows too (the cross spectrum's kernel has 8 and,
    up to 128 voxels, 16 columns)."""
    import numpy as np
    from phaser_amd.capi import Context
    cloud = np.ones((8, 4), np.float32)
    with Context(bandwidth=8, n_voxels=N, max_points=16) as ctx:
        ctx.set_tuning(fwd_x=tile, fwd_z=tile, fused_reg=fused)
        assert ctx.tuning()["fwd_x"] == tile
        hip.reset()
        ctx.register(cloud, cloud)
        log = hip.log()
    x = [l for l in log if "k_fft_x_occ" in l or "k_fft_colsILin1" in l]
    assert len(x) == 1
    assert (f"k_fft_x_occILi{N}E" if tile == 1 else f"k_fft_colsILin1ELi{tile}E") in x[0], x
    z = [l for l in log if "k_spat_cross" in l]
    assert len(z) == 1 and f"k_spat_cross_zzILi{8 if tile == 8 or N > 128 else 16}E" in z[0], z


@pytest.mark.parametrize("N,tile,fused", [(49, 8, 0), (49, 16, 0), (49, 32, 0), (127, 64, 0),
                                          (201, 16, 0), (100, 1, -1), (100, 8, -1), (200, 1, -1)])
def test_tiles_reach_the_kernels(fake, N, tile, fused):
    _run(fake, "tiles_of_a_call", N, tile, fused)


def tuned(hip, N, pad, costs, want, kernels):
    """phz_autotune under kernels of given costs, from a new context: the fields
    it changes, and the kernels that the next call then launches."""
    import numpy as np
    from phaser_amd.capi import Context
    cloud = np.ones((8, 4), np.float32)
    with Context(bandwidth=8, n_voxels=N, max_points=16, max_batch=3,
                 spatial_zero_padding=pad) as ctx:
        new = ctx.tuning()
        hip.reset()
        for kernel, ms in costs.items():
            hip.cost(kernel, ms)
        t = ctx.autotune(repeats=2)
        timed = {k for k in t if k.startswith("ms_")}
        assert {k: t[k] for k in t if k not in timed and t[k] != new[k]} == want
        assert t["ms_fused"] > 0 and t["ms_fwd_x"] > 0
        ctx.register(cloud, cloud)
        hip.reset()
        ctx.register(cloud, cloud)
        log = hip.log()
        assert len(host_runtime.launches(log, "k_fill_u32")) == 0
        for k in kernels:
            assert host_runtime.launches(log, k), (k, log)


@pytest.mark.parametrize("N,pad,costs,want,kernels", [
    # the plane pass beats the dense LDS passes, and not those of a call
    (100, 0, {"k_spat_plane_fwd": 5.0, "k_spat_r2cI": 9.0, "k_spat_r2c_rows": 0.5}, {},
     ["k_spat_r2c_rows", "k_fft_x_occ"]),
    # so does an LDS tile of a pass that a call does not run alone
    (100, 0, {"k_fft_lines": 9.0, "k_spat_cross_z_reg": 5.0, "k_spat_plane_fwd": 5.0}, {},
     ["k_spat_cross_zz_reg"]),
    # nothing differs by more than the margin
    (128, 0, {"k_spat": 1.0, "k_fft": 1.0, "k_spat_r2c_rows": 0.02, "k_fft_x_occ": 0.02,
                  "k_spat_plane_fwd": 0.95}, {},
     ["k_spat_r2c_rows", "k_spat_inv_plane"]),
    # whole forms that win
    (100, 0, {"k_spat_r2c_rows": 50.0, "k_spat_plane_fwd": 90.0}, {"fused_reg": -1},
     ["k_spat_r2cILb0E", "k_fft_x_occ", "k_spat_cross_zzI"]),
    (49, 0, {"k_spat_r2cI": 5.0, "k_fft_colsILin1E": 5.0}, {"plane_fwd": 1}, ["k_spat_plane_fwd"]),
    # tiles of the passes that a call runs
    (49, 0, {"k_spat_plane_fwd": 90.0, "k_fft_colsILin1ELi16E": 4.0, "k_fft_colsILin1ELi8E": 3.0,
             "k_spat_cross_zzILi16E": 2.0, "k_fft_colsILi1ELi16E": 2.0},
     {"fwd_x": 32, "fwd_z": 8, "inv_x": 8},
     ["k_fft_colsILin1ELi32E", "k_spat_cross_zzILi8E", "k_fft_colsILi1ELi8E"]),
    (200, 0, {"k_fft_linesILi1E": 2.0, "k_fft_colsILi1ELi16E": 1.0}, {"inv_x": 8},
     ["k_fft_colsILi1ELi8E", "k_spat_cross_zz_reg"]),
    (62, 3, {"k_fft_colsILin1ELi16E": 4.0, "k_spat_plane_fwd": 90.0}, {"fwd_x": 8, "fwd_z": 8},
     ["k_fft_colsILin1ELi8E", "k_spat_pad_gather"]),
])
def test_autotune_times_what_a_call_runs(fake, N, pad, costs, want, kernels):
    _run(fake, "tuned", N, pad, costs, want, kernels)


def failed_tuning(hip):
    """A launch that fails leaves the choices as they were and an error, and
    the next call clears the synthetic scan's voxels."""
    import numpy as np
    from phaser_amd.capi import Context, PhaserError
    cloud = np.ones((8, 4), np.float32)
    with Context(bandwidth=8, n_voxels=49, max_points=16) as ctx:
        ctx.set_tuning(fwd_x=32, nn_lanes=2)
        before = ctx.tuning()
        hip.reset()
        hip.fail("k_spat_cross_zz")
        with pytest.raises(PhaserError, match="autotune"):
            ctx.autotune(repeats=2)
        assert ctx.tuning() == before
        hip.reset()
        ctx.register(cloud, cloud)
        assert len(host_runtime.launches(hip.log(), "k_fill_u32")) == 6


def test_failed_autotune(fake):
    _run(fake, "failed_tuning")

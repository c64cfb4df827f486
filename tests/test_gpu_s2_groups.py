"""The S2 transform's grouping (k_phi_dft, k_legendre): one, two or four rows and
one or two signals to a workgroup, by the number of samples (2^18), rows (8192)
and sums (4096) of a launch.

The last groups partly filled (an odd number of signals at bandwidth 31: rows
two more than a multiple of four), bandwidths of one to three waves.  A
coefficient's sums run in one order whatever its group, so each pair of a batch
equals the pair alone bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cloud(seed, n=1500):
    rng = np.random.default_rng(seed)
    c = rng.normal(0.0, 14.0, (n, 4)).astype(np.float32)
    c[:, 2] *= 0.3
    c[:, 3] = rng.uniform(1.0, 100.0, n)
    return c


# signals on both sides of 2^18 samples (4 B^2 each), the smallest and the
# largest bandwidth
@pytest.mark.parametrize("bw,signals", [(2, 1), (2, 16), (31, 3), (64, 15), (64, 16), (75, 11),
                                        (75, 12), (160, 2), (160, 3), (160, 16)])
def test_grouped_coefficients_equal_single(po, bw, signals):
    """Each signal alone (one row to a workgroup up to bandwidth 160: 102400
    samples) bit for bit, and the transform in 64 bits: sums of at most 320
    terms in FP32 twice, 320 x 6e-8 of the norm at the worst."""
    from phaser_amd.capi import Context
    rng = np.random.default_rng(bw + signals)
    g = rng.uniform(0.0, 60.0, (signals, 4 * bw * bw)).astype(np.float32)
    with Context(bandwidth=bw, n_voxels=8, max_points=16) as ctx:
        got = ctx.s2_transform(g)
        for k in {0, signals // 2, signals - 1}:
            np.testing.assert_array_equal(ctx.s2_transform(g[k:k + 1])[0], got[k])
    want = po.fst(bw, g[-1].astype(np.float64))
    err = np.linalg.norm(got[-1] - want) / np.linalg.norm(want)
    print(f"bandwidth {bw}, {signals} signals: {err:.2e}", flush=True)
    assert err < 2e-5


# (bandwidth, method, sources): one signal per cloud (method 1) or two
@pytest.mark.parametrize("bw,method,sources", [(31, 1, 132), (32, 0, 65), (64, 0, 32),
                                               (129, 1, 32)])
def test_shared_target_batch_equals_single(bw, method, sources):
    """The rotation grid, which every coefficient enters, bit for bit."""
    from phaser_amd.capi import Context
    target, clouds = _cloud(1), [_cloud(i + 2) for i in range(sources)]
    n3 = (2 * bw) ** 3
    with Context(bandwidth=bw, n_voxels=8, max_points=1500, max_batch=sources,
                 method=method) as ctx:
        t, d = ctx.device_array(target), [ctx.device_array(c) for c in clouds]
        all_grids, grid = ctx.device_empty(sources * n3 * 4), ctx.device_empty(n3 * 4)
        batch = ctx.register_pairs_device([t.ptr], [len(target)], [c.ptr for c in d],
                                          [len(c) for c in clouds], shared_target=True,
                                          d_rot=all_grids.ptr)
        base = all_grids.ptr
        for k in [*range(0, sources, sources // 4), sources - 1]:
            a = ctx.register_pairs_device([t.ptr], [len(target)], [d[k].ptr], [len(clouds[k])],
                                          shared_target=True, d_rot=grid.ptr)[0]
            assert a["rot_index"] == batch[k]["rot_index"]
            assert a["rot_value"] == batch[k]["rot_value"]
            all_grids.ptr = base + k * n3 * 4  # the batch's grid k
            np.testing.assert_array_equal(grid.download((n3,), np.float32),
                                          all_grids.download((n3,), np.float32))
        all_grids.ptr = base
        for b in [t, grid, all_grids] + d:
            b.free()

"""The LDS transforms at lengths the register engine lacks: large primes, prime
squares, two primes above 5, odd smooth lengths, the longest ones; alone
against numpy in 64 bits, and the occupancy-skipping passes and the fused cross
spectrum built on them against the dense passes.

A line of length L is summed in at most log2 L radix stages or (L - 1) / 2 terms
of a prime stage: about 6e-8 sqrt(L / 2) of its norm at the worst, below 1e-6
for L <= 256 after the three passes each way, which mostly add in quadrature.
"""
import numpy as np
import pytest

from test_gpu_reg_lengths import _cloud, _rel_without_ties

pytestmark = pytest.mark.gpu

LENGTHS = [49, 62, 75, 77, 101, 121, 127, 129, 134, 169, 201, 254]


@pytest.mark.parametrize("N", LENGTHS)
def test_single_channel_against_numpy(N):
    from phaser_amd.capi import Context
    rng = np.random.default_rng(N)
    f = np.where(rng.random((N, N, N)) < 0.05, rng.uniform(1, 60, (N, N, N)), 0).astype(np.float32)
    g = np.roll(f, (3, 5, 7), axis=(0, 1, 2))
    with Context(bandwidth=8, n_voxels=8, max_points=16) as ctx:
        corr, arg = ctx.spatial_correlate_single(f, g, N)
    F, G = np.fft.rfftn(f.astype(np.float64)), np.fft.rfftn(g.astype(np.float64))
    want = np.fft.irfftn(F * np.conj(G), s=f.shape, axes=(0, 1, 2)).reshape(-1) * N ** 3
    err = np.linalg.norm(corr - want) / np.linalg.norm(want)
    print(f"N {N}: {err:.2e}", flush=True)
    assert err < 1e-6
    assert arg == int(want.argmax())


@pytest.mark.parametrize("channels", [2, 4])
@pytest.mark.parametrize("N", LENGTHS)
def test_occupancy_skipping_matches_dense(N, channels):
    """Separate and shared targets; a large pair first, so that the second one
    runs over spectra rows the first left behind, which must not be read."""
    from phaser_amd.capi import Context
    sets = [([_cloud(1), _cloud(2, 3000)], [_cloud(3), _cloud(4, 2500)]),
            ([_cloud(5, 800), _cloud(6, 300)], [_cloud(7, 500), _cloud(8, 200)])]
    got = {}
    with Context(bandwidth=8, n_voxels=N, max_points=6000, max_batch=2, channels=channels) as ctx:
        assert ctx.tuning()["fused_reg"] == -1
        grid = ctx.device_empty(2 * N ** 3 * 4)
        for occ in (1, -1):
            ctx.set_tuning(occ_fwd=occ)
            got[occ] = []
            for tg, sr in sets:
                d = [ctx.device_array(c) for c in tg + sr]
                e = [ctx.device_array(np.stack([c[:, 3] ** 2 / 100, 50 + c[:, 0]], 1)
                                      .astype(np.float32)) for c in tg + sr]
                ra = [a.ptr if channels == 4 else 0 for a in e]
                for shared in (False, True):
                    nt = 1 if shared else 2
                    res = ctx.register_pairs_channels_device(
                        [a.ptr for a in d[:nt]], ra[:nt], [len(c) for c in tg[:nt]],
                        [a.ptr for a in d[2:]], ra[2:], [len(c) for c in sr],
                        shared_target=shared, d_trans=grid.ptr)
                    got[occ].append((res, grid.download((2, N ** 3), np.float32)))
                for a in d + e:
                    a.free()
        grid.free()
    for (ra, ga), (rb, gb) in zip(got[1], got[-1]):
        for k in range(2):
            err, ties = _rel_without_ties(ga[k], gb[k], N)
            print(f"N {N}, {channels} channels, pair {k}: {err:.2e}, {ties} ties", flush=True)
            assert err < 1e-5
            assert ra[k]["trans_index"] == rb[k]["trans_index"]
            assert ra[k]["rot_index"] == rb[k]["rot_index"]


@pytest.mark.parametrize("N,x,z", [(49, 8, 8), (49, 32, 16), (62, 64, 8), (127, 64, 16), (127, 8, 8),
                                   (201, 16, 16), (100, 1, 8), (150, 1, 1), (200, 1, 8)])
def test_occupancy_skipping_tiles(N, x, z):
    """The tiles of the x pass and of the fused cross spectrum, and the register
    engine's x pass between the LDS passes, against the dense passes."""
    from phaser_amd.capi import Context
    tgt, src = _cloud(9), _cloud(10, 2000)
    with Context(bandwidth=8, n_voxels=N, max_points=6000) as ctx:
        ctx.set_tuning(x, z, fused_reg=-1)
        assert ctx.tuning()["fwd_x"] == x
        a = ctx.register(tgt, src, grids=True)
        ctx.set_tuning(8, 8, 8, fused_reg=-1, occ_fwd=-1)
        b = ctx.register(tgt, src, grids=True)
    err, ties = _rel_without_ties(a["trans_corr"], b["trans_corr"], N)
    print(f"N {N}, tiles {x} {z}: {err:.2e}, {ties} ties", flush=True)
    assert err < 1e-5
    assert a["trans_index"] == b["trans_index"]


@pytest.mark.parametrize("B", [31, 37, 49])
def test_rotation_grid_against_oracle(po, B):
    from phaser_amd.capi import Context
    rng = np.random.default_rng(B)
    f = po.fst(B, rng.normal(size=4 * B * B))
    h = po.fst(B, rng.normal(size=4 * B * B))
    mag = np.asarray(po.so3_correlate(B, f, h), np.float64)
    with Context(bandwidth=B, n_voxels=8, max_points=16) as ctx:
        assert ctx.tuning()["so3_reg"] == -1
        corr, am = ctx.so3_correlate_coef(f.astype(np.complex64), h.astype(np.complex64))
    assert np.max(np.abs(corr - mag)) / mag.max() < 2e-4
    assert am == int(mag.argmax())


@pytest.mark.parametrize("channels", [2, 4])
def test_nan_channel_loses_the_fusion(channels):
    """An intensity that is NaN at one point makes the packed intensity and
    range spectra NaN; the fusion passes to a later channel, with two channels
    to the absent ones' zero, in the fused pass as in the separate ones.  At
    two voxels per axis no frequency is a mean of the channels, so that the
    grid stays finite.  The sums of eight voxels differ by their order alone:
    1e-5 of the largest entry."""
    from phaser_amd.capi import Context, PhaserError
    N, tgt, src = 2, _cloud(11), _cloud(12)
    clouds = [tgt, src]
    extra = [np.stack([c[:, 3] ** 2 / 100, 50 + c[:, 0]], 1).astype(np.float32) for c in clouds]
    got = {}
    with Context(bandwidth=4, n_voxels=N, max_points=6000, channels=channels) as ctx:
        for i in range(len(tgt)):  # a point that no grid direction samples
            bad = tgt.copy()
            bad[i, 3] = np.nan
            if np.isfinite(ctx.sample_s2(bad)).all():
                break
        d = [ctx.device_array(bad), ctx.device_array(src)]
        e = [ctx.device_array(x) for x in extra]
        ra = [a.ptr if channels == 4 else 0 for a in e]
        grid = ctx.device_empty(N ** 3 * 4)
        for occ in (1, -1):
            ctx.set_tuning(occ_fwd=occ)
            grid.upload(np.full(N ** 3, 7.0, np.float32))
            try:
                ctx.register_pairs_channels_device([d[0].ptr], ra[:1], [len(bad)], [d[1].ptr],
                                                   ra[1:], [len(src)], d_trans=grid.ptr)
            except PhaserError as err:  # two channels: no positive peak
                print(f"{channels} channels, occ {occ}: {err}", flush=True)
            got[occ] = grid.download((N ** 3,), np.float32)
        for a in d + e + [grid]:
            a.free()
    print(got, flush=True)
    assert np.isfinite(got[-1]).all()
    assert np.abs(got[1] - got[-1]).max() <= 1e-5 * np.abs(got[-1]).max()
    if channels == 2:
        assert not got[-1].any()

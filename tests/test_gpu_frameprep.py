"""K5 frame prep on the GPU: bit-exact against the libswscale restatement."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def inputs(w, h, seed):
    rng = np.random.default_rng(seed)
    a = rng.integers(0, 256, (h, w, 3), dtype=np.uint8)
    b = rng.integers(0, 256, (h, w, 3), dtype=np.uint8)
    da = rng.uniform(0.1, 10.0, (h, w)).astype(np.float32)
    db = rng.uniform(0.1, 10.0, (h, w)).astype(np.float32)
    return a, da, b, db


def assert_planes_equal(got, ref):
    for name, g, r in zip("yuv", got, ref):
        assert g.shape == r.shape
        bad = np.argwhere(g != r)
        assert len(bad) == 0, f"plane {name}: {len(bad)} mismatches, first {bad[:3].tolist()}"


@pytest.mark.parametrize("mode", [0, 1])
def test_two_720p_inputs_composite_bit_exact(nes, oracle, mode):
    a, da, b, db = inputs(1280, 720, 0)
    assert_planes_equal(nes.frameprep(a, da, b, db, mode=mode),
                        oracle.frameprep(a, da, b, db, mode=mode))


@pytest.mark.parametrize("mode", [0, 1])
def test_single_input_conversion_bit_exact(nes, oracle, mode):
    a, _, _, _ = inputs(1280, 720, 1)
    assert_planes_equal(nes.frameprep(a, mode=mode), oracle.rgb24_to_yuv420p(a, mode))


@pytest.mark.parametrize("w,h", [(2, 2), (4, 2), (2, 8), (6, 4), (8, 10), (10, 12), (130, 98),
                                 (258, 66), (640, 480), (1440, 1600), (2064, 2208)])
def test_sizes_bit_exact(nes, oracle, w, h):
    a, da, b, db = inputs(w, h, w * 7 + h)
    for mode in (0, 1):
        assert_planes_equal(nes.frameprep(a, da, b, db, mode=mode),
                            oracle.frameprep(a, da, b, db, mode=mode))


def test_depth_ties_nan_and_extremes(nes, oracle):
    w, h = 96, 64
    rng = np.random.default_rng(5)
    a = np.zeros((h, w, 3), np.uint8)
    b = np.full((h, w, 3), 255, np.uint8)
    levels = np.array([0.0, -0.0, 1.0, np.inf, -np.inf, np.nan, 5.0], np.float32)
    da = levels[rng.integers(0, len(levels), (h, w))]
    db = levels[rng.integers(0, len(levels), (h, w))]
    for mode in (0, 1):
        assert_planes_equal(nes.frameprep(a, da, b, db, mode=mode),
                            oracle.frameprep(a, da, b, db, mode=mode))


def test_gray8_depth_stream_bit_exact(nes, oracle):
    rng = np.random.default_rng(6)
    for w, h in [(1280, 720), (66, 10)]:
        g = rng.integers(0, 256, (h, w), dtype=np.uint8)
        for mode in (0, 1):
            assert_planes_equal(nes.gray8_to_yuv420p(g, mode), oracle.gray8_to_yuv420p(g, mode))


def test_device_batch_bit_exact(nes, oracle):
    w, h, n = 640, 480, 6
    frames = [inputs(w, h, 100 + i) for i in range(n)]
    A = np.stack([f[0] for f in frames]); DA = np.stack([f[1] for f in frames])
    B = np.stack([f[2] for f in frames]); DB = np.stack([f[3] for f in frames])
    bufs = [nes.DeviceBuffer(x.nbytes) for x in (A, DA, B, DB)]
    for buf, x in zip(bufs, (A, DA, B, DB)):
        buf.upload(x)
    Y = nes.DeviceBuffer(n * w * h); U = nes.DeviceBuffer(n * w * h // 4)
    V = nes.DeviceBuffer(n * w * h // 4)
    ms = nes.frameprep_device(*bufs, w, h, n, Y, U, V, mode=0)
    assert ms > 0
    y = Y.download(np.empty((n, h, w), np.uint8))
    u = U.download(np.empty((n, h // 2, w // 2), np.uint8))
    v = V.download(np.empty((n, h // 2, w // 2), np.uint8))
    for i, f in enumerate(frames):
        assert_planes_equal((y[i], u[i], v[i]), oracle.frameprep(*f, mode=0))
    for buf in bufs + [Y, U, V]:
        buf.free()


def _device_planes(nes, bufs, w, h, n, mode, composite, off=0):
    """nes_frameprep_device over raw device inputs `off` bytes into their
    buffers, outputs `off` bytes into theirs; returns the planes."""
    import ctypes as C
    sizes = (n * w * h, n * (w // 2) * (h // 2), n * (w // 2) * (h // 2))
    outs = [nes.DeviceBuffer(s + 64) for s in sizes]
    guard = [np.full(s + 64, 0xA5, np.uint8) for s in sizes]
    for b, g in zip(outs, guard):
        b.upload(g)
    at = lambda b: None if b is None else C.c_void_p(b.ptr.value + off)  # noqa: E731
    a, da, b, db = bufs if composite else (bufs[0], None, None, None)
    nes.check(nes.lib().nes_frameprep_device(at(a), at(da), at(b), at(db), w, h, n, at(outs[0]), w,
                                             at(outs[1]), w // 2, at(outs[2]), w // 2, mode, None),
              "nes_frameprep_device")
    got = []
    for o, g, s in zip(outs, guard, sizes):
        o.download(g)
        assert (g[:off] == 0xA5).all() and (g[off + s:] == 0xA5).all()  # nothing beside the planes
        got.append(g[off:off + s].copy())
        o.free()
    return got


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("w,h,n,off", [
    (2, 2, 3, 0), (2, 40, 1, 0), (4, 24, 1, 0), (6, 12, 2, 0),     # narrow, lowest heights with 8 taps
    (254, 34, 1, 1), (258, 36, 1, 3), (262, 64, 2, 2),             # ragged strips at odd addresses
    (640, 480, 1, 0), (642, 360, 8, 0), (514, 482, 16, 0),         # 4, 8 and 16 chroma rows per tile
    (1282, 722, 21, 0),                                            # more than the Infinity Cache
])
def test_tile_shapes_and_alignments_bit_exact(nes, oracle, w, h, n, off, mode):
    """Every tile height, the last partial strip and tile, widths of 4k + 2 and
    2, addresses of any alignment and batches beyond the caches against the
    CPU restatement (of the first, a middle and the last frame)."""
    rng = np.random.default_rng(w * h + n)
    host = (rng.integers(0, 256, (n, h, w, 3), dtype=np.uint8),
            rng.uniform(0.1, 10.0, (n, h, w)).astype(np.float32),
            rng.integers(0, 256, (n, h, w, 3), dtype=np.uint8),
            rng.uniform(0.1, 10.0, (n, h, w)).astype(np.float32))
    host[1][:, ::7, ::3] = np.nan
    host[3][:, ::5, ::2] = np.nan
    host[1][:, 1::9, 1::4] = np.inf
    host[3][:, 2::6, ::5] = host[1][:, 2::6, ::5]
    bufs = []
    for x in host:
        b = nes.DeviceBuffer(x.nbytes + 64)
        b.upload(np.concatenate([np.zeros(off, np.uint8), x.reshape(-1).view(np.uint8)]))
        bufs.append(b)
    for composite in (True, False):
        y, u, v = _device_planes(nes, bufs, w, h, n, mode, composite, off)
        for i in sorted({0, n // 2, n - 1}):
            ref = (oracle.frameprep(host[0][i], host[1][i], host[2][i], host[3][i], mode=mode) if composite
                   else oracle.frameprep(host[0][i], host[1][i], mode=mode))
            for g, r in zip((y, u, v), ref):
                assert np.array_equal(g.reshape(n, *r.shape)[i], r), (composite, i)
    for b in bufs:
        b.free()


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("w,h", [(2, 2), (4, 4), (6, 10), (254, 12), (258, 36), (1030, 100)])
def test_gray_stream_shapes_bit_exact(nes, oracle, w, h, mode):
    g = np.random.default_rng(w + h).integers(0, 256, (h, w), dtype=np.uint8)
    for a, b in zip(nes.gray8_to_yuv420p(g, mode), oracle.gray8_to_yuv420p(g, mode)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("static", [False, True])
def test_more_tiles_than_one_grid_dimension(nes, oracle, static):
    """16400 frames of 2 x 8192 pixels, 4 chroma rows to a tile: 2^24 + 16384
    workgroups of 256 threads, more than one dimension of a launch takes.
    Every frame equals the oracle's."""
    w, h, n = 2, 8192, 16400
    src = np.random.default_rng(9).integers(0, 256, (3, h, w, 3), dtype=np.uint8)
    ref = [oracle.rgb24_to_yuv420p(x, 0) for x in src]
    which = np.arange(n) % 3
    rgb, sizes = nes.DeviceBuffer(n * h * w * 3), (h * w, h // 2, h // 2)
    out = [nes.DeviceBuffer(n * s) for s in sizes]
    rgb.upload(src[which])
    call = nes.frameprep_device_static if static else nes.frameprep_device
    call(rgb, None, None, None, w, h, n, *out)
    for k, (buf, s) in enumerate(zip(out, sizes)):
        got = buf.download(np.empty((n, s), np.uint8))
        for i in range(3):
            assert (got[which == i] == ref[i][k].reshape(-1)).all(), (k, i)
    for buf in [rgb] + out:
        buf.free()

"""Host-to-device uploads: large contiguous sets go through the staged path
(host threads copying slices through pinned buffers on their own streams),
smaller or padded sets through one copy; every byte must arrive."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ya():
    import yael_amd
    yael_amd.init()
    return yael_amd


@pytest.mark.parametrize("n,d", [(1000, 128), (131072 + 7, 128), (700001, 128), (90001, 200)])
def test_upload_roundtrip(ya, n, d):
    """(131072 + 7) x 128 and 700001 x 128 floats are 64 MB and 358 MB:
    staged, with slices and chunks that do not divide evenly; 90001 x 200
    is padded (row stride 208)."""
    from yael_amd import device
    rng = np.random.default_rng(n + d)
    x = rng.standard_normal((n, d)).astype(np.float32)
    x[-1] = np.arange(d, dtype=np.float32)  # the last row marks the tail
    print("upload n=%d d=%d (%.0f MB)" % (n, d, x.nbytes / 2**20), flush=True)
    V = device.DeviceSet(x)
    back = np.empty_like(x)
    ya.check(ya.lib().yk_download_vectors(back.ctypes.data, V.vec.ptr, n, d), "download")
    V.free()
    assert np.array_equal(back.view(np.uint32), x.view(np.uint32))


@pytest.mark.parametrize("n,d", [(1, 1), (5, 3), (2055, 157), (3, 1000), (409601, 41), (120000, 48)])
def test_copies_roundtrip_and_pad_columns(ya, n, d):
    """Rows spread to and collected from the padded layout (one dense piece,
    and 67 MB in two), and an unpadded set of 23 MB read back in slices: every
    byte comes back and the pad columns are zero."""
    from yael_amd import device
    rng = np.random.default_rng(n + d)
    x = rng.standard_normal((n, d)).astype(np.float32)
    print("copies n=%d d=%d (%.1f MB)" % (n, d, x.nbytes / 2**20), flush=True)
    V = device.DeviceSet(x)
    back = np.empty_like(x)
    ya.check(ya.lib().yk_download_vectors(back.ctypes.data, V.vec.ptr, n, d), "download")
    raw = V.vec.to_host(np.float32, (n, V.ld))
    V.free()
    assert np.array_equal(back, x)
    assert np.array_equal(raw[:, :d], x) and not raw[:, d:].any()


@pytest.mark.parametrize("nbytes", [(4 << 20) - 4, 4 << 20, (4 << 20) + 4, (8 << 20) + 4092,
                                    32 << 20, (32 << 20) + 4, (64 << 20) + 4, (97 << 20) - 4])
@pytest.mark.parametrize("shift", [0, 4])
def test_copies_down_in_pieces(ya, nbytes, shift):
    """From 4 MB on in quarters of up to 8 MB, whose buffers are taken again
    past 64 MB; each piece is shared by two to four threads.  Every byte
    comes, in its place, at any alignment, and none beside it, twice."""
    import ctypes
    from yael_amd import device
    rng = np.random.default_rng(nbytes + shift)
    x = rng.integers(0, 256, nbytes, np.uint8)
    print("down %d bytes, shift %d" % (nbytes, shift), flush=True)
    mem = device.DeviceBuffer(nbytes)
    ya.check(ya.lib().yk_memcpy_h2d(mem.ptr, x.ctypes.data, nbytes), "h2d")
    for fill in (0, 255):
        back = np.full(nbytes + 64, fill, np.uint8)
        ya.check(ya.lib().yk_memcpy_d2h(ctypes.c_void_p(back.ctypes.data + 32 + shift), mem.ptr,
                                        nbytes), "d2h")
        assert np.array_equal(back[32 + shift:32 + shift + nbytes], x)
        assert (back[:32 + shift] == fill).all() and (back[32 + shift + nbytes:] == fill).all()
    mem.free()


@pytest.mark.parametrize("n,d", [(1, 65), (500, 128), (600, 100), (2100, 128), (9001, 128),
                                 (11000, 100), (50000, 128), (180001, 100)])
def test_copies_of_pinned_host_memory(ya, n, d):
    """Host memory from yk_host_alloc, below and above the sizes at which
    pageable memory goes through the landing buffer (256 KB), the staging
    threads (4 and 16 MB) and the dense pieces (64 MB), dense and padded."""
    import ctypes
    from yael_amd import device
    L, vp = ya.lib(), ctypes.c_void_p
    rng = np.random.default_rng(n + d)
    x = rng.standard_normal((n, d)).astype(np.float32)
    p = vp()
    ya.check(L.yk_host_alloc(ctypes.byref(p), 2 * x.nbytes), "host_alloc")
    src, dst = np.frombuffer((ctypes.c_char * (2 * x.nbytes)).from_address(p.value),
                             np.float32).reshape(2, n, d)
    src[:], dst[:] = x, 0
    print("pinned n=%d d=%d (%.1f MB)" % (n, d, x.nbytes / 2**20), flush=True)
    V = device.DeviceSet(shape=(n, d))
    ya.check(L.yk_upload_vectors(V.vec.ptr, src.ctypes.data_as(vp), n, d), "upload")
    ya.check(L.yk_download_vectors(dst.ctypes.data_as(vp), V.vec.ptr, n, d), "download")
    raw = V.vec.to_host(np.float32, (n, V.ld))
    assert np.array_equal(raw[:, :d], x) and not raw[:, d:].any()
    assert np.array_equal(dst, x)
    if V.ld == d:
        dst[:] = 0
        ya.check(L.yk_memcpy_d2h(dst.ctypes.data_as(vp), V.vec.ptr, x.nbytes), "d2h")
        assert np.array_equal(dst, x)
    V.free()
    del src, dst
    ya.check(L.yk_host_free(p), "host_free")

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

"""Large copies between the caller's arrays and the device go through pinned
chunks on a few threads: what goes up comes down, at sizes just below and above
where that starts, whole chunks and not, from several threads at once, and
through pinned arrays, which are copied directly."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F32 = np.float32

def there_and_back(gpu, W, H, seed, wrap=lambda a: a):
    rng = np.random.default_rng(seed)
    b = wrap(rng.random((H, W), F32))
    d = wrap(rng.random((H, W), F32))
    f = wrap(rng.random((H, W, 4), F32))
    with gpu.Simulation(W, H) as s:
        s.upload(b, d, f)
        for _ in range(2):
            out = s.download(velocity=True)
            assert np.array_equal(out["depth"], d) and np.array_equal(out["flux"], f)
            rgba = s.download_reference_layout(0.25)
            assert np.array_equal(rgba["terrain_rgba"][..., 0], b)
            assert np.array_equal(rgba["terrain_rgba"][..., 3], d)
            assert np.array_equal(rgba["flow_rgba"], f)
        s.upload_reference_layout(rgba["terrain_rgba"][::-1].copy(), rgba["flow_rgba"][::-1].copy())
        out = s.download()
        assert np.array_equal(out["depth"], d[::-1]) and np.array_equal(out["flux"], f[::-1])


# flux and planes a row less than 5 MiB (downloads) and 24 MiB (uploads), as much
# and a row more, whole chunks, and sides that divide nothing
@pytest.mark.parametrize("W,H", [(1024, 319), (1024, 320), (1024, 321), (1024, 1280), (1024, 1535),
                                 (1024, 1536), (1024, 1537), (1024, 2048), (1331, 1024),
                                 (1403, 1397)])
def test_large_copies_are_exact(gpu, W, H):
    there_and_back(gpu, W, H, W + H)


def test_copies_from_several_threads(gpu):
    failed = []

    def work(i):
        try:
            there_and_back(gpu, 1300 + 13 * i, 1300 + 7 * i, i)
        except BaseException as e:  # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed


def test_pinned_arrays(gpu):
    hip = C.CDLL("libamdhip64.so.7")  # the runtime libtws.so itself uses
    kept = []

    def pinned(a):
        p = C.c_void_p()
        assert hip.hipHostMalloc(C.byref(p), C.c_size_t(a.nbytes), 0) == 0
        kept.append(p)
        out = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_float)), a.shape)
        out[...] = a
        return out

    try:
        there_and_back(gpu, 1024, 1600, 5, pinned)
    finally:
        for p in kept:
            hip.hipHostFree(p)

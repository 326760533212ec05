"""The application stages' host tables in page-locked memory that earlier work
of the same stream fills: read in stream order (MI355X only)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
D2H = 2   # hipMemcpyDeviceToHost


@pytest.fixture
def pinned(fd):
    """array -> page-locked copy of zeros, and a call that enqueues its filling
    behind some milliseconds of copies"""
    hip = fd.lib()   # its dependencies' symbols resolve through it
    vp = ctypes.c_void_p
    for f, args in (("hipHostMalloc", [ctypes.POINTER(vp), ctypes.c_size_t, ctypes.c_uint]), ("hipHostFree", [vp]),
                    ("hipMemcpyAsync", [vp, vp, ctypes.c_size_t, ctypes.c_int, vp])):
        getattr(hip, f).argtypes, getattr(hip, f).restype = args, ctypes.c_int
    big = [fd.DeviceBuffer(256 << 20) for _ in range(2)]
    keep = []

    def make(values):
        values = np.ascontiguousarray(values)
        p = vp()
        assert hip.hipHostMalloc(ctypes.byref(p), values.nbytes, 0) == 0
        keep.append(p)
        a = np.frombuffer((ctypes.c_char * values.nbytes).from_address(p.value), values.dtype).reshape(values.shape)
        a[...] = 0
        src = fd.DeviceBuffer.from_array(values)
        keep.append(src)

        def fill(stream):
            for _ in range(40):
                assert hip.fd_memcpy_dtod(vp(big[0].ptr), vp(big[1].ptr), big[0].nbytes, vp(stream.handle)) == 0
            assert hip.hipMemcpyAsync(p, vp(src.ptr), values.nbytes, D2H, vp(stream.handle)) == 0
        return a, fill

    yield make
    assert hip.fd_device_sync() == 0
    for k in keep:
        if isinstance(k, vp):
            assert hip.hipHostFree(k) == 0


def test_shade_samples_in_stream_order(fd, wl, pinned):
    w, h = 61, 37
    r = np.random.default_rng(2)
    sc = wl.gbuffer_scene_boxes(w, h, 6, 4)
    g = [fd.DeviceBuffer.from_array(np.ascontiguousarray(x, np.float32)) for x in wl.gbuffer_boxes_host(sc)]
    shadow = fd.DeviceBuffer.from_array(r.uniform(0, 1, w * h).astype(np.float32))
    samples = np.array([[0.5, -0.5, 6.0], [-0.3, 0.7, 5.0]], np.float32)
    table, fill = pinned(samples)
    out = []
    for tab in (samples, table):
        rgba = fd.DeviceBuffer(w * h * 16)
        strm = fd.Stream()
        if tab is table:
            fill(strm)
        fd.shade(w, h, tab, sc.eye, (0.2, 0.2, 0.2), (0.9, 0.9, 0.8), (0.5, 0.5, 0.5), shadow, *g, rgba, stream=strm)
        strm.sync()
        strm.close()
        out.append(rgba.download(np.uint32))
    assert np.array_equal(table, samples) and np.array_equal(out[0], out[1])


@pytest.mark.parametrize("which", ["boxes", "materials"])
def test_gbuffer_tables_in_stream_order(fd, wl, pinned, which):
    w, h = 131, 77
    sc = wl.gbuffer_scene_boxes(w, h, 12, 9)
    tables = dict(boxes=np.ascontiguousarray(sc.boxes, np.float64), materials=np.ascontiguousarray(sc.materials, np.float32))
    table, fill = pinned(tables[which])
    out = []
    for filled in (False, True):
        t = dict(tables, **({which: table} if filled else {}))
        g = [fd.DeviceBuffer(w * h * 16) for _ in range(4)]
        strm = fd.Stream()
        if filled:
            fill(strm)
        fd.gbuffer_boxes(w, h, t["boxes"], t["materials"], sc.eye, sc.at, sc.up, sc.fovy_deg, sc.ground_half, *g, stream=strm)
        strm.sync()
        strm.close()
        out.append([x.download(np.uint32) for x in g])
    assert np.array_equal(table, tables[which])
    assert all(np.array_equal(a, b) for a, b in zip(*out))

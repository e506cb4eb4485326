"""infer_f32's device conversions: the canvas region it writes and the floats it returns, bit for
bit against the host rounding rules, on every layout and at the values where rounding can go
wrong (ties, subnormals, overflow, NaN payloads)."""
import contextlib
import ctypes
import threading

import numpy as np
import pytest

from oracle import cnn_oracle as co
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _floats(rng, n):
    """Random floats, with every kind of special value among them."""
    x = rng.standard_normal(n).astype(np.float32) * np.float32(10.0) ** rng.integers(-9, 6, n)
    bits = np.array([0x00000000, 0x80000000, 0x7f800000, 0xff800000, 0x7f800001, 0x7fc00000,
                     0xffffe000, 0x7f802000, 0x33000000, 0x33000001, 0x32ffffff, 0x387fe000,
                     0x387ff000, 0x38801000, 0x477fefff, 0x477ff000, 0x3f801000, 0x3f803000,
                     0x00000001, 0xb3800000], np.uint32).view(np.float32)
    x = x.astype(np.float32)
    k = min(n, bits.size)
    x[rng.permutation(n)[:k]] = bits[:k]
    return x


def _half_bits(x):
    """The oracle's rounding (its scalar form for the NaNs, whose payload numpy treats its own way)."""
    x = np.ascontiguousarray(x, np.float32)
    with np.errstate(over="ignore"):
        h = x.astype(np.float16).view(np.uint16)
    for i in np.flatnonzero(np.isnan(x)):
        h[i] = orc.f32bits_to_f16(int(x.view(np.uint32)[i]))
    return h


def _widened(h):
    """fp32 bits of fp16 bits (exact; NaN payloads shifted, not quieted)."""
    h = np.ascontiguousarray(h, np.uint16)
    f = h.view(np.float16).astype(np.float32).view(np.uint32)
    nan = (h & 0x7c00) == 0x7c00
    f[nan] = ((h[nan].astype(np.uint32) & 0x8000) << 16) | 0x7f800000 | \
        ((h[nan].astype(np.uint32) & 0x3ff) << 13)
    return f


@pytest.mark.parametrize("C,W,extra", [(5, 1, 0), (3, 200, 0), (70000, 3, 0), (4, 64, 37)])
def test_token_rows(wavec, C, W, extra):
    """1-D inputs (ragged rows, more channels than a grid dimension holds, a short input)."""
    rng = np.random.default_rng(C + W)
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", C, 1, W, is_1d=True)
    g.add_swiglu("m", "x", "x", "y")
    g.set_output("y")
    plan = g.compile()
    plan.init_gpu()
    stride = (W + 63) // 64 * 64
    plan.write_canvas(0, np.full(C * stride, 7.0, np.float16))  # stale data of an earlier run
    n = C * W - extra
    x = _floats(rng, n)
    y = np.full((C, 1, W), -1.0, np.float32)
    ms = ctypes.c_float(0)
    fp = ctypes.POINTER(ctypes.c_float)
    assert plan._lib.wavec_gpu_infer_f32(plan._handle, x.ctypes.data_as(fp), n,
                                         y.ctypes.data_as(fp), y.size - extra,
                                         ctypes.byref(ms)) == 0
    full = np.zeros(C * W, np.float32)
    full[:n] = x
    want = np.zeros((C, stride), np.uint16)
    want[:, :W] = _half_bits(full).reshape(C, W)
    assert np.array_equal(plan.read_canvas(0, C * stride).reshape(C, stride), want)
    off = int(plan.cmds[-1]["y_off"])
    out = plan.read_canvas(off, C * stride).reshape(C, stride)[:, :W].reshape(-1)
    ref = _widened(out)
    got = y.reshape(-1)
    assert np.array_equal(got[:n].view(np.uint32), ref[:n])
    assert np.all(got[n:] == -1.0)  # elements past out_elems are not touched


@pytest.mark.parametrize("H,W,frames", [(6, 64, 1), (7, 20, 1), (5, 30, 3), (4, 6, 64), (600, 700, 1)])
def test_image_planes(wavec, H, W, frames):
    """Padded planes (aligned and masked widths, several frames, 64 interleaved frames) and an
    output of several transfer chunks."""
    rng = np.random.default_rng(H * W)
    C = 3
    g = wavec.WaveGraph(kv_cache_max_seq=0, batch_size=frames)
    g.add_input("img", C, H, W)
    g.add_maxpool("p", "img", "y", kernel_size=5, stride=1, pad=2)
    g.set_output("y")
    plan = g.compile()
    plan.init_gpu()
    lay = co.Layout2D(H, W, frames, tok64=frames >= 64)
    src = int(plan.cmds[0]["src_off"])
    plan.write_canvas(src, np.full(C * lay.channel_stride, 3.0, np.float16))
    x = _floats(rng, C * H * W).reshape(C, H, W)
    x[np.isnan(x)] = 0.5  # (the pool's treatment of NaN is not what is tested here)
    y, _ = plan.infer_f32(x)
    want = np.zeros(C * lay.channel_stride, np.uint16)
    want[lay.offsets(C)[0].ravel()] = _half_bits(x.ravel())
    assert np.array_equal(plan.read_canvas(src, want.size), want)
    out = plan.read_canvas(int(plan.cmds[-1]["y_off"]), C * lay.channel_stride)
    ref = _widened(out[lay.offsets(C)[0].ravel()])
    got = np.ascontiguousarray(y.reshape(frames, C, H, W)[0]).reshape(-1)
    assert np.array_equal(got.view(np.uint32), ref)


def test_token_rows_with_height(wavec):
    """A token input declared with several rows per channel keeps the last one given."""
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", 16, 3, 10, is_1d=True)
    g.add_linear("l", "x", "y", 16, 16, np.eye(16, dtype=np.float32))
    g.set_output("y")
    plan = g.compile()
    x = np.arange(16 * 3 * 10, dtype=np.float32).reshape(16, 3, 10)
    y, _ = plan.infer_f32(x)
    assert np.array_equal(y[:, 0], x[:, 2])


def _hip():
    """The HIP runtime this process already uses."""
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    return ctypes.CDLL(path)


@pytest.mark.parametrize("pinned,shift", [(False, 0), (True, 0), (True, 1)])
@pytest.mark.parametrize("rows,stride,cols,off", [
    (1, 5, 5, 0), (37, 64, 9, 3), (700, 128, 128, 8), (900, 1024, 1000, 64), (2000, 640, 577, 1)])
def test_canvas_reads(wavec, pinned, shift, rows, stride, cols, off):
    """read_canvas_2d into pageable memory (one and several transfer chunks) and into page-locked
    memory written in place, aligned and not; nothing past the destination is touched."""
    rng = np.random.default_rng(rows)
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", 2100, 1, 1024, is_1d=True)
    g.add_swiglu("m", "x", "x", "y")
    plan = g.compile()
    plan.init_gpu()
    data = rng.integers(0, 65536, off + rows * stride + 8, dtype=np.uint16)
    plan.write_canvas(0, data)
    want = np.lib.stride_tricks.as_strided(data[off:], (rows, cols), (2 * stride, 2)).reshape(-1)
    if not pinned:
        assert np.array_equal(plan.read_canvas_2d(off, rows, stride, cols).reshape(-1), want)
        assert np.array_equal(plan.read_canvas(off, rows * stride), data[off:off + rows * stride])
        return
    hip, p = _hip(), ctypes.c_void_p()
    n = rows * cols + 16
    assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(2 * n), 0) == 0
    buf = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_uint16)), (n,))
    buf[:] = 0xabcd
    try:
        dst = ctypes.cast(p.value + 2 * shift, ctypes.POINTER(ctypes.c_uint16))
        assert plan._lib.wavec_gpu_read_canvas_2d(plan._handle, off, rows, stride, cols, dst) == 0
        assert np.array_equal(buf[shift:shift + rows * cols], want)
        assert np.all(buf[:shift] == 0xabcd) and np.all(buf[shift + rows * cols:] == 0xabcd)
    finally:
        del buf
        hip.hipHostFree(p)


def _read_2d(plan, addr, off, rows, stride, cols):
    assert plan._lib.wavec_gpu_read_canvas_2d(plan._handle, off, rows, stride, cols,
                                              ctypes.cast(addr, ctypes.POINTER(ctypes.c_uint16))) == 0


def _filled_plan(wavec, channels=2100):
    """A plan whose first rows hold known words: (plan, words [channels * 1024])."""
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", channels, 1, 1024, is_1d=True)
    g.add_swiglu("m", "x", "x", "y")
    plan = g.compile()
    plan.init_gpu()
    data = np.random.default_rng(channels).integers(0, 65536, channels * 1024, dtype=np.uint16)
    plan.write_canvas(0, data)
    return plan, data


@pytest.mark.parametrize("rows,stride,cols,shift", [(1, 5, 5, 0), (40, 64, 64, 8), (900, 1024, 1000, 1)])
def test_reads_into_device_memory(wavec, rows, stride, cols, shift):
    """A destination on the GPU (as a copy takes it), up to several transfer chunks."""
    plan, data = _filled_plan(wavec)
    want = np.lib.stride_tricks.as_strided(data, (rows, cols), (2 * stride, 2)).reshape(-1)
    n = shift + want.size + 8
    hip, d = _hip(), ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(d), ctypes.c_size_t(2 * n)) == 0
    try:
        for two_d in (True, False):
            got = np.full(n, 0x5a5a, np.uint16)
            size, mem = ctypes.c_size_t(2 * n), got.ctypes.data_as(ctypes.c_void_p)
            assert hip.hipMemcpy(d, mem, size, 1) == 0  # host to device
            if two_d:
                _read_2d(plan, d.value + 2 * shift, 0, rows, stride, cols)
            else:
                want = data[:want.size]
                assert plan._lib.wavec_gpu_read_canvas(
                    plan._handle, 0, want.size,
                    ctypes.cast(d.value + 2 * shift, ctypes.POINTER(ctypes.c_uint16))) == 0
            assert hip.hipMemcpy(mem, d, size, 2) == 0  # device to host
            assert np.array_equal(got[shift:shift + want.size], want)
            assert np.all(got[:shift] == 0x5a5a) and np.all(got[shift + want.size:] == 0x5a5a)
    finally:
        hip.hipFree(d)


@contextlib.contextmanager
def _page_locked(n_bytes):
    hip, p = _hip(), ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(n_bytes), 0) == 0
    try:
        yield p.value
    finally:
        hip.hipHostFree(p)


def test_page_locked_reads_off_the_element_grid(wavec):
    """Destinations at odd bytes of page-locked memory (a host copy does not mind them)."""
    plan, data = _filled_plan(wavec, 700)
    with _page_locked(1 << 20) as base:
        mem = np.ctypeslib.as_array(ctypes.cast(base, ctypes.POINTER(ctypes.c_uint8)), (1 << 20,))
        for odd, rows, cols in ((1, 3, 5), (7, 64, 1024), (3, 300, 640)):
            mem[:] = 0xab
            _read_2d(plan, base + odd, 0, rows, 1024, cols)
            want = np.ascontiguousarray(data.reshape(-1, 1024)[:rows, :cols]).view(np.uint8).ravel()
            assert np.array_equal(mem[odd:odd + want.size], want)
            assert np.all(mem[:odd] == 0xab) and np.all(mem[odd + want.size:] == 0xab)


@pytest.mark.parametrize("byte", [0, 4, 2])
@pytest.mark.parametrize("C,W", [(5, 200), (1500, 1024)])
def test_infer_into_page_locked_memory(wavec, C, W, byte):
    """Results written in place, on the 16-byte grid, off it, and off the element grid."""
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", C, 1, W, is_1d=True)
    g.add_swiglu("m", "x", "x", "y")
    g.set_output("y")
    plan = g.compile()
    x = np.random.default_rng(W).standard_normal((C, 1, W)).astype(np.float32)
    want = plan.infer_f32(x)[0]
    fp = ctypes.POINTER(ctypes.c_float)
    with _page_locked(want.nbytes + 64) as base:
        mem = np.ctypeslib.as_array(ctypes.cast(base, ctypes.POINTER(ctypes.c_uint8)), (want.nbytes + 64,))
        mem[:] = 0xab
        assert plan._lib.wavec_gpu_infer_f32(plan._handle, x.ctypes.data_as(fp), x.size,
                                             ctypes.cast(base + byte, fp), want.size, None) == 0
        assert np.array_equal(mem[byte:byte + want.nbytes], want.view(np.uint8).ravel())
        assert np.all(mem[:byte] == 0xab) and np.all(mem[byte + want.nbytes:] == 0xab)


@pytest.mark.parametrize("C,W,extra", [(37, 200_000, 0), (5, 5_000_000, 0), (37, 200_000, 2_500_001)])
def test_inputs_of_several_stages(wavec, C, W, extra):
    """Inputs beyond the 16 MiB stage: several channels a pass, one channel larger than it, and one
    that ends inside a pass."""
    rng = np.random.default_rng(C)
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", C, 1, W, is_1d=True)
    g.add_sparse_wave("w", "x", "y", np.zeros((16, 4), np.uint32), np.ones((16, 4), np.float16), None,
                      cluster=1)
    g.set_output("y")
    plan = g.compile()
    plan.init_gpu()
    stride = (W + 63) // 64 * 64
    off = int(plan.cmds[0]["src_off"])
    plan.write_canvas(off, np.full(C * stride, 7.0, np.float16))
    n = C * W - extra
    x = rng.standard_normal(n, dtype=np.float32)
    y = np.zeros(1, np.float32)
    fp = ctypes.POINTER(ctypes.c_float)
    assert plan._lib.wavec_gpu_infer_f32(plan._handle, x.ctypes.data_as(fp), n, y.ctypes.data_as(fp), 1,
                                         None) == 0
    want = np.zeros((C, stride), np.float16)
    full = np.zeros(C * W, np.float16)
    full[:n] = x.astype(np.float16)
    want[:, :W] = full.reshape(C, W)
    assert np.array_equal(plan.read_canvas(off, C * stride), want.view(np.uint16).ravel())


def test_threads_reading_one_plan(wavec):
    """Threads that read different rows of one plan into pageable memory share its transfer ring."""
    plan, data = _filled_plan(wavec)
    jobs = [(0, 2048), (1024 * 100, 1 << 20), (1024 * 1000, 700_001), (7, 64)]
    wrong = []

    def work(off, n):
        for _ in range(20):
            if not np.array_equal(plan.read_canvas(off, n), data[off:off + n]):
                wrong.append((off, n))

    ts = [threading.Thread(target=work, args=j) for j in jobs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong

"""Device blocks kept between ps_free and ps_malloc: reuse, the size rule, and
giving them back."""
import ctypes
import time
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import powersparse_amd as ps
from powersparse_amd import _native
from gpu_util import say, setup

pytestmark = pytest.mark.gpu

MB = 1 << 20


def raw_free_bytes():
    """The driver's free memory, asked for without ps_mem_get_info's trim."""
    import torch
    return torch.cuda.mem_get_info()[0]


@pytest.mark.parametrize("first,second,same", [
    (64 * MB, 64 * MB, True), (64 * MB, 63 * MB + 5, True), (64 * MB, 52 * MB, True),
    (64 * MB, 50 * MB, False), (64 * MB, 65 * MB, False), (2 * MB, 2 * MB, True)])
def test_reuse_rule(first, second, same):
    # a kept block serves requests from four fifths of its size up to it
    setup()
    assert _native.hip().ps_mem_trim() == _native.PS_OK
    a = ps.DeviceBuffer(first)
    ptr = a.ptr
    a.free()
    b = ps.DeviceBuffer(second)
    say(f"{first} then {second}: {'same' if b.ptr == ptr else 'another'} block")
    got = b.ptr
    x = np.arange(second // 4, dtype=np.uint32)
    b.upload(x)
    np.testing.assert_array_equal(b.download(np.uint32, x.size), x)
    b.free()
    assert (got == ptr) == same


def test_given_back():
    setup()
    _native.hip().ps_mem_trim()
    free0 = raw_free_bytes()
    a = ps.DeviceBuffer(512 * MB)
    assert raw_free_bytes() <= free0 - 500 * MB
    a.free()
    assert raw_free_bytes() <= free0 - 500 * MB  # kept
    assert ps.mem_get_info()[0] >= free0 - 4 * MB  # counted as free, and given back
    assert raw_free_bytes() >= free0 - 4 * MB


def test_bounded():
    # blocks beyond a sixteenth of the device go back to the driver, oldest first
    setup()
    _native.hip().ps_mem_trim()
    total = ps.mem_get_info()[1]
    free0 = raw_free_bytes()
    n = total // 16 // (1024 * MB) + 3
    blocks = [ps.DeviceBuffer(1024 * MB) for _ in range(n)]
    for b in blocks:
        b.free()
    kept = free0 - raw_free_bytes()
    say(f"kept {kept >> 20} MB of {total >> 20} MB")
    assert total // 16 - 2048 * MB <= kept <= total // 16 + 4 * MB
    _native.hip().ps_mem_trim()


def test_threads_never_share_a_block():
    setup()

    def work(t):
        ps.set_device(0)
        rng = np.random.default_rng(t)
        for _ in range(30):
            n = int(rng.integers(2 * MB, 8 * MB)) // 4
            b = ps.DeviceBuffer(n * 4)
            x = rng.integers(0, 1 << 32, n, dtype=np.uint32)
            b.upload(x)
            np.testing.assert_array_equal(b.download(np.uint32, n), x)
            b.free()
        return True

    with ThreadPoolExecutor(8) as ex:
        assert all(ex.map(work, range(8)))


@pytest.mark.parametrize("nbytes", [-1, -(2 * MB) + 1, -(2 * MB)])
def test_sizes_beyond_the_address_range(nbytes):
    # (size_t)-1 and its neighbours: rounding them up to 2 MB must not wrap
    setup()
    p = ctypes.c_void_p(1)
    rc = _native.hip().ps_malloc(ctypes.byref(p), ctypes.c_size_t(nbytes))
    assert rc == _native.PS_ERR_RUNTIME and not p.value
    assert "out of memory" in _native.hip().ps_last_error().decode()
    # the failure is reported once, not by the next launch's check too
    x = ps.DeviceBuffer(4096)
    assert _native.hip().ps_fill_random_async(x.ptr, 1024, 1, 0.0, 1.0, 0, None) == _native.PS_OK
    ps.synchronize()


def test_second_free_is_refused():
    setup()
    hip = _native.hip()
    hip.ps_mem_trim()
    a = ps.DeviceBuffer(8 * MB)
    ptr = a.ptr
    assert hip.ps_free(ptr) == _native.PS_OK
    assert hip.ps_free(ptr) == _native.PS_ERR_RUNTIME
    a.ptr = None
    b, c = ps.DeviceBuffer(8 * MB), ps.DeviceBuffer(8 * MB)
    say(f"freed {ptr:#x}, then {b.ptr:#x} and {c.ptr:#x}")
    assert b.ptr == ptr and c.ptr != ptr
    for k, d in enumerate((b, c)):
        d.upload(np.full(2 * MB, k, np.uint32))
    for k, d in enumerate((b, c)):
        assert (d.download(np.uint32, 2 * MB) == k).all()
        d.free()


def kept_bytes():
    n = ctypes.c_size_t()
    assert _native.hip().ps_mem_kept(ctypes.byref(n)) == _native.PS_OK
    return n.value


def test_a_build_leaves_little():
    # one matrix built: its temporaries go back to the driver as the build ends,
    # with no later call; matrices built one after another keep theirs
    setup()
    _native.hip().ps_mem_trim()
    csr = ps.synth("C1", seed=3)
    free0 = raw_free_bytes()
    m = ps.PowerSparseMatrixGPU.from_csr(csr)
    say(f"first build: kept {kept_bytes() >> 20} MB, in use {free0 - raw_free_bytes() >> 20} MB")
    assert kept_bytes() <= 256 * MB
    m.close()
    own = kept_bytes()  # the destroyed matrix's blocks
    seen = []
    for _ in range(4):
        m = ps.PowerSparseMatrixGPU.from_csr(csr)
        seen.append((kept_bytes() >> 20, free0 - raw_free_bytes() >> 20))
        m.close()
    say(f"then kept / in use (MB): {seen}")
    assert own > 256 * MB and seen[-1] == seen[-2]  # nothing allocated, nothing given back
    _native.hip().ps_mem_trim()
    assert raw_free_bytes() >= free0 - 96 * MB  # (staging, code and the runtime's own)


def test_idle_blocks_go_back():
    setup()
    _native.hip().ps_mem_trim()
    free0 = raw_free_bytes()
    ps.DeviceBuffer(512 * MB).free()
    assert raw_free_bytes() <= free0 - 500 * MB
    time.sleep(10.5)
    ps.synchronize()
    assert kept_bytes() == 0 and raw_free_bytes() >= free0 - 4 * MB

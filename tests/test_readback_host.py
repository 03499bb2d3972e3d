"""What csrc/readback.hip asks of the HIP runtime and what it does when a call fails, on the host alone: the file is compiled
without its device code, with a model of the calls that it makes (fake_hip.cpp)."""
import ctypes as C
import subprocess
import threading
import time
from pathlib import Path

import numpy as np
import pytest

from turbogpt_amd import build

ROOT = Path(__file__).resolve().parents[1]
CHUNK = 2 << 20


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    folder = tmp_path_factory.mktemp("readback")
    library = folder / "libreadback.so"
    subprocess.run([build.HIPCC, "-x", "hip", "--offload-host-only", "-fuse-cuid=none", "-O1", "-std=c++17", "-fPIC", "-c",
                    str(ROOT / "tests/fake_hip.cpp"), "-o", str(folder / "readback.o")], check=True, capture_output=True)
    subprocess.run(["g++", "-shared", "-pthread", "-o", str(library), str(folder / "readback.o")], check=True, capture_output=True)
    lib = C.CDLL(str(library))
    lib.fake_stream.restype = lib.readback_open.restype = C.c_void_p
    lib.readback_error.restype = C.c_char_p
    lib.fake_hold.argtypes = [C.c_void_p, C.c_int]
    lib.fake_queued.argtypes = lib.readback_close.argtypes = [C.c_void_p]
    lib.readback_fetch.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int] + [C.c_void_p] * 4
    return lib


class Engine:
    """What an engine has of it: the staging memory, a device and a stream of that device."""

    def __init__(self, lib, device=0):
        self.lib, self.device = lib, device
        self.stream, self.handle = lib.fake_stream(device), lib.readback_open(device)

    def fetch(self, *sizes, seed=0, join=False):
        """-> whether the call succeeded and whether every byte arrived"""
        rng = np.random.default_rng(seed)
        sources = [rng.integers(0, 256, size, dtype=np.uint8) for size in sizes]
        results = [np.full(size, 0xaa, np.uint8) for size in sizes]
        count = len(sizes)
        halves = [(s.view(np.uint32) >> 16).astype(np.uint16) for s in sources], [s.view(np.uint32).astype(np.uint16) for s in sources]
        address = lambda arrays: (C.c_void_p * count)(*[a.ctypes.data for a in arrays])
        status = self.lib.readback_fetch(self.handle, self.stream, self.device, count, address(results), (C.c_size_t * count)(*sizes),
                                         address(halves[0] if join else sources),
                                         address(halves[1]) if join else (C.c_void_p * count)())
        return status == 0, all(np.array_equal(a, b) for a, b in zip(results, sources))

    def close(self):
        self.lib.readback_close(self.handle)


@pytest.mark.parametrize("sizes", [(16,), (CHUNK,), (CHUNK + 16,), (65536, 16, 86592), (5 * CHUNK - 32,), (40 * CHUNK + 48, 16)])
@pytest.mark.parametrize("join", [False, True])
def test_the_host_reads_what_the_kernels_wrote(host, sizes, join):
    engine = Engine(host)
    for seed in range(3):  # the buffers hold an earlier result from the second on
        assert engine.fetch(*sizes, seed=seed, join=join) == (True, True)
    engine.close()
    assert host.fake_pinned() == 0 and host.fake_events() == 0


@pytest.mark.parametrize("call", ["hipHostMalloc", "hipHostGetDevicePointer", "hipEventCreateWithFlags"])
@pytest.mark.parametrize("at", [1, 2, 4])
def test_a_buffer_that_could_not_be_made_is_not_used(host, call, at):
    engine = Engine(host)
    host.fake_fail(call.encode(), at)
    assert not engine.fetch(4 * CHUNK)[0]
    assert host.fake_pinned() == host.fake_events() == at - 1  # what was whole stays, the failed one is given back
    assert engine.fetch(4 * CHUNK, seed=1) == (True, True)
    engine.close()
    assert host.fake_pinned() == 0 and host.fake_events() == 0


@pytest.mark.parametrize("size", [16, CHUNK + 16, 2 * CHUNK, 3 * CHUNK, 20 * CHUNK])
@pytest.mark.parametrize("call,at", [("hipEventRecord", 1), ("hipEventRecord", 2), ("hipEventSynchronize", 1), ("hipLaunchKernel", 2)])
def test_a_failed_result_leaves_no_kernel_writing_to_the_shared_buffers(host, size, call, at):
    if at == 2 and size <= CHUNK:
        return  # the call is made once
    first, second = Engine(host), Engine(host)
    host.fake_fail(call.encode(), at)
    assert not first.fetch(size, seed=2)[0]
    assert b"injected" in host.readback_error()
    assert host.fake_queued(first.stream) == 0
    assert second.fetch(size, seed=3) == (True, True)
    first.close()
    second.close()


@pytest.mark.parametrize("size", [16, 3 * CHUNK, 40 * CHUNK])
def test_engines_on_two_devices(host, size):
    engines = [Engine(host, 0), Engine(host, 1), Engine(host, 0)]
    for seed in range(2):
        for engine in engines:
            assert engine.fetch(size, seed=seed) == (True, True), host.readback_error()
    held = host.fake_pinned()
    engines.pop(0).close()  # the other engine of device 0 goes on with the staging memory of the first
    assert host.fake_pinned() == held
    for engine in engines:
        assert engine.fetch(size, seed=5) == (True, True), host.readback_error()
        engine.close()
    assert host.fake_pinned() == host.fake_events() == 0


@pytest.mark.parametrize("behind,size", [(16, 16), (20 * CHUNK, 16), (20 * CHUNK, 20 * CHUNK)])
def test_a_result_does_not_wait_for_another_engines_kernels(host, behind, size):
    """While one engine's kernels still run, one thread waits for them, however large the result behind them; another engine of the
    device gets its own result meanwhile, and both have buffers of their own."""
    slow, other, results = Engine(host), Engine(host), {}
    host.fake_hold(slow.stream, 1)
    threads = [threading.Thread(target=lambda: results.update(slow=slow.fetch(behind, seed=1))),
               threading.Thread(target=lambda: results.update(other=other.fetch(size, seed=2)))]
    threads[0].start()
    end = time.monotonic() + 10
    while not host.fake_waiting() and time.monotonic() < end:
        time.sleep(0.01)
    threads[1].start()
    threads[1].join(5)
    meanwhile, waiting = dict(results), host.fake_waiting()
    host.fake_hold(slow.stream, 0)
    for thread in threads:
        thread.join()
    assert meanwhile == {"other": (True, True)} and waiting == 1
    assert results["slow"] == (True, True)
    held = host.fake_pinned()
    for seed in range(2):  # one after the other they need no more
        assert slow.fetch(behind, seed=seed) == (True, True) and other.fetch(size, seed=seed) == (True, True)
    assert host.fake_pinned() == held
    slow.close()
    other.close()
    assert host.fake_pinned() == host.fake_events() == 0

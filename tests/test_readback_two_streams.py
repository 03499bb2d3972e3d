"""Large results go by two streams in turn (csrc/readback.hip), on the host alone, with the model of the runtime in fake_hip.cpp: every
byte arrives whichever stream is behind, and a call that fails leaves nothing on either."""
import ctypes as C
import threading
import time

import pytest

from test_readback_host import CHUNK, Engine, host  # noqa: F401 (a fixture)


class TwoStreams(Engine):
    def __init__(self, lib, device=0):
        super().__init__(lib, device)
        self.second = lib.fake_stream(device)
        lib.readback_fetch_by_two.argtypes = [C.c_void_p] * 3 + [C.c_int] * 2 + [C.c_void_p] * 4
        outer = self

        class ByTwo:  # the library, with the second stream in its fetch
            @staticmethod
            def readback_fetch(handle, stream, *rest):
                return lib.readback_fetch_by_two(handle, stream, outer.second, *rest)

            def __getattr__(self, name):
                return getattr(lib, name)

        self.lib = ByTwo()


@pytest.mark.parametrize("sizes", [(16,), (CHUNK,), (CHUNK + 16,), (65536, 16, 86592), (40 * CHUNK + 48, 16)])
@pytest.mark.parametrize("join", [False, True])
def test_the_host_reads_what_the_kernels_wrote(host, sizes, join):  # noqa: F811
    engine = TwoStreams(host)
    for seed in range(3):
        assert engine.fetch(*sizes, seed=seed, join=join) == (True, True)
        assert host.fake_queued(engine.stream) == host.fake_queued(engine.second) == 0
    engine.close()
    assert host.fake_pinned() == 0 and host.fake_events() == 0


@pytest.mark.parametrize("size", [2 * CHUNK, 3 * CHUNK, 20 * CHUNK])
@pytest.mark.parametrize("call,at", [("hipEventRecord", 2), ("hipEventRecord", 3), ("hipEventSynchronize", 1), ("hipEventSynchronize", 2),
                                     ("hipLaunchKernel", 2), ("hipLaunchKernel", 3)])
def test_a_failed_result_leaves_nothing_on_either_stream(host, size, call, at):  # noqa: F811
    first, other = TwoStreams(host), TwoStreams(host)
    host.fake_fail(call.encode(), at)
    assert not first.fetch(size, seed=2)[0]
    assert b"injected" in host.readback_error()
    assert host.fake_queued(first.stream) == host.fake_queued(first.second) == 0
    assert other.fetch(size, seed=3) == (True, True)
    first.close()
    other.close()


@pytest.mark.parametrize("behind", ["stream", "second"])
@pytest.mark.parametrize("size", [2 * CHUNK, 30 * CHUNK])
def test_either_stream_may_be_behind(host, behind, size):  # noqa: F811
    """The call returns when the last chunk of both is there, and no sooner."""
    engine, results = TwoStreams(host), []
    host.fake_hold(getattr(engine, behind), 1)
    thread = threading.Thread(target=lambda: results.append(engine.fetch(size, seed=4)))
    thread.start()
    end = time.monotonic() + 10
    while not host.fake_waiting() and time.monotonic() < end:
        time.sleep(0.01)
    time.sleep(0.05)
    waiting, early = host.fake_waiting(), list(results)
    host.fake_hold(getattr(engine, behind), 0)
    thread.join()
    assert waiting and not early
    assert results == [(True, True)]
    engine.close()

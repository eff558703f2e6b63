"""The threaded copy out of the device (host_copy.h), on the CPU against a
stand-in for the HIP runtime: values and padding, and what it does when pinned
memory, an event or a copy fails."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
MB = 1 << 20
INVALID, NO_MEMORY = 1, 2  # hipErrorInvalidValue, hipErrorOutOfMemory


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_copy") / "stub")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "host_copy_stub.cpp"), "-o", exe], check=True)

    def run(rows, row_bytes, pitch, calls=1, alloc=0, event=0, copy=0):
        out = subprocess.run([exe] + [str(x) for x in (rows, row_bytes, pitch, calls, alloc, event, copy)], check=True,
                             capture_output=True, text=True, timeout=60).stdout.split("\n")
        return ([tuple(map(int, x.split())) for x in out[:calls]],
                dict(zip(("allocs", "chunks", "plain", "syncs", "workers", "live", "error", "device", "other"), map(int, out[calls].split()))))
    return run


SHAPES = [(1, 33 * MB + 40, 33 * MB + 40), (11, 3 * MB + 17, 3 * MB + 17), (11, 3 * MB + 17, 3 * MB + 81), (20, 2 * MB, 2 * MB + 64),
          (3000, 11200, 11216)]


@pytest.mark.parametrize("rows,row_bytes,pitch", SHAPES)
def test_large_results(stub, rows, row_bytes, pitch):
    got, n = stub(rows, row_bytes, pitch, calls=2)
    assert got == [(0, 1, 1)] * 2
    assert n["live"] == 0 and n["error"] == 0
    if n["workers"]:  # two CPUs for two workers: four at least
        assert n["allocs"] == 1 and n["plain"] == 0 and n["chunks"] > 0 and n["syncs"] == 2
    else:
        assert n["plain"] == 2


def test_the_callers_device_stays_current(stub):
    """Workers of their own take the context's device (0); the calling thread,
    which is on another (3), stays there."""
    _, n = stub(*SHAPES[2], calls=2)
    assert n["device"] == 3 and n["other"] == 0


def test_small_results_pin_nothing(stub):
    got, n = stub(1, 32 * MB - 8, 32 * MB - 8)
    assert got == [(0, 1, 1)]
    assert n["allocs"] == 0 and n["plain"] == 1 and n["workers"] == 0


@pytest.mark.parametrize("alloc,event", [(1, 0), (0, 1), (0, 3), (0, 4)])
def test_without_pinned_memory_or_events_the_plain_copy_does_it(stub, alloc, event):
    """Nothing is thrown, kept or left as the runtime's last error, and it is
    not tried again."""
    if (os.cpu_count() or 1) < 4:
        pytest.skip("one worker: no slots are made")
    got, n = stub(*SHAPES[2], calls=3, alloc=alloc, event=event)
    assert got == [(0, 1, 1)] * 3
    assert n["allocs"] == 1 and n["plain"] == 3 and n["chunks"] == 0 and n["workers"] == 0
    assert n["live"] == 0 and n["error"] == 0


@pytest.mark.parametrize("k", [1, 2, 7, 20])
def test_a_failing_copy_is_reported(stub, k):
    if (os.cpu_count() or 1) < 4:
        pytest.skip("one worker: no chunks are made")
    got, n = stub(*SHAPES[0][:1], 80 * MB, 80 * MB, calls=2, copy=k)
    assert got[0][0] == INVALID and got[1] == (0, 1, 1)
    assert n["live"] == 0

"""The copy of large outputs through pinned buffers (qstem_amd/csrc/qs_copyout.hpp) over a host
stand-in of the runtime: sizes around the chunks, a runtime that cannot give the buffers or
one of the events (the plain copy then, also in later calls, and a new attempt), and a
transfer that fails (reported, after the stream has been waited for)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "qstem_amd", "csrc")
MB = 1 << 20


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("copyout") / "harness")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + CSRC, os.path.join(HERE, "copyout_harness.cpp"), "-o", exe,
                    "-lpthread"], check=True)

    def call(*args):
        out = subprocess.run([exe, *args], capture_output=True, text=True, check=True, timeout=60).stdout.splitlines()
        copies = [tuple(int(v) for v in line.split()) for line in out[:4]]
        last = out[4].split()
        return copies, dict(buffers=int(last[1]), events=int(last[2]), null=int(last[4]), records=int(last[6]))
    return call


@pytest.mark.parametrize("size,chunks", [(1, 0), (16 * MB - 1, 0), (16 * MB, 16), (16 * MB + 1, 17), (21 * MB + 12345, 22)])
def test_data_arrive(run, size, chunks):
    copies, end = run("bytes=%d" % size)
    assert copies == [(0, 1, 0)] * 4
    assert end == dict(buffers=0, events=0, null=0, records=4 * chunks)


@pytest.mark.parametrize("what", ["host_alloc:1", "event_create:1", "event_create:4", "event_create:10"])
def test_setup_that_fails_once(run, what):
    copies, end = run("bytes=%d" % (18 * MB), "fail=" + what)
    assert copies == [(0, 1, 0)] * 4
    assert end == dict(buffers=0, events=0, null=0, records=3 * 18)


@pytest.mark.parametrize("what", ["copy:3", "event_record:5", "event_wait:7", "set_device:2"])
def test_failed_transfer_is_reported_once_the_stream_is_idle(run, what):
    copies, end = run("bytes=%d" % (18 * MB), "fail=" + what)
    assert copies[0][0] == 1 and copies[0][2] == 1
    assert copies[1:] == [(0, 1, 0)] * 3
    assert end["buffers"] == end["events"] == end["null"] == 0

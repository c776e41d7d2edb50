"""The host side of rnnt_hip_check_lengths_begin / _end, on a stand-in for the HIP runtime
(host_runtime.cpp): which device is asked, which tickets are honoured, what becomes of a
slot when something fails.  No device is needed; the kernel itself is tested in test_gpu_torch.py."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(os.path.dirname(HERE), "transducer_amd", "librnnt_hip.so")

PRELUDE = r"""
import ctypes, sys
rt = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
def knob(name): return ctypes.c_int.in_dll(rt, name)
lib.rnnt_hip_last_error.restype = ctypes.c_char_p
P, I = ctypes.c_void_p, ctypes.c_int
lib.rnnt_hip_check_lengths_begin.argtypes = [P, P, I, I, I, P, P]
lib.rnnt_hip_check_lengths_end.argtypes = [I, P, P]
keep = []
def begin(inputs=(6, 6), labels=(3, 3), stream=None, T=6, U=4):
    arrays = [(I * len(x))(*x) for x in (inputs, labels)]
    keep.append(arrays)
    ticket = I(-7)
    status = lib.rnnt_hip_check_lengths_begin(arrays[0], arrays[1], len(inputs), T, U, stream,
                                              ctypes.byref(ticket))
    return status, ticket.value
def end(ticket, stream=None):
    verdict = I(-7)
    status = lib.rnnt_hip_check_lengths_end(ticket, stream, ctypes.byref(verdict))
    return status, verdict.value
OK, INVALID, HIP_ERROR = 0, 1, 2
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("runtime") / "libruntime.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", out,
                           os.path.join(HERE, "host_runtime.cpp")])
    return out


def run(runtime, body):
    """`body` in a process of its own, the stand-in loaded ahead of the library."""
    subprocess.run([sys.executable, "-c", PRELUDE + body, runtime, LIB], check=True, timeout=60)


def test_the_stream_is_asked_on_the_device_of_the_check(runtime):
    """The null stream's handle is the same on every device: with another device current when the
    answer is waited for, an idle stream of that one says nothing about the check."""
    run(runtime, r"""
knob("current_device").value = 1
status, ticket = begin(inputs=(6, 7))
assert status == OK
knob("current_device").value = 0
knob("delay").value = 3
assert end(ticket) == (OK, 1), lib.rnnt_hip_last_error()
assert knob("asked").value == 4 and knob("current_device").value == 0
""")


def test_verdicts(runtime):
    run(runtime, r"""
for inputs, labels, want in (((6, 6), (3, 3), 0), ((7, 1), (3, 3), 1), ((6, 6), (0, 4), 2),
                             ((1, 2**31 - 1), (4, 4), 3), ((-5, 0), (-1, 0), 0)):
    status, ticket = begin(inputs, labels)
    assert status == OK and end(ticket) == (OK, want)
""")


def test_an_error_somebody_else_left_behind_does_not_release_a_slot_in_use(runtime):
    """The kernel is enqueued although an earlier call in this thread failed: its slot must not
    go to the next check while it is still to be written."""
    run(runtime, r"""
knob("delay").value = 1 << 30
knob("last_error").value = 1
status, first = begin(inputs=(7, 7))
assert status == OK and knob("launches").value == 1
assert knob("last_error").value == 1      # it is not this call's to take back
second = begin()
assert second[0] == OK and second[1] != first
knob("delay").value = 0
assert end(first) == (OK, 1) and end(second[1]) == (OK, 0)
""")


def test_a_launch_that_fails_gives_its_slot_back_only_after_a_wait(runtime):
    run(runtime, r"""
knob("launch_error").value = 98
for _ in range(1000):                     # the stream could be waited for: no slot is lost
    assert begin()[0] == HIP_ERROR
    assert knob("last_error").value == 0  # nor is an error left for the next launch to report
knob("launch_error").value = 0
assert begin()[0] == OK
knob("launch_error").value, knob("sync_error").value = 98, 98
for _ in range(255):                      # it could not: the slots stay out of use
    assert begin()[0] == HIP_ERROR
knob("launch_error").value = 0
assert begin()[0] == INVALID and b"under way" in lib.rnnt_hip_last_error()
""")


def test_a_ticket_is_good_for_one_end(runtime):
    run(runtime, r"""
assert end(0)[0] == INVALID               # nothing was ever begun
a, b = begin(inputs=(7, 7))[1], begin()[1]
for never in (-1, 256, 255 - a if 255 - a not in (a, b) else 17):
    assert end(never)[0] == INVALID
assert end(a) == (OK, 1)
for _ in range(300):                      # (each of these once put the slot on the free list)
    assert end(a)[0] == INVALID
tickets = [begin() for _ in range(255)]   # with b 256 under way, each on a slot of its own
assert all(t[0] == OK for t in tickets)
assert len({t[1] for t in tickets} | {b}) == 256
assert begin()[0] == INVALID and b"under way" in lib.rnnt_hip_last_error()
assert all(end(t[1]) == (OK, 0) for t in tickets) and end(b) == (OK, 0)
assert begin()[0] == OK
""")


def test_a_ticket_belongs_to_its_stream(runtime):
    run(runtime, r"""
a = begin(stream=0x10, inputs=(7, 7))[1]
assert end(a, stream=0x20)[0] == INVALID and end(a)[0] == INVALID
assert end(a, stream=0x10) == (OK, 1)
""")


def test_a_ticket_is_spent_by_an_end_that_fails(runtime):
    """A stream that reports an error ends the wait; what is on its way to the slot is not known
    then, so the slot stays out of use.  Where the stream has run out of work without the check, the
    slot is free again."""
    run(runtime, r"""
a = begin()[1]
knob("query_error").value = 719
assert end(a)[0] == HIP_ERROR and knob("last_error").value == 0
knob("query_error").value = 0
assert end(a)[0] == INVALID
others = [begin() for _ in range(255)]
assert all(t[0] == OK and t[1] != a for t in others) and begin()[0] == INVALID
for t in others: assert end(t[1]) == (OK, 0)
knob("lose").value = 1
for _ in range(300):
    status, t = begin()
    assert status == OK and end(t)[0] == HIP_ERROR and b"idle" in lib.rnnt_hip_last_error()
""")


def test_a_capturing_stream_is_refused(runtime):
    """The verdict of a captured kernel never comes: _end would wait for good."""
    run(runtime, r"""
for status in (1, 2):
    knob("capturing").value = status
    assert begin()[0] == INVALID and b"captur" in lib.rnnt_hip_last_error()
assert knob("launches").value == 0
knob("capturing").value = 0
assert end(begin()[1]) == (OK, 0)
knob("capture_error").value = 906         # the null stream while another thread captures
assert begin()[0] == HIP_ERROR and knob("last_error").value == 0 and knob("launches").value == 1
""")

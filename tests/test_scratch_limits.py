"""What an entry point does where the device has less memory than it would like: scratch that only
makes a call faster is given up, and the call goes through.  On the stand-in for the HIP runtime
(host_runtime.cpp): nothing is allocated and no kernel runs."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

BODY = r"""
import ctypes, sys
rt = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
from transducer_amd import capi
lib = capi.load()
knob = lambda name, t=ctypes.c_int: t.in_dll(rt, name)
limit, last = (knob(n, ctypes.c_uint64) for n in ("pool_limit", "pool_last"))
knob("lose").value = 1
p = 1 << 41  # stands for any device array
calls = {
    "viterbi_decode": (lib.rnnt_hip_viterbi_decode, [p] * 5, (1, 500, 41, 1000, 0)),
    "viterbi_decode_bf16": (lib.rnnt_hip_viterbi_decode_bf16, [p] * 5, (2, 700, 41, 999, 0)),
    "viterbi": (lib.rnnt_hip_viterbi, [p] * 6, (1, 500, 41, 1000, 0)),
    "maxplus_table": (lib.rnnt_hip_maxplus_table, [p] * 6, (3, 1000, 65, 600, 0)),
    "dense_grads": (lib.rnnt_hip_dense_grads, [p] * 9, (2, 10000, 101, 4000)),
}
f, arrays, sizes = calls[sys.argv[3]]
call = lambda: f(*arrays, *sizes, None)
assert call() == 0, lib.rnnt_hip_last_error()
liked = last.value
limit.value = liked - 1
assert call() == 0, lib.rnnt_hip_last_error()
assert last.value < liked and knob("last_error").value == 0
limit.value = last.value - 1
assert call() == 2 and b"HIP error" in lib.rnnt_hip_last_error()
"""


@pytest.mark.parametrize("entry", ["viterbi_decode", "viterbi_decode_bf16", "viterbi", "maxplus_table",
                                   "dense_grads"])
def test_less_memory_than_liked_is_enough(entry, tmp_path):
    out = str(tmp_path / "libruntime.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", out,
                           os.path.join(HERE, "host_runtime.cpp")])
    subprocess.run([sys.executable, "-c", BODY, out, ROOT, entry], check=True, timeout=60)

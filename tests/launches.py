"""Which kernels a call of the library launches, without a GPU.

The library is loaded in a child process after launch_recorder.cpp, whose HIP
runtime records launches and function attributes instead of doing anything.
"""

import ctypes as C
from dataclasses import dataclass
from functools import lru_cache
import json
from pathlib import Path
import shutil
import subprocess
import sys
import tempfile

import pytest

from venturi_amd import native

SOURCE = Path(__file__).resolve().parent / "launch_recorder.cpp"
CODES = {C.c_void_p: "P", C.c_int: "i", C.c_uint64: "Q", C.c_float: "f"}
POINTER = 1 << 30  # a device address that every alignment check accepts; never followed

CHILD = """
import ctypes as C, json, sys
recorder = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
recorder.recorder_take.restype = recorder.recorder_kernels.restype = C.c_char_p
library = C.CDLL(sys.argv[2])
library.venturi_blocks_error.restype = C.c_char_p
types = {"P": C.c_void_p, "i": C.c_int, "Q": C.c_uint64, "f": C.c_float}
results = []
for device, entry, signature, args in json.load(sys.stdin):
    function = getattr(library, entry)
    function.argtypes, function.restype = [types[t] for t in signature], C.c_int
    recorder.recorder_device(device)
    status = function(*args)
    results.append((status, library.venturi_blocks_error().decode(), recorder.recorder_take().decode()))
json.dump([results, recorder.recorder_kernels().decode()], sys.stdout)
"""


@dataclass(frozen=True)
class Launch:
    kernel: str  # name and template arguments
    device: int
    blocks: int
    threads: int
    shared: int


@dataclass(frozen=True)
class LdsLimit:
    kernel: str
    device: int
    bytes: int


@lru_cache(maxsize=1)
def _recorder():
    if shutil.which("g++") is None or not native.DEFAULT_LIBRARY.exists():
        pytest.skip("needs g++ and the built library")
    folder = tempfile.TemporaryDirectory(prefix="venturi-recorder-")  # kept by the cache, removed at exit
    target = Path(folder.name) / "recorder.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", str(SOURCE), "-o", str(target)], check=True)
    return folder, target


def _event(line):
    kind, kernel, *numbers = line.split("|")
    return (Launch if kind == "launch" else LdsLimit)(kernel, *map(int, numbers))


def _run(calls):
    coded = [(device, entry, "".join(CODES[t] for t in native.SIGNATURES[entry][0]), args) for device, entry, args in calls]
    done = subprocess.run([sys.executable, "-c", CHILD, str(_recorder()[1]), str(native.DEFAULT_LIBRARY)],
                          input=json.dumps(coded), capture_output=True, text=True, check=True, timeout=120)
    return json.loads(done.stdout)


def record(calls):
    """The events of each call (device, entry point, arguments), in order, in one process."""
    events = []
    for (status, message, text), call in zip(_run(calls)[0], calls):
        assert status == 0, (call, message)
        events.append([_event(line) for line in text.splitlines()])
    return events


def built(name):
    """Every instantiation of a kernel template in the library."""
    return {kernel for kernel in _run([])[1].splitlines() if kernel.split("<")[0] == name}


def kernels(calls):
    """The kernel names that each call launches."""
    return [[e.kernel for e in events if isinstance(e, Launch)] for events in record(calls)]


def padded(k):
    return (k + 127) // 128 * 128


def pointers(count):
    """Addresses of buffers 64 GiB apart."""
    return [POINTER + (i << 36) for i in range(count)]


def q8_prefill(tokens, n, k, *, scales_offset=0):
    x, codes, scales, out = pointers(4)
    return "venturi_q8_prefill_run", [x, codes, scales + scales_offset, out, tokens, n, k, padded(k), 0, None]


def a8_gemm(tokens, n, k, passes, *, scales_offset=0):
    workspace, codes, scales, out = pointers(4)
    return "venturi_q8_a8_gemm_run", [workspace, 1 << 35, codes, scales + scales_offset, out, tokens, n, k, padded(k),
                                      passes, None]


def a8_tiled(tokens, n, k, passes):
    workspace, codes, scales, out, slots = pointers(5)
    return "venturi_q8_a8_tiled_run", [workspace, 1 << 35, codes, scales, out, tokens, n, k, padded(k), passes, slots,
                                       1 << 30, None]


def q4_gemm(tokens, n, k):
    x, codes, scales, out = pointers(4)
    return "venturi_q4_gemm_run", [x, codes, scales, out, tokens, n, k, padded(k), 0, None]


def moe(tokens, hidden, experts, top_k, inter):
    x, ids, scores, gc, gs, dc, ds, out, workspace = pointers(9)
    return "venturi_moe_q4_run", [x, ids, scores, gc, gs, dc, ds, out, workspace, 1 << 35, tokens, top_k, experts, hidden,
                                  inter, None]

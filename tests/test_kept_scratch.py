"""The scratch that a thread keeps between the standalone ops.  On the CPU, over a
model of the allocator: no use and no free of memory that a device reset took
away, nor of what the program allocated at the same address since.  On the GPU:
the runtime's identifiers that this rests on, and an op before and after its
scratch is released."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from tatara_amd._lib import check
from tatara_amd.build import HIPCC
from tatara_amd.trainer import DeviceArray

ROOT = Path(__file__).resolve().parents[1]


def test_kept_scratch(tmp_path):
    cxx = shutil.which("g++")
    include = Path(HIPCC).resolve().parents[1] / "include"
    if cxx is None or not (include / "hip").is_dir():
        pytest.skip("no host C++ compiler or HIP headers")
    exe = tmp_path / "kept_scratch"
    subprocess.run([cxx, "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", f"-I{include}", "-pthread",
                    str(ROOT / "tests" / "kept_scratch.cpp"), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout


@pytest.mark.gpu
def test_identifiers_of_allocations(gpu):
    """Never given twice, and none for memory that was freed."""
    hip, buffer_id, seen = C.CDLL("libamdhip64.so.7"), 7, set()
    query = lambda p, out: hip.hipPointerGetAttribute(C.byref(out), C.c_int(buffer_id), C.c_void_p(p))  # noqa: E731
    for _ in range(8):
        p, ident = C.c_void_p(), C.c_uint64()
        check(gpu.tatara_malloc(C.byref(p), 1 << 20))
        assert query(p.value, ident) == 0
        assert ident.value not in seen
        seen.add(ident.value)
        check(gpu.tatara_free(p))
        assert query(p.value, ident) != 0
        hip.hipGetLastError()


@pytest.mark.gpu
def test_op_after_release(gpu):
    w = np.random.default_rng(1).normal(0, 0.3, (300, 64)).astype(np.float32)
    dw, out = DeviceArray(w), []
    for _ in range(3):
        d, n = DeviceArray(np.zeros(3 * w.size, np.uint8)), C.c_uint64()
        check(gpu.tatara_op_quantise_ft(dw.ptr, 300, 64, 0, 127.0, 1, d.ptr, 3 * w.size, C.byref(n)))
        out.append(d.to_host()[:n.value].tobytes())
        check(gpu.tatara_release_scratch())
        check(gpu.tatara_release_scratch())  # nothing left: nothing to do
    assert out[0] == out[1] == out[2]

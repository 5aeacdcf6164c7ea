"""The table quantiser's kernels at their edges, against the export oracle.

Values on both sides of every rounding and length line (k + 0.5, the 1/2/3 byte
lines at 63.5, -64.5, 8191.5, -8192.5, the i16 limits, NaN, infinities), tables
of one value up to several tiles of 4096 and several scans of 1024 tiles, and an
output that starts at each place in a 16-byte block, with guard bytes round it.
Whole numbers: equal, no tolerance.
"""
import ctypes as C

import numpy as np
import pytest

from oracle import export as ox
from tatara_amd import _lib
from tatara_amd.trainer import DeviceArray, check

pytestmark = pytest.mark.gpu

GUARD = 0xA5


def edge_values(n, seed):
    lines = [0.5, 1.5, 62.5, 63.5, 64.5, 65.5, 8190.5, 8191.5, 8192.5, 32766.5, 32767.5, 32768.5, 1e9, np.inf]
    x = np.array(lines + [-v for v in lines] + [0.0, -0.0, np.nan], np.float32)
    x = np.concatenate([x, np.nextafter(x, np.float32(np.inf)), np.nextafter(x, np.float32(-np.inf))])
    rng = np.random.default_rng(seed)
    v = (rng.normal(0, 1, n) * 10.0 ** rng.uniform(-1, 5, n)).astype(np.float32)
    pick = rng.random(n) < 0.5
    v[pick] = rng.choice(x, int(pick.sum()))
    return v


def run(w, rows, cols, pi, scale, shift):
    n = rows * cols
    cap = 3 * n
    dw, dout = DeviceArray(w), DeviceArray(np.full(cap + 64, GUARD, np.uint8))
    nbytes = C.c_uint64()
    check(_lib.load().tatara_op_quantise_ft(dw.ptr, rows, cols, pi, scale, 1, dout.ptr + 16 + shift, cap,
                                            C.byref(nbytes)))
    host = dout.to_host()
    end = 16 + shift + nbytes.value
    assert (host[:16 + shift] == GUARD).all() and (host[end:] == GUARD).all()
    return host[16 + shift:end].tobytes()


@pytest.mark.parametrize("rows,cols,pi,shift", [(1, 1, 0, 0), (1, 1, 0, 15), (3, 5, 2, 1), (1, 4095, 0, 7),
                                                (1, 4096, 0, 9), (1, 4097, 1, 3), (64, 64, 63, 4), (8, 2048, 3, 8),
                                                (5, 1000, 1, 13), (4100, 1028, 9, 2)])
@pytest.mark.parametrize("scale", [1.0, 127.0, 0.1])
def test_edges_of_rounding_lengths_and_tiles(gpu, rows, cols, pi, shift, scale):
    with np.errstate(over="ignore"):
        w = (edge_values((rows + pi) * cols, rows + cols) / np.float32(scale)).astype(np.float32)
    want = ox.leb128_encode(ox.quantise(ox.coalesce(w, rows, pi, cols), scale, ox.Q_LS_I16))
    assert run(w, rows, cols, pi, scale, shift) == want


def test_a_stream_longer_than_its_room_is_refused_and_nothing_written(gpu):
    w = np.full(5000, 100.0, np.float32)  # two bytes a value
    dw, dout = DeviceArray(w), DeviceArray(np.full(10000, GUARD, np.uint8))
    nbytes = C.c_uint64(7)
    lib = _lib.load()
    assert lib.tatara_op_quantise_ft(dw.ptr, 1, 5000, 0, 1.0, 1, dout.ptr, 9999, C.byref(nbytes)) != 0
    assert nbytes.value == 0 and (dout.to_host() == GUARD).all()
    check(lib.tatara_op_quantise_ft(dw.ptr, 1, 5000, 0, 1.0, 1, dout.ptr, 10000, C.byref(nbytes)))
    assert nbytes.value == 10000

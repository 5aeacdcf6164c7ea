"""The FT weight gradient of a caller's dft read in place and from a copy (GPU).

A row-major dft of whole 256-column chunks at an aligned address is read where
it lies; other widths and addresses go through a chunk-major copy (four values a
lane, or one).  Every layout gives the oracle's sums bit for bit in f32, the
occurrence-list fallback included, and the same bits for the same f16 values."""
import ctypes as C

import numpy as np
import pytest

from tatara_amd import _lib
from tatara_amd._lib import check
from tatara_amd.synthetic import small_spec, structured_batch
from tatara_amd.trainer import DeviceArray

from test_gpu_ops import _oracle_grad

pytestmark = pytest.mark.gpu

PI, KB, MA = 96, 3, 24


def rows(b, fallback):
    spec = small_spec(king_buckets=KB, piece_inputs=PI, max_active=MA)
    bt, _ = structured_batch(b, spec, num_buckets=1, seed=b, nnz_min=MA - 6)
    si = bt.stm_indices.copy()
    if fallback:
        si[1, 1] = (int(si[1, 0]) // PI + 1) % KB * PI  # a feature of another block
    return si, bt.nstm_indices, bt.nnz


def run(gpu, op, dft, idx, b, ft_out, shift, inv=None):
    """op on a dft placed `shift` values past an aligned address."""
    flat = np.concatenate([np.zeros(shift, dft.dtype), dft.ravel()])
    D, I = DeviceArray(flat), [DeviceArray(np.ascontiguousarray(x, np.int32)) for x in idx]
    G = DeviceArray(np.full((KB * PI, ft_out), np.nan, np.float32))
    used = C.c_uint32(9)
    head = [D.ptr + shift * dft.itemsize] + ([C.c_float(inv)] if inv is not None else [])
    check(op(*head, *(x.ptr for x in I), G.ptr, b, ft_out, KB * PI, MA, PI, C.byref(used)))
    return G.to_host(), used.value


@pytest.mark.parametrize("fallback", [False, True], ids=["scan", "lists"])
@pytest.mark.parametrize("b,ft_out", [(1, 256), (33, 512), (130, 260), (64, 4), (257, 768)])
def test_f32_layouts_bit_exact(gpu, b, ft_out, fallback):
    if fallback and b < 2:
        fallback = False
    idx = rows(b, fallback)
    dft = np.random.default_rng(b).normal(0, 1, (2, b, ft_out)).astype(np.float32)
    want = _oracle_grad(dft, *idx, b, ft_out, KB * PI, MA).reshape(KB * PI, ft_out)
    for shift in (0, 1, 4):
        got, used = run(gpu, gpu.tatara_op_ft_weight_grad_blocked, dft, idx, b, ft_out, shift)
        assert used == (0 if fallback else 1)
        assert np.array_equal(got, want), shift


@pytest.mark.parametrize("ft_out", [260, 384, 388])
def test_padding_of_the_copy_is_not_looked_at(gpu, ft_out):
    """The chunk-major copy's columns past ft_out hold what an earlier call left:
    after a call of NaN values the sums are the same bits as after one of zeros
    (a non-finite value in a row makes the matrix-core form add row by row)."""
    b, out = 200, []
    idx = rows(b, False)
    dft = np.random.default_rng(ft_out).normal(0, 1, (2, b, ft_out)).astype(np.float16).view(np.uint16)
    for left in (0.0, np.nan):
        run(gpu, gpu.tatara_op_ft_weight_grad_mfma_f16, np.full((2, b, 508), left, np.float16).view(np.uint16), idx, b,
            508, 0, 1.0)
        got, used = run(gpu, gpu.tatara_op_ft_weight_grad_mfma_f16, dft, idx, b, ft_out, 0, 1.0)
        assert used == 1
        out.append(got)
    assert np.array_equal(*out)


@pytest.mark.parametrize("b,ft_out", [(1, 256), (66, 512), (130, 260)])
def test_f16_layouts_agree(gpu, b, ft_out):
    idx = rows(b, False)
    dft = (np.random.default_rng(b).normal(0, 1, (2, b, ft_out)) * 8).astype(np.float16).view(np.uint16)
    exact = _oracle_grad(dft.view(np.float16).astype(np.float32), *idx, b, ft_out, KB * PI, MA).reshape(KB * PI, ft_out)
    inv = 1.0 / 64
    for op in (gpu.tatara_op_ft_weight_grad_blocked_f16, gpu.tatara_op_ft_weight_grad_mfma_f16):
        first = None
        for shift in (0, 2, 4, 1):
            got, used = run(gpu, op, dft, idx, b, ft_out, shift, inv)
            assert used == 1
            # h <= 2b terms of magnitude <= 64: f32 sums in any order within 2b * 2b * 64 * 2^-24
            assert np.abs(got - exact * np.float32(inv)).max() <= (2 * b) ** 2 * 64 * 2.0 ** -24 * inv + 1e-30
            first = got if first is None else first
            assert np.array_equal(got, first), shift


def test_kept_scratch_grows_and_is_each_threads_own(gpu):
    """Calls of growing, shrinking and fallback sizes from three threads at once."""
    import threading

    def work(seed, bad):
        try:
            for b, ft_out, fallback in ((5, 256, False), (300, 260, False), (40, 512, True), (700, 768, False)):
                b += seed
                idx = rows(b, fallback)
                dft = np.random.default_rng(b).normal(0, 1, (2, b, ft_out)).astype(np.float32)
                want = _oracle_grad(dft, *idx, b, ft_out, KB * PI, MA).reshape(KB * PI, ft_out)
                got, used = run(gpu, gpu.tatara_op_ft_weight_grad_blocked, dft, idx, b, ft_out, 0)
                if used != (0 if fallback else 1) or not np.array_equal(got, want):
                    bad.append((seed, b))
        except Exception as e:
            bad.append(repr(e))

    bad = []
    threads = [threading.Thread(target=work, args=(k, bad)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad

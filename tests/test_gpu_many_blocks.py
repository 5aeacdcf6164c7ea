"""Factorized tables of 128 king blocks, the most that the block scan takes, and
of more, which take occurrence lists (GPU).

The batch's rows lie in the first 128 blocks: nothing in such a batch tells the
scan's tables that the network has more.  Moments that are not zero show
whether the rows past block 127 are updated, and the virtual rows' moments
whether the fold adds the gradients of all blocks and no others."""
import ctypes as C

import numpy as np
import pytest

from oracle import layerstack as ols
from oracle import simple as osi
from tatara_amd._lib import check
from tatara_amd.synthetic import small_spec, structured_batch
from tatara_amd.trainer import (GROUPS, SIMPLE_GROUPS, DeviceArray, LayerStackConfig, LayerStackTrainer, Sigmoid,
                                SimpleConfig, SimpleTrainer)

import test_gpu_mixed as gm
import test_gpu_simple as gs
import test_gpu_trainer as gt
from test_gpu_ops import _oracle_grad

pytestmark = pytest.mark.gpu

PI, MA, B = 48, 16, 96


def rows(kb, seed):
    spec = small_spec(king_buckets=min(kb, 128), piece_inputs=PI, max_active=MA)
    return structured_batch(B, spec, num_buckets=8, seed=seed, nnz_min=10)


def some_moments(n, seed):
    """Inside the range of f16 moments (m 2^28, v 2^40)."""
    rng = np.random.default_rng(seed)
    return rng.normal(0, 1e-5, n).astype(np.float32), (1e-8 * (1 + rng.random(n))).astype(np.float32)


@pytest.mark.parametrize("kb", [128, 130])
def test_simple_step(gpu, kb):
    sh = osi.SimpleShape(ft_in=kb * PI, max_active=MA, piece_inputs=PI, ft_out=256, l1=32, l2=32)
    cfg = SimpleConfig(ft_in=sh.ft_in, max_active=MA, piece_inputs=PI, ft_out=256, l1_out=32, l2_out=32, max_batch=B,
                       optimizer="adamw", weight_decay=0.01)
    batch, _ = rows(kb, 1)
    st, loss = osi.default_init(sh), gs.WRM290
    m, v = some_moments(st["ft_w"]["w"].size, 2)
    st["ft_w"]["m"], st["ft_w"]["v"] = m.copy(), v.copy()
    with SimpleTrainer(cfg) as t:
        t.set("ft_w", m, "m")
        t.set("ft_w", v, "v")
        t.train_step(batch, 1e-3, 0.25, loss)
        osi.train_step(sh, st, gs.as_dict(batch), osi.OptConfig(), 1e-3, 0.25, gs.loss_dict(loss), 1)
        for name in SIMPLE_GROUPS:
            for k in ("w", "m", "v"):
                gs.close(t.get(name, k), st[name][k], 1e-5, atol=1e-6 if k == "w" else 0.0,
                         atol_frac=1e-5 if k != "w" else 0.0, what=f"{name}.{k}")


@pytest.mark.parametrize("kb,mixed", [(128, False), (130, False), (128, True), (130, True)])
def test_layerstack_step(gpu, kb, mixed):
    sh = ols.LsShape(ft_in=kb * PI, max_active=MA, piece_inputs=PI, ft_out=512, l1=16, l2=32, nb=8)
    cfg = LayerStackConfig(ft_in=sh.ft_in, max_active=MA, piece_inputs=PI, ft_out=512, num_buckets=8, max_batch=B,
                           optimizer="adamw", weight_decay=0.01)
    cfg = cfg.all_optim() if mixed else cfg
    prec = ols.Precision.all_optim() if mixed else ols.FP32
    batch, bucket = rows(kb, 3)
    st, loss = ols.default_init(sh), Sigmoid()
    m, v = some_moments(st["ft_w"]["w"].size, 4)
    st["ft_w"]["m"], st["ft_w"]["v"] = m.copy(), v.copy()
    if mixed:
        ols.to_f16_state(st)
    opt = ols.OptConfig(optimizer="adamw", weight_decay=0.01)
    with LayerStackTrainer(cfg) as t:
        t.set("ft_w", m, "m")
        t.set("ft_w", v, "v")
        t.train_step(batch, bucket, 8.75e-4, 0.25, loss)
        _, a, g = ols.train_step(sh, st, gt.as_dict(batch, bucket), opt, 8.75e-4, 0.25, gt.loss_dict(loss), 1, prec)
        bound = gm.f16_grad_bound(sh, gt.as_dict(batch, bucket), a, B, kb <= 128) if mixed else None
        gm.check_moments(t, st, prec, f"{kb} blocks", g=g["ft_w"], g_bound=bound, opt=opt)
        if not mixed:
            for name in GROUPS:
                gt.close(t.get(name), st[name]["w"], 1e-5, atol=1e-6, what=name)


@pytest.mark.parametrize("kb,ft_out", [(128, 256), (129, 256), (200, 256), (129, 260)])
def test_gradient_op(gpu, kb, ft_out):
    batch, _ = rows(kb, 5)
    idx = (batch.stm_indices, batch.nstm_indices, batch.nnz)
    dft = (np.random.default_rng(kb).integers(-64, 64, (2, B, ft_out)) / 64).astype(np.float32)  # exact in f16
    want = _oracle_grad(dft, *idx, B, ft_out, kb * PI, MA).reshape(kb * PI, ft_out)
    d32, d16 = DeviceArray(dft), DeviceArray(dft.astype(np.float16).view(np.uint16))
    I = [DeviceArray(np.ascontiguousarray(x, np.int32)) for x in idx]
    for op, head in ((gpu.tatara_op_ft_weight_grad_blocked, [d32.ptr]),
                     (gpu.tatara_op_ft_weight_grad_blocked_f16, [d16.ptr, C.c_float(1.0)]),
                     (gpu.tatara_op_ft_weight_grad_mfma_f16, [d16.ptr, C.c_float(1.0)])):
        G, used = DeviceArray(np.full((kb * PI, ft_out), np.nan, np.float32)), C.c_uint32(9)
        check(op(*head, *(x.ptr for x in I), G.ptr, B, ft_out, kb * PI, MA, PI, C.byref(used)))
        # sums of multiples of 1/64 below 2^18: exact in f32 in any order
        assert np.array_equal(G.to_host(), want)
        assert used.value == (1 if kb <= 128 else 0)

"""The dense kernels at the edges of their tiles (GPU): batches of one row tile
and one more row, waves whose columns end inside the row, buckets without
rows, and batches large enough that a workgroup takes several tiles.
One step against the oracle with the one-step bars of the trainer tests."""
import numpy as np
import pytest

from oracle import layerstack as ols
from oracle import simple as osi
from tatara_amd.trainer import GROUPS, SIMPLE_GROUPS, LayerStackTrainer, Sigmoid, SimpleTrainer

import test_gpu_mixed as gm
import test_gpu_simple as gs
import test_gpu_trainer as gt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ft_out,l1,l2,b", [(32, 8, 16, 1), (96, 16, 32, 17), (160, 32, 64, 33), (96, 32, 32, 255),
                                            (64, 8, 32, 16), (32, 32, 16, 40000)])
def test_simple_edges(gpu, ft_out, l1, l2, b):
    sh, cfg = gs.make(ft_out=ft_out, l1=l1, l2=l2, optimizer="adamw", b=b)
    batch = gs.batch_for(b, b)
    st = osi.default_init(sh)
    with SimpleTrainer(cfg) as t:
        t.train_step(batch, 1e-3, 0.25, gs.WRM290)
        _, a, g = osi.train_step(sh, st, gs.as_dict(batch), osi.OptConfig(), 1e-3, 0.25, gs.loss_dict(gs.WRM290), 1)
        gs.close(t.activation("l1_pre", b * l1), a["l1_pre"], 1e-5, atol=1e-6, what="l1_pre")
        gs.close(t.activation("net_output", b), a["net"], 1e-5, atol=1e-6, what="net_output")
        for name in ("dft_stm", "dft_nstm"):
            top = max(np.abs(a[name]).max(), 1e-30)
            gs.close(t.activation(name, b * ft_out), a[name], 1e-4, atol=1e-5 * top, what=name)
        for name in SIMPLE_GROUPS:
            gs.close(t.get(name, "grad"), g[name], 1e-4, atol_frac=1e-5, what=f"grad {name}")


@pytest.mark.parametrize("ft_out,l1,l2,b,factorize", [(128, 8, 16, 16, True), (384, 16, 32, 48, True),
                                                      (128, 32, 64, 272, False), (640, 32, 16, 1040, True),
                                                      (128, 16, 64, 34000, False),
                                                      # 255 and 256 tiles: the L1 forward's line at 128 columns
                                                      (128, 32, 16, 3936, False), (128, 32, 16, 3952, False)])
def test_layerstack_edges(gpu, ft_out, l1, l2, b, factorize):
    sh, cfg = gt.make(ft_out=ft_out, l1=l1, l2=l2, b=b, factorize=factorize)
    batch, bucket = gt.batch_for(b, b, sh.nb)
    bucket[bucket == 2] = 5  # a bucket without rows
    st = ols.default_init(sh)
    loss = Sigmoid()
    with LayerStackTrainer(cfg) as t:
        t.train_step(batch, bucket, 8.75e-4, 0.25, loss)
        _, a, g = ols.train_step(sh, st, gt.as_dict(batch, bucket), ols.OptConfig(), 8.75e-4, 0.25,
                                 gt.loss_dict(loss), 1)
        gt.close(t.activation("l1_total", b * l1), a["l1_total"], 1e-5, atol=1e-6, what="l1_total")
        gt.close(t.activation("net_output", b), a["net"], 1e-5, atol=1e-6, what="net_output")
        for name in ("dft_stm", "dft_nstm"):
            top = max(np.abs(a[name]).max(), 1e-30)
            gt.close(t.activation(name, b * ft_out), a[name], 1e-4, atol=1e-5 * top, what=name)
        for name in GROUPS:
            gt.close(t.get(name, "grad"), g[name], 1e-4, atol_frac=1e-5, what=f"grad {name}")


# The input gradient's row blocks hold eight tiles from tiles * ft_out / 64 = 32768
# on: 1366 and 1367 tiles of 16 rows end in a block of 6 and 7 (f32 writes a whole
# ft_b partial and a shorter one there, f16 one).  The mixed form below that at
# columns of one and three workgroups.
@pytest.mark.parametrize("mixed,ft_out,l1,b", [(False, 1536, 8, 21712), (False, 1536, 16, 21728), (True, 1536, 8, 21712),
                                               (True, 1536, 32, 21728), (True, 128, 32, 272), (True, 384, 8, 1040)])
def test_input_gradient_row_blocks(gpu, mixed, ft_out, l1, b):
    prec = ols.Precision.all_optim() if mixed else ols.FP32
    sh, cfg = gt.make(ft_out=ft_out, l1=l1, l2=16, b=b, factorize=False)
    cfg = cfg.all_optim() if mixed else cfg
    batch, bucket = gt.batch_for(b, b, sh.nb)
    st = gm.oracle_state(sh, prec)
    bf, loss = b * ft_out, Sigmoid()
    with LayerStackTrainer(cfg) as t:
        t.train_step(batch, bucket, 8.75e-4, 0.25, loss)
        _, a, g = ols.train_step(sh, st, gt.as_dict(batch, bucket), ols.OptConfig(), 8.75e-4, 0.25,
                                 gt.loss_dict(loss), 1, prec)
        for name in ("dft_stm", "dft_nstm"):
            if mixed:
                gt.close(t.activation(name, bf), a[name + "16"], 2e-3, atol=gm.SUB16, what=name)
            else:
                gt.close(t.activation(name, bf), a[name], 1e-4, atol=1e-5 * np.abs(a[name]).max(), what=name)
        for name in GROUPS:
            if name != "ft_w":
                gt.close(t.get(name, "grad"), g[name], 1e-4, atol_frac=1e-5, what=f"grad {name}")


@pytest.mark.parametrize("arch", ["simple", "layerstack", "unfactorized"])
def test_dense_gradients_beside_the_table_gradient(gpu, arch):
    """The dense side stream against the one stream of a profiled trainer: equal bits after four steps."""
    b, out = 720, []
    for profiled in (False, True):
        if arch == "simple":
            _, cfg = gs.make(ft_out=256, l1=32, l2=32, optimizer="adamw", b=b)
            t, groups, args = SimpleTrainer(cfg), SIMPLE_GROUPS, (gs.batch_for(b, b),)
        else:
            sh, cfg = gt.make(ft_out=512, l1=16, l2=32, b=b, factorize=arch == "layerstack")
            t, groups, args = LayerStackTrainer(cfg), GROUPS, gt.batch_for(b, b, sh.nb)
        with t:
            t.set_profiling(profiled)
            losses = [t.train_step(*args, 1e-3, 0.25, Sigmoid()) for _ in range(4)]
            losses.append(t.flush_pending_loss())
            out.append([np.array(losses)] + [t.get(n, k) for n in groups for k in ("w", "m", "v")])
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("arch", ["simple", "layerstack"])
def test_rows_without_an_occurrence(gpu, arch):
    """Gradients of absent rows unwritten against a trainer that keeps every
    gradient: equal bits over batches whose rows come and go (what an earlier
    step left in the gradients is not used), one position, and a batch with a
    feature of another king block (every gradient comes from the other kernel)."""
    out = []
    for keep in (False, True):
        if arch == "simple":
            _, cfg = gs.make(ft_out=256, l1=32, l2=32, optimizer="adamw", b=64)
            cfg.keep_grads = keep
            t, groups = SimpleTrainer(cfg), SIMPLE_GROUPS
        else:
            sh, cfg = gt.make(ft_out=512, l1=16, l2=32, b=64, factorize=True)
            cfg.keep_grads = keep
            t, groups = LayerStackTrainer(cfg), GROUPS
        with t:
            for b, seed, stray in ((64, 1, False), (16, 2, False), (32, 3, True), (48, 4, False)):
                if arch == "simple":
                    args = (gs.batch_for(seed, b),)
                else:
                    args = gt.batch_for(seed, b, sh.nb)
                if stray:
                    idx = args[0].stm_indices.reshape(b, -1)
                    idx[5, 0] = (int(idx[5, 0]) + cfg.piece_inputs) % cfg.ft_in
                t.train_step(*args, 1e-2, 0.25, Sigmoid())
            out.append([t.get(n, k) for n in groups for k in ("w", "m", "v")])
    for x, y in zip(*out):
        assert np.array_equal(x, y)

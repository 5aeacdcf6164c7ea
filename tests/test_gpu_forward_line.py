"""The FT forward on both sides of the line between the LDS-resident gather and
the row gather (GPU): the oracle's sums bit for bit, whichever form a trainer
takes for its batch capacity.

The line is drawn over 2 * max_batch * max_active / table rows, so each shape
comes with a capacity just below it and one on it, with a row whose features
lie in two king blocks, king blocks of the largest width held in LDS and
rows padded to 40 and to 48 slots.
"""
import numpy as np
import pytest

from oracle import layerstack as ols
from oracle import simple as osi
from tatara_amd.synthetic import small_spec, structured_batch
from tatara_amd.trainer import Batch, LayerStackConfig, LayerStackTrainer, Sigmoid, SimpleConfig, SimpleTrainer, Wrm

pytestmark = pytest.mark.gpu

SIGMOID = {"kind": "sigmoid", "scale": 1.0 / 290.0}
WRM = {"kind": "wrm", "nnue2score": 600.0, "in_scaling": 340.0, "in_offset": 270.0, "target_offset": 270.0,
       "target_scaling": 380.0, "pow_exp": 2.0, "qp_asymmetry": 0.0, "w1": 0.0, "w2": 0.5}


def a_batch(b, spec, seed):
    batch, bucket = structured_batch(b, spec, num_buckets=8, seed=seed, nnz_min=spec["max_active"] - 10)
    stm = batch.stm_indices.copy()
    pi, kb = spec["piece_inputs"], spec["king_buckets"]
    stm[9, 1] = (int(stm[9, 0]) // pi + 1) % kb * pi + 5  # a feature of another king block
    return Batch(stm, batch.nstm_indices, batch.nnz, batch.score, batch.wdl), bucket


# (king blocks, pieces, slots, columns, occurrences per table row on the line)
@pytest.mark.parametrize("mixed,kb,pi,ma,ft_out,line",
                         [(False, 10, 64, 40, 512, 20), (False, 10, 64, 44, 640, 20), (False, 10, 64, 38, 768, 16),
                          (False, 2, 1791, 40, 384, 20), (True, 10, 64, 40, 640, 20), (True, 10, 64, 44, 512, 80),
                          (False, 10, 64, 40, 128, 16), (False, 10, 64, 38, 256, 20), (True, 10, 64, 44, 128, 12),
                          (True, 10, 64, 40, 256, 20)])
def test_layerstack_forward_on_both_sides(gpu, mixed, kb, pi, ma, ft_out, line):
    spec = small_spec(king_buckets=kb, piece_inputs=pi, max_active=ma)
    sh = ols.LsShape(ft_in=kb * pi, max_active=ma, piece_inputs=pi, ft_out=ft_out, l1=16, l2=32, nb=8)
    on = -(-line * kb * pi // (2 * ma * 16)) * 16
    prec = ols.Precision.all_optim() if mixed else ols.FP32
    for b in (on - 16, on):
        cfg = LayerStackConfig(ft_in=kb * pi, max_active=ma, piece_inputs=pi, ft_out=ft_out, num_buckets=8,
                               max_batch=b)
        batch, bucket = a_batch(b, spec, b)
        st = ols.default_init(sh)
        with LayerStackTrainer(cfg.all_optim() if mixed else cfg) as t:
            _, net = t.validate_step(batch, bucket, 0.0, Sigmoid())
            a, _ = ols.forward(sh, st, dict(stm=batch.stm_indices, nstm=batch.nstm_indices, nnz=batch.nnz,
                                            bucket=bucket, score=batch.score, wdl=batch.wdl), 0.0, SIGMOID, prec)
            for name, key in (("ft_stm_out", "ft_stm"), ("ft_nstm_out", "ft_nstm"), ("combined", "combined")):
                assert np.array_equal(t.activation(name, b * ft_out), a[key]), (b, name)
            assert np.allclose(net, a["net"], rtol=1e-5, atol=1e-6), b


@pytest.mark.parametrize("kb,pi,ma,ft_out,line", [(10, 64, 44, 256, 32), (10, 64, 38, 512, 20), (2, 1791, 40, 128, 32),
                                                  (10, 64, 40, 32, 8), (2, 1791, 38, 128, 10), (10, 64, 44, 224, 14)])
def test_simple_forward_on_both_sides(gpu, kb, pi, ma, ft_out, line):
    spec = small_spec(king_buckets=kb, piece_inputs=pi, max_active=ma)
    sh = osi.SimpleShape(ft_in=kb * pi, max_active=ma, piece_inputs=pi, ft_out=ft_out, l1=32, l2=32)
    on = -(-line * kb * pi // (2 * ma))
    for b in (on - 1, on):
        batch, _ = a_batch(b, spec, b)
        st = osi.default_init(sh)
        with SimpleTrainer(SimpleConfig(ft_in=kb * pi, max_active=ma, piece_inputs=pi, ft_out=ft_out,
                                        max_batch=b)) as t:
            _, net = t.validate_step(batch, 0.0, Wrm())
            a, _ = osi.forward(sh, st, dict(stm=batch.stm_indices, nstm=batch.nstm_indices, nnz=batch.nnz,
                                            score=batch.score, wdl=batch.wdl), 0.0, WRM)
            for name, key, n in (("ft_stm_out", "ft_stm", 1), ("ft_nstm_out", "ft_nstm", 1), ("combined", "combined", 2)):
                assert np.array_equal(t.activation(name, n * b * ft_out), a[key]), (b, name)
            assert np.allclose(net, a["net"], rtol=1e-5, atol=1e-6), b


# The row gather takes the positions by king block above 320 MB of gathered rows
# (validation), or 256 MB and 2048 positions (a step), and in the batch's order
# below.
@pytest.mark.parametrize("arch,ft_out", [("simple", 512), ("simple", 256), ("layerstack", 1280), ("mixed", 1280)])
@pytest.mark.parametrize("train", [False, True])
def test_row_gather_in_either_order(gpu, arch, ft_out, train):
    kb, pi, ma = 100, 128, 40
    spec = small_spec(king_buckets=kb, piece_inputs=pi, max_active=ma)
    lo = (256 if train else 320) * 2 ** 20 // (2 * ma * ft_out * (2 if arch == "mixed" else 4)) // 16 * 16
    lo = max(lo, 2048) if train else lo
    batch, bucket = a_batch(lo + 16, spec, lo)
    first = Batch(batch.stm_indices[:lo], batch.nstm_indices[:lo], batch.nnz[:lo], batch.score[:lo], batch.wdl[:lo])
    out = []
    for b, args in ((lo, (first, bucket[:lo])), (lo + 16, (batch, bucket))):
        shape = dict(ft_in=kb * pi, max_active=ma, piece_inputs=pi, ft_out=ft_out, max_batch=lo + 16)
        if arch == "simple":
            cfg = SimpleConfig(l1_out=32, l2_out=32, **shape)
            cls, args = SimpleTrainer, args[:1]
        else:
            cfg = LayerStackConfig(num_buckets=8, **shape)
            cfg, cls = cfg.all_optim() if arch == "mixed" else cfg, LayerStackTrainer
        with cls(cfg) as t:
            if train:
                t.train_step(*args, 1e-3, 0.0, Wrm())
            else:
                t.validate_step(*args, 0.0, Wrm())
            wide = ft_out * (2 if arch == "simple" else 1)
            out.append([t.activation(n, b * w)[:lo * w] for n, w in
                        (("ft_stm_out", ft_out), ("ft_nstm_out", ft_out), ("combined", wide))])
    for x, y in zip(*out):
        assert np.array_equal(x, y)


# A trainer chooses by its capacity whether it stages the whole table or gathers
# rows: the same small batch on a capacity far above the line and on one below it.
@pytest.mark.parametrize("arch,ft_out", [("simple", 256), ("layerstack", 512), ("layerstack", 128), ("mixed", 640)])
@pytest.mark.parametrize("train", [False, True])
def test_small_batch_on_a_large_capacity(gpu, arch, ft_out, train):
    kb, pi, ma, b = 10, 64, 40, 48
    spec = small_spec(king_buckets=kb, piece_inputs=pi, max_active=ma)
    batch, bucket = a_batch(b, spec, 7)
    out = []
    for capacity in (b, 4096):
        shape = dict(ft_in=kb * pi, max_active=ma, piece_inputs=pi, ft_out=ft_out, max_batch=capacity)
        if arch == "simple":
            cfg, cls, args = SimpleConfig(l1_out=32, l2_out=32, **shape), SimpleTrainer, (batch,)
        else:
            cfg, cls, args = LayerStackConfig(num_buckets=8, **shape), LayerStackTrainer, (batch, bucket)
            cfg = cfg.all_optim() if arch == "mixed" else cfg
        with cls(cfg) as t:
            if train:
                t.train_step(*args, 1e-3, 0.0, Wrm())
                t.flush_pending_loss()
            wide = ft_out * (2 if arch == "simple" else 1)
            got = [np.float64(t.validate_step(*args, 0.0, Wrm())[1])]  # with the weights after the step
            out.append(got + [t.activation(n, b * w) for n, w in
                              (("ft_stm_out", ft_out), ("ft_nstm_out", ft_out), ("combined", wide))])
    for x, y in zip(*out):
        assert np.array_equal(x, y)

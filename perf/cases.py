"""The work that a user of this library has it do, as cases that can be timed and compared.

A training program decodes PSV records into batches, steps a LayerStack or a
Simple network over them, scores held-out batches and, now and then, exports
the quantised network.  The cases take these calls through the public entry
points: the step API of `tatara_amd.trainer` and the C ABI of
include/tatara_hip.h, over the feature sets, network shapes, batch sizes,
optimizers, losses and precisions that the configurations, the tests and the
benchmark use.

Positions are seeded shogi positions of the benchmark's kind (40 pieces, 15%
of them in hand, 10% of the promotable ones promoted, scores ~ N(0, 600)).
Weights are those of a network that has been trained for a while: feature sums
that mostly lie inside the clipped range, dense layers of unit gain, a
factorizer that is not zero.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from tatara_amd import _lib
from tatara_amd.dataloader import (BUCKET_MODES, FEATURE_SETS, KPABS_WEIGHTS, ProgressWeights, device_batch_to_host,
                                   feature_set_info, psv_to_device_batch)
from tatara_amd.trainer import (Batch, DeviceBatch, LayerStackConfig, LayerStackTrainer, Sigmoid, SimpleConfig,
                                SimpleTrainer, Wrm)

DEV = "cuda"
FT_POST_SCALE = L1_SQR_SCALE = 127.0 / 128.0
QUANT_CLAMP = 127.0 / 64.0
BATCHES = 4  # different batches that a training case cycles through


def listed() -> list[dict]:
    return [
        # Every batch of a training run starts as 40-byte records: the headline
        # configuration's batch, with the progress buckets.
        dict(name="decode_hm_65536", kind="decode", features="halfka-hm-merged", bucket="progress8kpabs", n=65536),
        # A short, ragged read: the last records of a small file, for a Simple network.
        dict(name="decode_halfkp_1023", kind="decode", features="halfkp", bucket="none", n=1023),
        # The feature transformer alone, forward and backward: the sparse layer
        # that a program with its own dense layers calls.
        dict(name="ft_forward_768_16384", kind="ft_forward", features="halfka-hm-merged", ft_out=768, n=16384),
        dict(name="ft_grad_768_16381", kind="ft_grad", features="halfka-hm-merged", ft_out=768, n=16381, half=False),
        dict(name="ft_grad_f16_1536_16384", kind="ft_grad", features="halfka-hm-merged", ft_out=1536, n=16384,
             half=True),
        # The headline training configuration, f32 and in mixed precision:
        # superbatches that end with the loss flushed and the weights read back.
        dict(name="train_ls1536_65536", kind="train", arch="layerstack", features="halfka-hm-merged", ft_out=1536,
             l1=16, l2=32, n=65536, steps=12, mixed=False, factorize=True, bucket="progress8kpabs", loss="sigmoid",
             optimizer="ranger", resident=True),
        dict(name="train_ls1536_mixed_65536", kind="train", arch="layerstack", features="halfka-hm-merged",
             ft_out=1536, l1=16, l2=32, n=65536, steps=12, mixed=True, factorize=True, bucket="progress8kpabs",
             loss="sigmoid", optimizer="ranger", resident=True),
        # The smaller LayerStack at the default batch size, fed from host arrays
        # as the reference's step API is.
        dict(name="train_ls768_host_16384", kind="train", arch="layerstack", features="halfka-hm-merged", ft_out=768,
             l1=8, l2=32, n=16384, steps=24, mixed=False, factorize=True, bucket="kingrank9", loss="wrm",
             optimizer="ranger", resident=False),
        # One superbatch of 64 small steps of the Simple network.
        dict(name="train_simple256_4096", kind="train", arch="simple", features="halfkp", ft_out=256, l1=32, l2=32,
             n=4096, steps=64, mixed=False, factorize=True, bucket="none", loss="wrm", optimizer="adamw",
             resident=True),
        # Without the factorizer (the reference's --no-ft-factorize), with the
        # widest dense layers and a small batch.
        dict(name="train_ls512_plain_2048", kind="train", arch="layerstack", features="halfka-hm-merged", ft_out=512,
             l1=32, l2=64, n=2048, steps=32, mixed=False, factorize=False, bucket="progress8kpabs", loss="wrm_ext",
             optimizer="radam", resident=True),
        # Held-out scoring of a small batch: the smallest whole call.
        dict(name="validate_ls768_1008", kind="validate", arch="layerstack", features="halfka-hm-merged", ft_out=768,
             l1=8, l2=32, n=1008, mixed=False, factorize=True, bucket="kingrank9", loss="sigmoid", resident=True),
        # The feature table of a checkpoint's quantised network.
        dict(name="export_ft_1536", kind="export", features="halfka-hm-merged", ft_out=1536, factorize=True,
             leb128=True),
    ]


def _log_int(rng, lo: int, hi: int, multiple: int = 1) -> int:
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / multiple)) * multiple))


def draw(rng) -> dict:
    features = rng.choice(["halfka-hm-merged", "halfka-hm-merged", "halfkp", "halfka-hm-split"])
    kind = rng.choice(["decode", "ft_forward", "ft_grad", "train", "train", "train", "validate", "export"])
    if kind == "decode":
        return dict(kind=kind, features=rng.choice([features, "halfka-split", "halfka-merged"]),
                    bucket=rng.choice(["none", "kingrank9", "progress8kpabs"]), n=_log_int(rng, 256, 65536))
    if kind in ("ft_forward", "ft_grad"):
        c = dict(kind=kind, features=features, ft_out=128 * rng.randint(2, 12), n=_log_int(rng, 512, 32768))
        if kind == "ft_grad":
            c["half"] = rng.random() < 0.4
        return c
    if kind == "export":
        return dict(kind=kind, features=features, ft_out=128 * rng.randint(1, 10), factorize=rng.random() < 0.7,
                    leb128=rng.random() < 0.6)
    arch = rng.choice(["layerstack", "layerstack", "simple"])
    c = dict(kind=kind, arch=arch, features="halfkp" if arch == "simple" else features)
    c["ft_out"] = 128 * rng.randint(1, 4) if c["features"] == "halfkp" else 128 * rng.randint(1, 9)
    c.update(l1=rng.choice([8, 16, 32]), l2=rng.choice([16, 32, 64]),
             n=_log_int(rng, 512, 49152, 16 if arch == "layerstack" else 1),
             mixed=arch == "layerstack" and rng.random() < 0.4, factorize=rng.random() < 0.75,
             bucket="none" if arch == "simple" else rng.choice(["kingrank9", "progress8kpabs"]),
             loss=rng.choice(["sigmoid", "wrm", "wrm_ext"]))
    if kind == "train":
        c.update(steps=rng.randint(6, 16), resident=rng.random() < 0.7,
                 optimizer=rng.choice(["ranger", "radam", "adamw"] if arch == "layerstack" else ["radam", "adamw"]))
    else:
        c.update(resident=rng.random() < 0.5)
    return c


# ---------------------------------------------------------------------------
# positions
# ---------------------------------------------------------------------------

# piece types 1..7: pawn, lance, knight, silver, bishop, rook, gold; Huffman
# pattern (first bit lowest) and length, without promotion and colour
_PATTERN = (0, 0x01, 0x03, 0x0B, 0x07, 0x1F, 0x3F, 0x0F)
_LENGTH = (1, 2, 4, 4, 4, 6, 6, 5)
_PIECES = [6] * 2 + [5] * 2 + [7] * 4 + [4] * 4 + [3] * 4 + [2] * 4 + [1] * 18


def _records(n: int, seed: int) -> torch.Tensor:
    """[n, 40] uint8 PSV records of seeded positions, on the GPU."""
    g = torch.Generator(device=DEV).manual_seed(seed)

    def rand(*shape):
        return torch.rand(*shape, device=DEV, generator=g)

    def below(hi, *shape):
        return torch.randint(0, hi, shape, device=DEV, generator=g)

    types = torch.tensor(_PIECES, device=DEV)
    pattern, length = torch.tensor(_PATTERN, device=DEV), torch.tensor(_LENGTH, device=DEV)
    square = torch.argsort(rand(n, 81), dim=1)[:, :40]  # two kings, then the pieces
    owner = below(2, n, 38)
    in_hand = rand(n, 38) < 0.15
    gold = types == 7
    promoted = ((rand(n, 38) < 0.1) & ~gold).long()
    val, ln = pattern[types].expand(n, 38), length[types].expand(n, 38)
    # board: code, promotion bit (not gold), colour; an empty square is one 0 bit
    bval = torch.where(gold, val | (owner << ln), val | (promoted << ln) | (owner << (ln + 1)))
    blen = ln + torch.where(gold, 1, 2)
    board_v = torch.zeros(n, 82, dtype=torch.long, device=DEV)
    board_l = torch.ones(n, 82, dtype=torch.long, device=DEV)
    at = torch.where(in_hand, torch.full_like(owner, 81), square[:, 2:])
    board_v.scatter_(1, at, bval)
    board_l.scatter_(1, at, blen)
    board_l.scatter_(1, square[:, :2], 0)  # a king's square has no code
    # hand: the code without its first bit, a zero bit (not gold), colour
    hval = torch.where(gold, (val >> 1) | (owner << (ln - 1)), (val >> 1) | (owner << ln))
    hlen = torch.where(in_hand, ln + torch.where(gold, 0, 1), 0)
    one = torch.ones(n, 1, dtype=torch.long, device=DEV)
    v = torch.cat([below(2, n, 1), square[:, :2], board_v[:, :81], torch.where(in_hand, hval, 0)], 1)
    ln_all = torch.cat([one, 7 * one, 7 * one, board_l[:, :81], hlen], 1)
    off = torch.cumsum(ln_all, 1) - ln_all
    bits = torch.zeros(n, 257, dtype=torch.uint8, device=DEV)
    for j in range(8):
        bits.scatter_(1, torch.where(j < ln_all, off + j, 256), ((v >> j) & 1).to(torch.uint8))
    weight = 1 << torch.arange(8, device=DEV)
    out = torch.zeros(n, 40, dtype=torch.uint8, device=DEV)
    out[:, :32] = (bits[:, :256].view(n, 32, 8) * weight).sum(2).to(torch.uint8)
    score = (torch.randn(n, device=DEV, generator=g) * 600).round().clamp(-3000, 3000).long() & 0xFFFF
    out[:, 32], out[:, 33] = (score & 255).to(torch.uint8), (score >> 8).to(torch.uint8)
    out[:, 36] = below(256, n).to(torch.uint8)
    out[:, 38] = ((below(3, n) - 1) & 255).to(torch.uint8)
    return out


def _progress_weights(seed: int) -> np.ndarray:
    return np.random.default_rng(seed).normal(0.0, 0.1, KPABS_WEIGHTS)


def _num_buckets(mode: str) -> int:
    return {"kingrank9": 9, "progress8kpabs": 8, "none": 1}[mode]


def _batch(case: dict, seed: int) -> DeviceBatch:
    progress = ProgressWeights(_progress_weights(seed)) if case["bucket"] == "progress8kpabs" else None
    return psv_to_device_batch(_records(case["n"], seed).cpu().numpy(), case["features"], case["bucket"],
                               _num_buckets(case["bucket"]), progress)


def _host(batch: DeviceBatch) -> tuple[Batch, np.ndarray]:
    h = device_batch_to_host(batch)
    return Batch(h["stm"], h["nstm"], h["nnz"], h["score"], h["wdl"]), h["bucket"]


def _index_rows(case: dict, seed: int) -> dict:
    """Index rows of a batch as tensors on the GPU."""
    c = dict(case, bucket="none")
    h = device_batch_to_host(_batch(c, seed))
    return {k: torch.from_numpy(h[k]).to(DEV) for k in ("stm", "nstm", "nnz")}


def _normal(g, shape, std, mean=0.0) -> torch.Tensor:
    return torch.randn(shape, device=DEV, generator=g) * std + mean


# ---------------------------------------------------------------------------
# networks
# ---------------------------------------------------------------------------

def _shapes(case: dict) -> dict:
    """Parameter groups and their shapes, in the step API's order."""
    info = feature_set_info(case["features"])
    d, l1, l2 = case["ft_out"], case["l1"], case["l2"]
    rows = info["ft_in"] + (info["piece_inputs"] if case["factorize"] else 0)
    if case["arch"] == "simple":
        return dict(ft_w=(rows, d), ft_b=(d,), l1_w=(2 * d, l1), l1_b=(l1,), l2_w=(l1, l2), l2_b=(l2,),
                    l3_w=(l2, 1), l3_b=(1,))
    nb = _num_buckets(case["bucket"])
    return dict(ft_w=(rows, d), ft_b=(d,), l1_w=(nb, l1, d), l1_b=(nb, l1), l1_shared_weight=(d, l1),
                l1_shared_bias=(l1,), l2_w=(nb, l2, 2 * (l1 - 1)), l2_b=(nb, l2), l3_w=(nb, l2), l3_b=(nb,))


def _weights(case: dict, seed: int) -> dict:
    """Seeded weights of every group, f32 on the GPU."""
    g = torch.Generator(device=DEV).manual_seed(seed + 7)
    info, out = feature_set_info(case["features"]), {}
    for name, shape in _shapes(case).items():
        if name == "ft_w":
            w = _normal(g, shape, 0.04)
            w[info["ft_in"]:] *= 0.5
        elif name.endswith("_b") or name == "l1_shared_bias":
            w = _normal(g, shape, 0.05, 0.4 if name == "ft_b" else 0.1)
        else:
            fan = {"l1_w": case["ft_out"], "l1_shared_weight": case["ft_out"], "l2_w": 2 * case["l1"],
                   "l3_w": case["l2"]}[name]
            w = _normal(g, shape, 1.5 / math.sqrt(fan))
        out[name] = w.clamp(-1.9, 1.9)
    return out


def _loss(case: dict):
    if case["loss"] == "sigmoid":
        return Sigmoid(1.0 / 290.0) if case["arch"] == "layerstack" else Sigmoid(1.0)
    if case["loss"] == "wrm":
        return Wrm(nnue2score=290.0, in_scaling=290.0, in_offset=0.0, target_offset=0.0, target_scaling=290.0)
    return Wrm(pow_exp=2.5, qp_asymmetry=0.3, weight_boost_w1=0.5, weight_boost_w2=0.5)


LR = {"ranger": 8.75e-4, "radam": 8.75e-4, "adamw": 1e-3}


def _second_moment(name: str) -> float:
    """AdamW has no warm-up of its own, so its cases take a run that is under
    way: second moments of the gradients' size, the same in a group."""
    return 1e-6 if name == "ft_w" else 1e-2


def _trainer(case: dict):
    info = feature_set_info(case["features"])
    cfg = dict(ft_in=info["ft_in"], max_active=info["max_active"], ft_out=case["ft_out"], l1_out=case["l1"],
               piece_inputs=info["piece_inputs"] if case["factorize"] else 0, l2_out=case["l2"],
               max_batch=case["n"], optimizer=case.get("optimizer", "ranger"), weight_decay=0.01)
    if case["arch"] == "simple":
        return SimpleTrainer(SimpleConfig(**cfg))
    c = LayerStackConfig(num_buckets=_num_buckets(case["bucket"]), **cfg)
    return LayerStackTrainer(c.all_optim() if case["mixed"] else c)


def _read_back(t, name: str, out: torch.Tensor) -> None:
    """A group's weights into the program's own pinned array."""
    _lib.check(t._lib.tatara_trainer_get_tensor(t._h, name.encode(), 0, C.cast(out.data_ptr(), _lib.c_f32p),
                                                out.numel()))


def _ptr(t: torch.Tensor | None):
    return None if t is None else t.data_ptr()


# ---------------------------------------------------------------------------
# what a program holds before the call, and the call
# ---------------------------------------------------------------------------

def prepare(case: dict, seed: int) -> dict:
    info = feature_set_info(case["features"])
    kind, s = case["kind"], dict(case=case, info=info)
    g = torch.Generator(device=DEV).manual_seed(seed + 1)
    if kind == "decode":
        n, ma = case["n"], info["max_active"]
        s["psv"] = _records(n, seed)
        s["weights"] = (torch.from_numpy(_progress_weights(seed).astype(np.float32)).to(DEV)
                        if case["bucket"] == "progress8kpabs" else None)
        s["out"] = {k: torch.empty(shape, dtype=t, device=DEV) for k, shape, t in (
            ("stm", (n, ma), torch.int32), ("nstm", (n, ma), torch.int32), ("nnz", (n,), torch.int32),
            ("bucket", (n,), torch.int32), ("score", (n,), torch.float32), ("wdl", (n,), torch.float32))}
    elif kind == "ft_forward":
        n, d = case["n"], case["ft_out"]
        s["rows"] = _index_rows(case, seed)
        s["w"], s["b"] = _normal(g, (info["ft_in"], d), 0.04), _normal(g, (d,), 0.05, 0.4)
        s["out"] = {k: torch.empty(n, d, device=DEV) for k in ("stm", "nstm", "combined")}
    elif kind == "ft_grad":
        n, d = case["n"], case["ft_out"]
        s["rows"] = _index_rows(case, seed)
        # the gradient of the clipped activations: zero where they are clipped
        dft = _normal(g, (2, n, d), 1.0 / n) * (torch.rand(2, n, d, device=DEV, generator=g) < 0.7)
        s["inv"] = 1.0
        if case["half"]:
            scale = 16384.0 * n  # the mixed-precision step's loss scale
            s["inv"] = 1.0 / scale
            dft = (dft * 1e-3 * scale).half()
        s["dft"] = dft
        s["grad"] = torch.empty(info["ft_in"], d, device=DEV)
    elif kind == "export":
        rows = info["ft_in"] + (info["piece_inputs"] if case["factorize"] else 0)
        s["w"] = _normal(g, (rows, case["ft_out"]), 0.25)
        s["out"] = torch.zeros(info["ft_in"] * case["ft_out"] * (3 if case["leb128"] else 2), dtype=torch.uint8,
                               device=DEV)
    else:
        s["trainer"] = _trainer(case)
        weights = _weights(case, seed)
        s["read"] = {k: torch.empty(w.shape, pin_memory=True).copy_(w) for k, w in weights.items()}
        for k, w in s["read"].items():
            s["trainer"].set(k, w.numpy())
            if case.get("optimizer") == "adamw":
                s["trainer"].set(k, torch.full(w.shape, _second_moment(k), pin_memory=True).numpy(), "v")
        del weights
        dev = [_batch(case, seed + 100 * k) for k in range(BATCHES if kind == "train" else 1)]
        s["batches"] = [(b, None) if case["resident"] else _host(b) for b in dev]
        s["loss"] = _loss(case)
    # the library's own calls below run on the null stream and its trainers'
    torch.cuda.synchronize()
    return s


def run(s: dict):
    case, info, kind = s["case"], s["info"], s["case"]["kind"]
    lib = _lib.load()
    if kind == "decode":
        o = s["out"]
        _lib.check(lib.tatara_psv_to_batch(
            s["psv"].data_ptr(), case["n"], FEATURE_SETS[case["features"]], BUCKET_MODES[case["bucket"]],
            _num_buckets(case["bucket"]), _ptr(s["weights"]), o["stm"].data_ptr(), o["nstm"].data_ptr(),
            o["nnz"].data_ptr(), o["bucket"].data_ptr(), o["score"].data_ptr(), o["wdl"].data_ptr()))
        return o
    if kind == "ft_forward":
        r, o = s["rows"], s["out"]
        _lib.check(lib.tatara_op_ft_forward_pairwise(
            s["w"].data_ptr(), r["stm"].data_ptr(), r["nstm"].data_ptr(), r["nnz"].data_ptr(), s["b"].data_ptr(),
            o["stm"].data_ptr(), o["nstm"].data_ptr(), o["combined"].data_ptr(), case["n"], case["ft_out"],
            info["ft_in"], info["max_active"], info["piece_inputs"], FT_POST_SCALE))
        return o
    if kind == "ft_grad":
        r = s["rows"]
        head = [s["dft"].data_ptr()] + ([s["inv"]] if case["half"] else [])
        op = lib.tatara_op_ft_weight_grad_mfma_f16 if case["half"] else lib.tatara_op_ft_weight_grad_blocked
        _lib.check(op(*head, r["stm"].data_ptr(), r["nstm"].data_ptr(), r["nnz"].data_ptr(), s["grad"].data_ptr(),
                      case["n"], case["ft_out"], info["ft_in"], info["max_active"], info["piece_inputs"], None))
        return s["grad"]
    if kind == "export":
        n = C.c_uint64()
        _lib.check(lib.tatara_op_quantise_ft(
            s["w"].data_ptr(), info["ft_in"], case["ft_out"], info["piece_inputs"] if case["factorize"] else 0, 127.0,
            int(case["leb128"]), s["out"].data_ptr(), s["out"].numel(), C.byref(n)))
        return dict(table=s["out"], bytes=n.value)
    t = s["trainer"]
    if kind == "validate":
        (b, bucket), = s["batches"]
        return (t.validate_step(b, 0.25, s["loss"]) if case["arch"] == "simple"
                else t.validate_step(b, bucket, 0.25, s["loss"]))
    lr, total = LR[case["optimizer"]], 0.0
    for k in range(case["steps"]):
        b, bucket = s["batches"][k % len(s["batches"])]
        total += (t.train_step(b, lr, 0.25, s["loss"]) if case["arch"] == "simple"
                  else t.train_step(b, bucket, lr, 0.25, s["loss"]))
    total += t.flush_pending_loss()
    for name, out in s["read"].items():
        _read_back(t, name, out)
    return dict(loss=total, **s["read"])


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how close another one has to come
# ---------------------------------------------------------------------------

def work(case: dict) -> dict:
    info = feature_set_info(case["features"])
    ma, rows, kind = info["max_active"], info["ft_in"], case["kind"]
    if kind == "export":
        cells = rows * case["ft_out"]
        # most values take two bytes as LEB128
        return dict(bytes=cells * (4 + 2), flops=2 * cells)
    n = case["n"]
    inputs = n * (2 * 4 * ma + 4 * 4)
    if kind == "decode":
        return dict(bytes=n * 40 + inputs, flops=0)
    d = case["ft_out"]
    gathered = 2 * n * ma * d  # additions of one pass over the active features
    if kind == "ft_forward":
        return dict(bytes=4 * rows * d + inputs + 3 * 4 * n * d, flops=gathered)
    if kind == "ft_grad":
        return dict(bytes=4 * rows * d + inputs + (2 if case["half"] else 4) * 2 * n * d, flops=gathered)
    sizes = {k: math.prod(v) for k, v in _shapes(case).items()}
    dense_in = 2 * d if case["arch"] == "simple" else d
    mults = 2 * n * dense_in * case["l1"] * (1 if case["arch"] == "simple" else 2) + 2 * n * 2 * case["l1"] * case["l2"]
    if kind == "validate":
        table = min(sizes["ft_w"], 2 * n * ma * d)  # the rows that are read
        return dict(bytes=4 * table + inputs + 4 * n, flops=gathered + mults)
    p = sum(sizes.values())
    # weights and both moments read and written in every step, then the weights read back
    state = 2 * (4 * p + (2 if case["mixed"] else 4) * 2 * p)
    return dict(bytes=case["steps"] * (state + inputs) + 4 * p, flops=case["steps"] * (2 * gathered + 3 * mults))


def tolerance(case: dict):
    """Four times, or more, what was seen against 64 bits and between orders of the same sums."""
    kind = case["kind"]
    if kind in ("decode", "export"):
        return "exact"
    if kind in ("ft_forward", "ft_grad"):
        return dict(rel=1e-6, max=1e-4)
    if case["mixed"]:  # one f16 step of an activation travels on
        return dict(rel=2e-3)
    return dict(rel=4e-6) if kind == "validate" else dict(rel=2e-4)


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

class _Blocks:
    """The rows of each king block: their 0/1 matrices and its part of the table."""

    def __init__(self, info: dict, index: torch.Tensor, nnz: torch.Tensor):
        self.pi, self.cells = info["piece_inputs"], info["ft_in"]
        index = torch.where(torch.arange(index.shape[1], device=DEV) < nnz[:, None], index.long(), -1)
        block = index[:, 0].div(self.pi, rounding_mode="floor")
        self.n, self.parts = index.shape[0], []
        for k in range(info["king_buckets"]):
            at = (block == k).nonzero()[:, 0]
            self.parts.append((k, at, index[at]))

    def _hits(self, k, index):
        h = torch.zeros(index.shape[0], self.pi + 1, dtype=torch.float64, device=DEV)
        h.scatter_(1, torch.where(index >= 0, index - k * self.pi, self.pi), 1.0)
        return h[:, : self.pi]

    def forward(self, w):
        out = torch.zeros(self.n, w.shape[1], dtype=torch.float64, device=DEV)
        for k, at, index in self.parts:
            if at.numel():
                out[at] = self._hits(k, index) @ w[k * self.pi:(k + 1) * self.pi]
        return out

    def backward(self, dft, grad):
        for k, at, index in self.parts:
            if at.numel():
                grad[k * self.pi:(k + 1) * self.pi] += self._hits(k, index).T @ dft[at]


def _pairs(raw, bias):
    x = (raw + bias).clamp(0, 1)
    half = x.shape[1] // 2
    return x[:, :half] * x[:, half:] * FT_POST_SCALE


def _net(case, p, raw_s, raw_n, bucket):
    if case["arch"] == "simple":
        x = torch.cat([(raw_s + p["ft_b"]).clamp(0, 1), (raw_n + p["ft_b"]).clamp(0, 1)], 1)
        x = (x @ p["l1_w"] + p["l1_b"]).clamp(0, 1)
        x = (x @ p["l2_w"] + p["l2_b"]).clamp(0, 1)
        return (x @ p["l3_w"] + p["l3_b"])[:, 0]
    x = torch.cat([_pairs(raw_s, p["ft_b"]), _pairs(raw_n, p["ft_b"])], 1)
    shared = x @ p["l1_shared_weight"] + p["l1_shared_bias"]
    net = torch.zeros(x.shape[0], dtype=torch.float64, device=DEV)
    for k in range(p["l1_w"].shape[0]):
        at = (bucket == k).nonzero()[:, 0]
        total = x[at] @ p["l1_w"][k].T + p["l1_b"][k] + shared[at]
        main, skip = total[:, :-1], total[:, -1]
        y = torch.cat([main * main * L1_SQR_SCALE, main], 1).clamp(0, 1)
        y = (y @ p["l2_w"][k].T + p["l2_b"][k]).clamp(0, 1)
        net = net.index_add(0, at, y @ p["l3_w"][k] + p["l3_b"][k] + skip)
    return net


def _position_losses(loss, net, score, wdl, lam):
    if isinstance(loss, Sigmoid):
        target = lam * wdl + (1 - lam) * torch.sigmoid(score * loss.scale)
        return (torch.sigmoid(net * loss.scale) - target) ** 2
    t = 0.5 * (1 + torch.sigmoid((score - loss.target_offset) / loss.target_scaling)
               - torch.sigmoid((-score - loss.target_offset) / loss.target_scaling))
    target = lam * wdl + (1 - lam) * t
    s = net * loss.nnue2score
    pred = 0.5 * (1 + torch.sigmoid((s - loss.in_offset) / loss.in_scaling)
                  - torch.sigmoid((-s - loss.in_offset) / loss.in_scaling))
    err = pred - target
    if not loss.extended:
        return err ** 2
    weight = 1 + (2.0 ** loss.weight_boost_w1 - 1) * ((t - 0.5) ** 2 * t * (1 - t)) ** loss.weight_boost_w2
    asym = torch.where(pred > target, 1.0 + loss.qp_asymmetry, 1.0)
    return asym * err.abs() ** loss.pow_exp * weight * (net.shape[0] / weight.sum())


def _step_size(optimizer: str, step: int) -> tuple[float, bool, float]:
    """RAdam's scalars, which the reference computes once a step in f32: (step size, divide, beta1)."""
    f, beta1, beta2 = np.float32, np.float32(0.99 if optimizer == "ranger" else 0.9), np.float32(0.999)
    if optimizer == "adamw":
        return 1.0, True, float(beta1)
    bt = np.power(beta2, f(step), dtype=f)
    most = f(2) / (f(1) - beta2) - f(1)
    sma = most - f(2) * f(step) * bt / (f(1) - bt)
    bc = f(1) - np.power(beta1, f(step), dtype=f)
    if sma > f(5):
        r = np.sqrt((f(1) - bt) * ((sma - f(4)) / (most - f(4))) * ((sma - f(2)) / sma) * (most / (most - f(2))))
        return float(r / bc), True, float(beta1)
    return float(f(1) / bc), False, float(beta1)


def _update(case, p, m, v, slow, grads, step):
    size, divide, beta1 = _step_size(case["optimizer"], step)
    beta2, eps, lr = float(np.float32(0.999)), float(np.float32(1e-8)), float(np.float32(LR[case["optimizer"]]))
    rate, decay = lr * size, float(np.float32(0.01))
    free = ("ft_w", "ft_b", "l3_b")
    for k in p:
        g = grads.pop(k)
        m[k].mul_(beta1).add_(g, alpha=1 - beta1)
        v[k].mul_(beta2).addcmul_(g, g, value=1 - beta2)
        step_k = m[k] / (v[k].sqrt() + eps) if divide else m[k]
        p[k].mul_(1 - decay * rate).sub_(step_k, alpha=rate)
        if k not in free:
            p[k].clamp_(-QUANT_CLAMP, QUANT_CLAMP)
        if case["optimizer"] == "ranger" and step % 6 == 0:
            p[k].add_(slow[k]).mul_(0.5)
            slow[k].copy_(p[k])


def _train_exact(case: dict, seed: int):
    info, loss, lam = feature_set_info(case["features"]), _loss(case), 0.25
    p = {k: w.double() for k, w in _weights(case, seed).items()}
    train = case["kind"] == "train"
    m, v, slow = ({k: torch.zeros_like(w) for k, w in p.items()} if train else {} for _ in range(3))
    if case.get("optimizer") == "adamw":
        v = {k: torch.full_like(w, float(np.float32(_second_moment(k)))) for k, w in p.items()}
    batches = []
    for k in range(BATCHES if train else 1):
        h = {a: torch.from_numpy(x).to(DEV) for a, x in device_batch_to_host(_batch(case, seed + 100 * k)).items()}
        batches.append((h, _Blocks(info, h["stm"], h["nnz"]), _Blocks(info, h["nstm"], h["nnz"])))
    cells, pi, total = info["ft_in"], info["piece_inputs"], 0.0
    for step in range(1, case.get("steps", 1) + 1):
        h, bs, bn = batches[(step - 1) % len(batches)]
        table = p["ft_w"][:cells]
        if case["factorize"]:
            table = (table.view(-1, pi, case["ft_out"]) + p["ft_w"][cells:]).view(cells, -1)
        leaf = {k: w.detach().requires_grad_(train) for k, w in p.items() if k != "ft_w"}
        raw_s, raw_n = (b.forward(table).requires_grad_(train) for b in (bs, bn))
        net = _net(case, leaf, raw_s, raw_n, h["bucket"])
        each = _position_losses(loss, net, h["score"].double(), h["wdl"].double(), lam)
        if not train:
            return (float(each.detach().sum()), net)
        total += float(each.detach().sum())
        (each.sum() / case["n"]).backward()
        grads = {k: w.grad for k, w in leaf.items()}
        gw = torch.zeros_like(p["ft_w"])
        bs.backward(raw_s.grad, gw)
        bn.backward(raw_n.grad, gw)
        if case["factorize"]:
            gw[cells:] = gw[:cells].view(-1, pi, case["ft_out"]).sum(0)
        grads["ft_w"] = gw
        del raw_s, raw_n, net, each, table, leaf
        _update(case, p, m, v, slow, grads, step)
    return dict(loss=total, **p)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("decode", "export"):
        return None  # whole numbers and bytes
    if kind in ("train", "validate"):
        with torch.enable_grad():
            return _train_exact(case, seed)
    s = prepare(case, seed)
    bs, bn = (_Blocks(s["info"], s["rows"][k], s["rows"]["nnz"]) for k in ("stm", "nstm"))
    if kind == "ft_forward":
        raw = [b.forward(s["w"].double()) for b in (bs, bn)]
        return dict(stm=raw[0], nstm=raw[1], combined=torch.cat([_pairs(r, s["b"].double()) for r in raw], 1))
    grad = torch.zeros(s["grad"].shape, dtype=torch.float64, device=DEV)
    bs.backward(s["dft"][0].double(), grad)
    bn.backward(s["dft"][1].double(), grad)
    return grad * s["inv"]

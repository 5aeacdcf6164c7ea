"""PSV decode at the edges of a workgroup and of a record (GPU): record counts
around the 64 a workgroup takes, and records whose codes fill the 256 bits
with board pieces, with hand pieces, or end inside a code.  Every feature set
and bucket mode, bit for bit against the CPU feature oracle."""
import numpy as np
import pytest

from tatara_amd import psv

from test_gpu_features import FS, compare

pytestmark = pytest.mark.gpu


def crafted():
    """Valid kings, then every repeated code of up to eight bits."""
    recs = []
    for length in (1, 2, 3, 4, 5, 6, 7, 8):
        for pattern in range(1 << length):
            if length > 5 and pattern % 7:
                continue
            bits = np.zeros(256, np.uint8)
            head = 1 | (40 << 1) | ((pattern % 81) << 8)
            bits[:15] = [(head >> i) & 1 for i in range(15)]
            bits[15:] = [(pattern >> (i % length)) & 1 for i in range(241)]
            rec = np.zeros(40, np.uint8)
            rec[:32] = np.packbits(bits, bitorder="little")
            rec[32:] = (pattern * 37 + length) % 251
            recs.append(rec)
    return np.stack(recs)


def full_hands():
    """An empty board and one hand of every count of one piece, up to a record's
    room.  From three rooks on, the hand's feature is no longer below the board's
    first (90), where the reference mirrors it like a board piece's."""
    codes = {2: [1, 0, 0], 4: [1, 1, 0], 5: [1, 1, 1, 0], 6: [1, 1, 1, 1, 0], 7: [1, 1, 1, 1, 1]}  # first bit lowest
    recs = []
    for piece, code in codes.items():
        entry = code + ([] if piece == 5 else [0])  # not in the piece box (gold has no such bit)
        for owner in (0, 1):
            for count in range(1, 162 // (len(entry) + 1) + 1):
                kings = (count * 7 % 81, (count * 31 + 40) % 81)
                head = (count & 1) | kings[0] << 1 | kings[1] << 8
                bits = [(head >> i) & 1 for i in range(15)] + [0] * (81 - len(set(kings)))
                bits += (entry + [owner]) * count
                bits += [0, 1, 0] * 60  # pawns in the piece box
                rec = np.zeros(40, np.uint8)
                rec[:32] = np.packbits(np.array(bits[:256], np.uint8), bitorder="little")
                recs.append(rec)
    return np.stack(recs)


@pytest.mark.parametrize("fs", FS)
def test_hands_of_any_count(gpu, fs):
    compare(full_hands(), fs, "none")
    compare(full_hands(), fs, "progress", 9, np.random.default_rng(3).normal(0.0, 0.05, 81 * 1548))


@pytest.mark.parametrize("fs", FS)
def test_record_counts_and_full_records(gpu, fs):
    rng = np.random.default_rng(9)
    weights = rng.normal(0.0, 0.05, 81 * 1548)
    rnd = rng.integers(0, 256, (160, 40), dtype=np.uint8)
    rnd[:, :2] = psv.synthetic_psv(160, seed=3)[:, :2]  # valid kings
    rnd[::2, 2:12] = 0  # a nearly empty board: hands fill the record
    recs = np.concatenate([crafted(), rnd, psv.synthetic_psv(64, seed=4)])
    for n in (1, 63, 64, 65, 129, len(recs)):
        compare(recs[-n:], fs, "none")
        compare(recs[:n], fs, "kingrank9")
        compare(recs[:n], fs, "progress", 9, weights)

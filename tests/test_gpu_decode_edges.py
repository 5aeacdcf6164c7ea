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

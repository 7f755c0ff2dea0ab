"""The heap replay of tied bf16 rows (csrc/g4s_heap.h) against the oracle's
DoSelectTopKIndices: heaps held in the lanes (K <= 64), in LDS and in device
memory, at the sizes where their layout changes, on rows whose insertions are
few (random), dense ties, or every element (ascending: the screened segments
overflow), and rows with NaNs (one element at a time).  Everything must
equal the oracle's bits.
"""
import numpy as np
import pytest

from gemma4_sampler import hip, native
from test_gpu_wide import _params, _run, _widen

pytestmark = pytest.mark.gpu
F32 = np.float32
CAP = 30.0


def _rows(rng, n, vocab):
    """bf16-valued rows: peaky random, ascending, few levels, ascending with
    plateaus and late larger values."""
    rows = np.empty((n, vocab), F32)
    for r in range(n):
        kind = r % 4
        if kind == 0:
            rows[r] = rng.normal(0, 3, vocab)
        elif kind == 1:
            rows[r] = np.sort(rng.normal(0, 3, vocab))
        elif kind == 2:
            rows[r] = rng.integers(0, 4, vocab)
            rows[r][rng.random(vocab) < 0.2] = -np.inf
        else:
            rows[r] = np.floor(np.arange(vocab) * 40.0 / vocab)
            rows[r][rng.choice(vocab, max(1, vocab // 50))] = 41.0
    return _widen((rows.view(np.uint32) >> 16).astype(np.uint16))


@pytest.mark.parametrize("batch", [8, 12])  # both top-k launches
@pytest.mark.parametrize("vocab, ks", [
    (70, [2, 3, 31, 32, 33, 62, 63, 64]),
    (1031, [2, 20, 63, 64, 65, 127, 128, 129]),
    (5003, [33, 64, 65, 200, 255, 256, 257, 1000]),
    (20011, [40, 64, 511, 512, 513, 1022, 1023, 1024]),
])
def test_replay_sizes(orc, vocab, ks, batch):
    rng = np.random.default_rng(vocab + batch)
    rows = _rows(rng, batch, vocab)
    u = np.floor(rng.random(batch) * 2**32) / 2**32
    t = np.full(batch, 0.7, F32)
    p = np.full(batch, 0.95, F32)
    seen = 0
    for i in range(2):
        k = np.array([ks[(r + 3 * i) % len(ks)] for r in range(batch)], np.int32)
        seen |= _run(orc, rows, t, k, p, u, CAP, "bf16", f"V={vocab}", capacity=1024)
        small = np.minimum(k, 64).astype(np.int32)
        seen |= _run(orc, rows, t, small, p, u, CAP, "bf16", f"V={vocab} K<=64", capacity=64)
    assert seen & native.FLAG_HEAP_REPLAY


@pytest.mark.parametrize("vocab, ks", [
    (6007, [1025, 1026, 4000, 6006]),
    (40009, [15355, 15356, 15357, 20001]),  # the last heaps of LDS, the first of device memory
])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_replay_wide(orc, vocab, ks, dtype):
    rng = np.random.default_rng(vocab)
    rows = _rows(rng, 8, vocab)
    k = np.array([ks[r % 4] for r in range(4)] + [ks[(r + 1) % 4] for r in range(4)], np.int32)
    u = np.floor(rng.random(8) * 2**32) / 2**32
    seen = _run(orc, rows, np.ones(8, F32), k, np.full(8, 0.9, F32), u, CAP, dtype, f"V={vocab}")
    assert seen & native.FLAG_HEAP_REPLAY


@pytest.mark.parametrize("vocab, nans, ks", [
    (3001, [1, 2, 3, 4, 5, 6, 7, 8], [5, 20, 63, 64, 2, 40, 64, 33]),
    (100003, [4, 16, 16, 32, 64, 64, 16, 512], [5, 20, 64, 20, 65, 200, 2, 1000]),
    (262144, [4, 16, 16, 16, 64, 64, 16, 64], [5, 20, 20, 20, 64, 128, 5, 20]),
])
@pytest.mark.parametrize("batch", [8, 16])  # both top-k launches
def test_replay_nan(orc, vocab, nans, ks, batch):
    """The reference's comparisons let a NaN into the heap, where it breaks the
    order: later insertions can lift it to the root, which then falls again.
    From a row's first NaN on, every element meets the root of its own turn."""
    rng = np.random.default_rng(vocab + batch)
    rows = _widen((rng.normal(0, 3, (batch, vocab)).astype(F32).view(np.uint32) >> 16)
                  .astype(np.uint16))
    for r in range(batch):
        rows[r, rng.choice(vocab, nans[r % 8])] = np.nan
    k = np.array([ks[r % 8] for r in range(batch)], np.int32)
    stride = (vocab + 7) // 8 * 8
    b16 = np.full((batch, stride), 0xFF80, np.uint16)
    b16[:, :vocab] = rows.view(np.uint32) >> 16
    s = native.Sampler(vocab, max_batch=batch, softcap=CAP)
    d = hip.Buffer.from_array(b16)
    outs = native.DeviceOutputs(batch, 1024)
    s.sample(d, batch, _params(np.ones(batch), k, np.ones(batch)), np.full(batch, 0.5),
             row_stride=stride, outputs=outs.struct, dtype=native.DTYPE_BF16, check=False)
    o = outs.read()
    s.close()
    replayed, bad = 0, []
    for r in range(batch):
        if o["flags"][r] & native.FLAG_HEAP_REPLAY:
            want = orc.select_topk_indices(rows[r], int(k[r]))
            replayed += 1
            if o["count"][r] != len(want) or not np.array_equal(o["indices"][r][:len(want)], want):
                bad.append((r, int(k[r])))
    assert replayed and not bad, f"{len(bad)} of {replayed} rows differ: {bad}"

"""The heap replay of tied bf16 rows (csrc/g4s_heap.h) against the oracle's
DoSelectTopKIndices: heaps held in the lanes (K <= 64), in LDS and in device
memory, at the sizes where their layout changes, on rows whose insertions are
few (random), dense ties, or every element (ascending: the screened segments
overflow), and rows with NaNs (the lanes' heap moves to LDS).  Everything must
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


def test_replay_nan(orc):
    """The reference's comparisons let a NaN into the heap, where it sinks to
    a leaf and breaks the order: the replay makes them one by one."""
    vocab, B = 3001, 8
    rng = np.random.default_rng(3)
    rows = _rows(rng, B, vocab)
    for r in range(B):
        rows[r, rng.choice(vocab, 1 + r)] = np.nan
    k = np.array([5, 20, 63, 64, 2, 40, 64, 33], np.int32)
    b16 = np.full((B, 3008), 0xFF80, np.uint16)
    b16[:, :vocab] = rows.view(np.uint32) >> 16
    s = native.Sampler(vocab, max_batch=B, softcap=CAP)
    d = hip.Buffer.from_array(b16)
    outs = native.DeviceOutputs(B, 64)
    s.sample(d, B, _params(np.ones(B), k, np.ones(B)), np.full(B, 0.5), row_stride=3008,
             outputs=outs.struct, dtype=native.DTYPE_BF16, check=False)
    o = outs.read()
    replayed = 0
    for r in range(B):
        if o["flags"][r] & native.FLAG_HEAP_REPLAY:
            want = orc.select_topk_indices(rows[r], int(k[r]))
            assert o["count"][r] == len(want)
            assert np.array_equal(o["indices"][r][:len(want)], want), r
            replayed += 1
    s.close()
    assert replayed

"""GPU parity of the Q4_0 LM head (g4s_lmhead_q4_0) against the oracle's
CpuMatVecQ4 restatement (src/Gemma4.Tensors.pas:546-598), and of the
LM head + sampler workload (B=32 hidden vectors, 262144 x 2560 weights, the
decode-stream sampling settings) through the C ABI.

Logits must equal the oracle's bit for bit: the kernel evaluates every
term in the reference's order with one binary32 fma, which is what the
reference's Extended-precision step rounds to for these magnitudes.  The
sampled ids are then the sampler's, compared against the oracle sampler on
the same logits.
"""
import numpy as np
import pytest

from gemma4_sampler import hip, native, workload as wl

pytestmark = pytest.mark.gpu
F32 = np.float32
D = wl.HIDDEN_GEMMA4
V = wl.V_GEMMA4


def _lmhead(s, w_host_or_buf, rows, cols, hidden):
    B = hidden.shape[0]
    dw = w_host_or_buf if isinstance(w_host_or_buf, hip.Buffer) else \
        hip.Buffer.from_array(w_host_or_buf)
    dh = hip.Buffer.from_array(np.ascontiguousarray(hidden, F32))
    dl = hip.Buffer(4 * B * rows)
    s.lmhead_q4_0(dw, rows, cols, dh, B, dl, rows)
    hip.synchronize()
    return dl.download(F32).reshape(B, rows)


@pytest.mark.parametrize("batch", [1, 5, 32, 40])
def test_lmhead_small_bit_exact(orc, batch):
    rows, cols = 700, D
    w = wl.host_q4_weights(77, rows, cols)
    hidden = wl.host_hidden(78 + batch, batch, cols)
    s = native.Sampler(V, max_batch=1, softcap=30.0)
    got = _lmhead(s, w, rows, cols, hidden)
    want = orc.matvec_q4_batch(w, hidden, rows, cols)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), \
        f"{np.sum(got != want)} logits differ"
    s.close()


def test_lmhead_odd_block_count_and_unaligned_hidden(orc):
    """An odd number of Q4_0 blocks per row and a hidden matrix that starts 4
    bytes past a 16-byte boundary."""
    rows, cols, B = 300, 5 * 32, 3
    w = wl.host_q4_weights(81, rows, cols)
    hidden = wl.host_hidden(82, B, cols)
    s = native.Sampler(V, max_batch=1, softcap=30.0)
    dw = hip.Buffer.from_array(w)
    dh = hip.Buffer(4 * (B * cols + 1))
    dh.upload(np.ascontiguousarray(hidden, F32), offset=4)
    dl = hip.Buffer(4 * B * rows)
    s.lmhead_q4_0(dw, rows, cols, dh.offset(4), B, dl, rows)
    hip.synchronize()
    got = dl.download(F32).reshape(B, rows)
    want = orc.matvec_q4_batch(w, hidden, rows, cols)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), \
        f"{np.sum(got != want)} logits differ"
    s.close()


@pytest.mark.parametrize("rows, cols, batches", [
    (1, 32, [1, 5]), (63, 16 * 32, [1, 33]),               # fewer rows than a wave has
    (64, 15 * 32, [1, 2]), (65, 17 * 32, [1, 3]),          # a partial and a second stage of blocks
    (127, 33 * 32, [1, 9]), (64 * 3 + 1, 32, [7]),         # odd row pitch; rows shorter than a stage
    (64 * 100, 7 * 32, [10, 11, 48, 70]),                  # several slices of the batch
    # more row groups than SIMDs: two vectors a wave, then 4 * NG with NG = 1..8 and two passes
    (64 * 1025 + 3, 3 * 32, [1, 2, 3, 5, 9, 13, 17, 21, 25, 32, 33]),
    (64 * 1025, 18 * 32, [1, 2, 8, 32]),
])
@pytest.mark.parametrize("shift", [0, 2, 5])
def test_lmhead_rows_splits(orc, rows, cols, batches, shift):
    """Every split of rows and vectors over waves, stages that the block count
    does not fill, rows that start on any byte, and weights that fill their
    buffer to the last byte."""
    if shift == 5 and rows > 1000:
        pytest.skip("the same kernels as shift 2")
    w = wl.host_q4_weights(rows + cols, rows, cols)
    hidden = wl.host_hidden(rows, max(batches), cols)
    want = orc.matvec_q4_batch(w, hidden, rows, cols, threads=8)
    s = native.Sampler(V, max_batch=1, softcap=30.0)
    dw = hip.Buffer(w.nbytes + shift)
    dw.upload(w, offset=shift)
    dh = hip.Buffer(4 * (hidden.size + 1))
    dh.upload(np.ascontiguousarray(hidden, F32), offset=4)
    stride = rows + 1
    for B in batches:
        dl = hip.Buffer.from_array(np.full((B, stride), 7.0, F32))
        s.lmhead_q4_0(dw.offset(shift), rows, cols, dh.offset(4), B, dl, stride)
        hip.synchronize()
        got = dl.download(F32).reshape(B, stride)
        bad = got[:, :rows].view(np.uint32) != want[:B].view(np.uint32)
        assert not bad.any(), f"B={B}: {bad.sum()} logits differ"
        assert np.all(got[:, rows] == 7.0)
    s.close()


def test_lmhead_scale_edge_cases(orc):
    """fp16 scales that are zero, subnormal (the reference's own decoding of
    them, Types.pas:452-466), the largest finite, and negative; tiny and
    large hidden values."""
    rows, cols = 64, 256
    rng = np.random.default_rng(5)
    w = wl.host_q4_weights(79, rows, cols).reshape(rows * cols // 32, 18)
    specials = [0x0000, 0x8000, 0x0001, 0x0200, 0x03FF, 0x8155, 0x0400, 0x7BFF, 0xFBFF, 0x3C00]
    for i in range(w.shape[0]):
        if i % 3 == 0:
            v = specials[(i // 3) % len(specials)]
            w[i, 0], w[i, 1] = v & 0xFF, v >> 8
    w = w.reshape(-1)
    hidden = rng.normal(0, 1, (3, cols)).astype(F32)
    hidden[1] *= 1e-20
    hidden[2] *= 1e3
    s = native.Sampler(V, max_batch=1, softcap=30.0)
    got = _lmhead(s, w, rows, cols, hidden)
    want = orc.matvec_q4_batch(w, hidden, rows, cols)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    s.close()


@pytest.mark.parametrize("batch", [1, 2, 3, 9, 13, 17, 25, 30])
@pytest.mark.parametrize("rows", [64, 64 * 1025 + 5])  # a vector a wave and all of them
@pytest.mark.parametrize("layout", ["rows", "tiled"])
def test_lmhead_infinite_scales(orc, layout, rows, batch):
    """Infinite and NaN scales: (nibble - 8) * s is an infinity, NaN for nibble
    8; the rows beside them keep their sums."""
    cols = 3 * 32
    w = wl.host_q4_weights(83, rows, cols).reshape(rows, 3, 18)
    rng = np.random.default_rng(6)
    w[:, 1, 2:] = rng.choice([0x99, 0xA9, 0xFB], (rows, 16))                  # 1..7: one sign
    w[8::16, 1, 2:] = rng.choice([0x91, 0x28, 0xF0], (len(w[8::16]), 16))     # mixed signs, zeros
    for i, v in enumerate([0x7C00, 0xFC00, 0x7E00, 0x7BFF]):
        w[i::8, 1, 0], w[i::8, 1, 1] = v & 0xFF, v >> 8
    hidden = np.abs(rng.normal(0, 1, (batch, cols))).astype(F32)
    hidden[1::3] *= -1
    s = native.Sampler(V, max_batch=1, softcap=30.0)
    if layout == "rows":
        got = _lmhead(s, w.reshape(-1), rows, cols, hidden)
    else:
        src = hip.Buffer.from_array(w.reshape(-1))
        tiles = hip.Buffer(native.q4_0_device_bytes(rows, cols, native.Q4_LAYOUT_TILED64))
        native.q4_0_repack(src, rows, cols, tiles)
        dh = hip.Buffer.from_array(hidden)
        dl = hip.Buffer(4 * batch * rows)
        s.lmhead_q4_0_tiled(tiles, rows, cols, dh, batch, dl, rows)
        hip.synchronize()
        got = dl.download(F32).reshape(batch, rows)
    s.close()
    want = orc.matvec_q4_batch(w.reshape(-1), hidden, rows, cols, threads=8)
    nan = np.isnan(want)
    assert nan.any() and np.isposinf(want).any() and (batch < 2 or np.isneginf(want).any())
    assert np.array_equal(np.isnan(got), nan)
    bad = got.view(np.uint32)[~nan] != want.view(np.uint32)[~nan]
    assert not bad.any(), f"{bad.sum()} logits differ"


def test_lmhead_hand_built_blocks():
    """Hand-built Q4_0 blocks with written-out expected logits: byte j holds
    element 2j in its low nibble and 2j+1 in its high nibble (Tensors.pas:
    581-593), and the row sum runs left to right in binary32."""
    cols = 32
    w = np.frombuffer(bytes([0x00, 0x3C, 0x9A, 0x0F, 0xF0] + [0x88] * 13) +
                      bytes([0x00, 0x3C, 0x99, 0x79] + [0x88] * 14), np.uint8)
    h = np.zeros((2, cols), F32)
    h[0, :6] = [1, 10, 100, 1000, 0.5, 0.25]     # row 0 weights 2, 1, 7, -8, -8, 7
    h[1, :4] = [2.0 ** 24, 1.0, 1.0, 2.0 ** 24]   # row 1 weights 1, 1, 1, -1
    s = native.Sampler(V, max_batch=1, softcap=30.0)
    got = _lmhead(s, w, 2, cols, h)
    # 2 + 10 + 700 - 8000 - 4 + 1.75; ((2^24 + 1) + 1) - 2^24 = 0 left to right
    assert got[0, 0] == F32(-7290.25) and got[1, 1] == F32(0.0), got
    s.close()


def test_lmhead_plus_sampler_full_size(orc):
    """The full LM head + sampler workload: 32 hidden vectors ~ N(0,1),
    262144 x 2560 Q4_0 weights (generated on the device and, bit-identically,
    on the host), T=0.7, K=64, P=0.95.  Every one of the 32 x 262144 logits
    is checked against the oracle's CpuMatVecQ4, and every sampled id against
    the oracle's DoSample applied to the oracle's own logits (end to end)."""
    B, rows, cols = 32, V, D
    nblocks = rows * (cols // 32)
    dw = hip.Buffer(nblocks * 18)
    wl.dev_q4_weights(dw, 80, rows, cols)
    hidden = wl.host_hidden(81, B, cols)
    s = native.Sampler(V, max_batch=B, softcap=30.0)
    logits = _lmhead(s, dw, rows, cols, hidden)
    w_host = wl.host_q4_weights(80, rows, cols, threads=16)
    want = orc.matvec_q4_batch(w_host, hidden, rows, cols, threads=16)
    del w_host
    nbad = int(np.sum(logits.view(np.uint32) != want.view(np.uint32)))
    assert nbad == 0, f"{nbad} of {B * rows} logits differ from CpuMatVecQ4"
    # sampling on the device-resident logits
    dl = hip.Buffer.from_array(logits)
    t = np.full(B, 0.7, F32)
    k = np.full(B, 64, np.int32)
    p = np.full(B, 0.95, F32)
    u = wl.host_row_u(82, 0, B)
    _, ids = s.sample(dl, B, [native.TSamplingParams.make(0.7, 64, 0.95)] * B, u)
    want_ids = orc.sample_batch(want, 0, V, V, (t, k, p), u, softcap=30.0, threads=16)
    assert np.array_equal(ids, want_ids), (ids, want_ids)
    print(f"LM head + sampler: {B * rows} logits and {B} ids bit-exact end to end")
    s.close()

"""Performance cases of the sampler library: what a decode loop or a serving
loop asks of it, through the public Python binding (gemma4_sampler.native)
over the C ABI.

Kinds of case:
  topk    sample rows of logits with 0 < TopK <= 1024 (the default setting is
          TopK 64 of TSamplingParams)
  wide    sample with TopK above g4s_max_top_k()
  full    sample with TopK disabled: softmax and draw over the vocabulary
  lmhead  the Q4_0 LM head, on TILED64 weights or on the engine's own rows
  fused   LM head + sample in one call, with or without the logits written
  step    a decode step's tail: embedding lookup of the last tokens, then the
          fused LM head + sample on the result

call "sync" is g4s_sample_ex (host parameters in, ids out on return), "async"
is the stream-ordered entry point that a serving loop uses, with parameters
on the device.  The library promises the reference's bits, so every case is
compared exactly.
"""
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "gemma4.pas_amd"))

from gemma4_sampler import native  # noqa: E402

V = 262144      # the model's vocabulary
HIDDEN = 2560   # and hidden size
CAP = 30.0      # final logit softcap
DEVICE = "cuda"


def listed():
    return [
        # one sequence, one token: the call the engine makes per decode step
        dict(name="topk_b1_f32", kind="topk", call="sync", dtype="f32", dist="peaky", vocab=V,
             batch=1, k=64),
        # a few sequences of a smaller, odd vocabulary, bf16 logits, survivors wanted
        dict(name="topk_b5_bf16_odd", kind="topk", call="async", dtype="bf16", dist="peaky",
             vocab=100003, batch=5, k=40),
        # a serving batch whose requests all bring their own settings (k 0: mixed 1/20/64/256)
        dict(name="topk_b64_mixed_f32", kind="topk", call="async", dtype="f32", dist="peaky",
             vocab=V, batch=64, k=0),
        # a request with a very large TopK next to nobody else
        dict(name="wide_b4_f32", kind="wide", call="async", dtype="f32", dist="peaky", vocab=V,
             batch=4, k=4000),
        # pure nucleus sampling of one sequence on the engine's fp32 logits
        dict(name="full_b1_f32", kind="full", call="sync", dtype="f32", dist="peaky", vocab=V,
             batch=1, probs=False),
        # the same for a batch, odd vocabulary, every probability returned
        dict(name="full_b24_f32_odd", kind="full", call="async", dtype="f32", dist="peaky",
             vocab=100003, batch=24, probs=True),
        # a large serving batch on flat bf16 logits
        dict(name="full_b256_bf16", kind="full", call="async", dtype="bf16", dist="flat", vocab=V,
             batch=256, probs=False),
        # LM head of one sequence's decode step on the repacked weights
        dict(name="lmhead_b1", kind="lmhead", layout="tiled", vocab=V, cols=HIDDEN, batch=1),
        # the same on the weights as the engine stores them
        dict(name="lmhead_rows_b1", kind="lmhead", layout="rows", vocab=V, cols=HIDDEN, batch=1),
        # LM head of a batch of sequences
        dict(name="lmhead_b32", kind="lmhead", layout="tiled", vocab=V, cols=HIDDEN, batch=32),
        # a whole decode-step tail for a few sequences, logits kept
        dict(name="step_b8", kind="step", vocab=V, cols=HIDDEN, batch=8, k=64),
        # LM head + sample of a batch, nothing but the tokens and survivors wanted
        dict(name="fused_b32_nologits", kind="fused", vocab=V, cols=HIDDEN, batch=32, k=64,
             logits=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["topk", "topk", "wide", "full", "full", "lmhead", "lmhead", "fused", "step"])
    vocab = V if rng.random() < 0.3 else _log_int(rng, 8000, V)
    if kind in ("topk", "wide", "full"):
        dtype = rng.choice(["f32", "bf16"])
        c = dict(kind=kind, call=rng.choice(["sync", "async"]), dtype=dtype,
                 dist=rng.choice(["peaky", "peaky", "flat"]), vocab=vocab)
        if kind == "topk":
            c.update(batch=_log_int(rng, 1, 96), k=rng.choice([0, 1, 40, 64, 200, 1000]))
        elif kind == "wide":
            c.update(batch=_log_int(rng, 1, 8), k=_log_int(rng, 1100, min(vocab // 2, 20000)))
        else:
            c.update(batch=_log_int(rng, 1, 128 if dtype == "bf16" else 64),
                     probs=rng.random() < 0.25)
        return c
    cols = HIDDEN if rng.random() < 0.4 else 32 * _log_int(rng, 16, 128)
    most = max(1, min(64, V * HIDDEN * 32 // (vocab * cols)))
    batch = _log_int(rng, 1, most)
    if kind == "lmhead":
        return dict(kind=kind, layout=rng.choice(["tiled", "tiled", "rows"]), vocab=vocab,
                    cols=cols, batch=min(batch, 32) if cols > HIDDEN else batch)
    if kind == "step":
        return dict(kind=kind, vocab=vocab, cols=cols, batch=batch, k=rng.choice([1, 64, 200]))
    return dict(kind=kind, vocab=vocab, cols=cols, batch=batch, k=rng.choice([1, 64, 200]),
                logits=rng.random() < 0.5)


# --------------------------------------------------------------- inputs


def _stride(case):
    """Logits per row: the vocabulary, padded to whole 16-byte vectors."""
    return (case["vocab"] + 7) // 8 * 8


def _gen(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _logits(case, seed):
    """peaky: N(0, 3^2) with 16 candidates raised by 6..12 in each row, as a
    trained model's logits look; flat: N(0, 0.5^2)."""
    g = _gen(seed)
    B, n = case["batch"], case["vocab"]
    x = torch.zeros(B, _stride(case), device=DEVICE)
    x[:, :n] = torch.randn(B, n, generator=g, device=DEVICE) * (3.0 if case["dist"] == "peaky" else 0.5)
    if case["dist"] == "peaky":
        at = torch.randint(0, n, (B, 16), generator=g, device=DEVICE)
        up = 6.0 + 6.0 * torch.rand(B, 16, generator=g, device=DEVICE)
        x.scatter_(1, at, x.gather(1, at) + up)
    return x if case["dtype"] == "f32" else x.to(torch.bfloat16)


def _settings(case, seed):
    """(temperature, top_k, top_p, u) of every row."""
    r = np.random.RandomState(seed % (1 << 31))
    B = case["batch"]
    u = r.randint(0, 1 << 32, B, dtype=np.uint64) / 4294967296.0
    if case["kind"] == "full":
        return np.full(B, 1.0, "f4"), np.zeros(B, "i4"), np.full(B, 0.99, "f4"), u
    if case["k"] == 0:
        return ((0.3 + 1.2 * r.rand(B)).astype("f4"), r.choice([1, 20, 64, 256], B).astype("i4"),
                r.choice([0.8, 0.9, 0.95, 1.0], B).astype("f4"), u)
    return np.full(B, 0.7, "f4"), np.full(B, case["k"], "i4"), np.full(B, 0.95, "f4"), u


def _weights(case, seed):
    """Q4_0 rows: 18-byte blocks, fp16 scale in 0.001..0.02, 16 nibble bytes."""
    g = _gen(seed + 7)
    n = case["vocab"] * (case["cols"] // 32)
    w = torch.empty(n, 18, dtype=torch.uint8, device=DEVICE)
    w[:, 2:] = torch.randint(0, 256, (n, 16), generator=g, device=DEVICE, dtype=torch.uint8)
    s = (0.001 + 0.019 * torch.rand(n, 1, generator=g, device=DEVICE)).to(torch.float16)
    w[:, :2] = s.view(torch.uint8)
    return w


def _hidden(case, seed):
    return torch.randn(case["batch"], case["cols"], generator=_gen(seed + 8), device=DEVICE)


def _tokens(case, seed):
    return torch.randint(0, case["vocab"], (case["batch"],), generator=_gen(seed + 9),
                         device=DEVICE, dtype=torch.int32)


def _embed_scale(case):
    return float(np.float32(np.sqrt(np.float32(case["cols"]))))


def _params(settings):
    return [native.TSamplingParams.make(t, k, p) for t, k, p in zip(*settings[:3])]


def _outputs(case, capacity):
    """The optional device outputs, and the tensors behind them."""
    B = case["batch"]
    i32 = dict(dtype=torch.int32, device=DEVICE)
    o = dict(count=torch.zeros(B, **i32), argmax=torch.zeros(B, **i32),
             lsum=torch.zeros(B, device=DEVICE))
    if capacity:
        o["probs"] = torch.zeros(B, capacity, device=DEVICE)
        if case["kind"] != "full":
            o["indices"] = torch.zeros(B, capacity, **i32)
    at = {k: t.data_ptr() for k, t in o.items()}
    return o, native.Outputs(at["count"], at.get("indices"), at.get("probs"), capacity,
                             at["argmax"], at["lsum"], None)


def prepare(case, seed):
    st = dict(case=case)
    B = case["batch"]
    st["sampler"] = native.Sampler(case["vocab"], max_batch=B, softcap=CAP)
    if case["kind"] in ("topk", "wide", "full"):
        sets = _settings(case, seed)
        st["logits"] = _logits(case, seed)
        st["params"], st["u"] = _params(sets), sets[3]
        if case["call"] == "async":
            rec = np.zeros(B, dtype=[("t", "f4"), ("k", "i4"), ("p", "f4"), ("r", "f4")])
            rec["t"], rec["k"], rec["p"], rec["r"] = sets[0], sets[1], sets[2], 1.0
            st["d_params"] = torch.from_numpy(rec.view(np.uint8).copy()).to(DEVICE)
            st["d_u"] = torch.from_numpy(sets[3]).to(DEVICE)
            st["d_ids"] = torch.zeros(B, dtype=torch.int32, device=DEVICE)
            kmax = int(sets[1].max())
            st["k_bound"] = 0 if case["kind"] == "full" else kmax
            cap = kmax if case["kind"] != "full" else case["vocab"] if case["probs"] else 0
            st["out"], st["struct"] = _outputs(case, cap)
        return st
    w = _weights(case, seed)
    if case["kind"] == "lmhead" and case["layout"] == "rows":
        st["weights"] = w
    else:
        n = native.q4_0_device_bytes(case["vocab"], case["cols"], native.Q4_LAYOUT_TILED64)
        st["weights"] = torch.empty(n, dtype=torch.uint8, device=DEVICE)
        native.q4_0_repack(w.data_ptr(), case["vocab"], case["cols"], st["weights"].data_ptr())
    st["stride"] = _stride(case)
    if case["kind"] == "step":
        st["table"], st["tokens"] = w, _tokens(case, seed)
        st["hidden"] = torch.empty(B, case["cols"], device=DEVICE)
    else:
        st["hidden"] = _hidden(case, seed)
    if case["kind"] != "fused" or case["logits"]:
        st["logits"] = torch.zeros(B, st["stride"], device=DEVICE)
    if case["kind"] != "lmhead":
        sets = _settings(case, seed)
        st["params"], st["u"] = _params(sets), sets[3]
        st["out"], st["struct"] = _outputs(case, case["k"])
    return st


def run(st):
    case, s = st["case"], st["sampler"]
    B, kind = case["batch"], case["kind"]
    if kind in ("topk", "wide", "full"):
        dtype = native.DTYPE_F32 if case["dtype"] == "f32" else native.DTYPE_BF16
        if case["call"] == "sync":
            return s.sample(st["logits"].data_ptr(), B, st["params"], st["u"], dtype=dtype,
                            row_stride=_stride(case))[1]
        s.sample_async(st["logits"].data_ptr(), B, st["d_params"].data_ptr(), st["d_u"].data_ptr(),
                       st["k_bound"], kind == "full", st["d_ids"].data_ptr(), dtype=dtype,
                       row_stride=_stride(case), outputs=st["struct"])
        return dict(st["out"], ids=st["d_ids"])
    hidden = st["hidden"].data_ptr()
    logits = st["logits"].data_ptr() if "logits" in st else None
    weights = st["weights"].data_ptr()
    if kind == "lmhead":
        f = s.lmhead_q4_0_tiled if case["layout"] == "tiled" else s.lmhead_q4_0
        f(weights, case["vocab"], case["cols"], hidden, B, logits, st["stride"])
        return st["logits"]
    if kind == "step":
        s.embed_q4_0(st["table"].data_ptr(), case["vocab"], case["cols"], st["tokens"].data_ptr(),
                     B, _embed_scale(case), hidden)
    ids = s.lmhead_sample_q4_0(weights, case["cols"], hidden, B, logits, st["params"], st["u"],
                               logits_stride=st["stride"], outputs=st["struct"])[1]
    r = dict(st["out"], ids=ids)
    if kind == "step":
        r["hidden"] = st["hidden"]
    if logits is not None:
        r["logits"] = st["logits"]
    return r


def work(case):
    B, n = case["batch"], case["vocab"]
    if case["kind"] in ("topk", "wide", "full"):
        each = 4 if case["dtype"] == "f32" else 2
        out = 4 * n if case.get("probs") else 0 if case["kind"] == "full" else 8 * (case["k"] or 64)
        return {"bytes": B * (n * each + out + 40), "flops": 0}
    cols = case["cols"]
    size = n * (cols // 32) * 18 + 4 * B * cols
    if case["kind"] == "step":
        size += B * (cols // 32) * 18 + 4 * B * cols
    if case["kind"] != "fused" or case["logits"]:
        size += 4 * B * n
    return {"bytes": size, "flops": 2 * B * n * cols}


def tolerance(case):
    # ids, survivors, probabilities, sums and logits are the reference's bits
    return "exact"


# ------------------------------------------------------------- 64 bits


def _rows64(w, cols, lo, hi):
    """Dequantised rows lo..hi of Q4_0 blocks, in 64 bits."""
    nblk = cols // 32
    b = w[lo * nblk:hi * nblk]
    sc = b[:, :2].contiguous().view(torch.float16).double()
    q = torch.stack((b[:, 2:] & 15, b[:, 2:] >> 4), dim=2).reshape(-1, 32).double() - 8.0
    return (q * sc).reshape(hi - lo, cols)


def _softmax64(case, x, settings):
    """(e, sum) of every row's softcapped, tempered logits."""
    t = torch.from_numpy(settings[0].astype("f8")).to(x.device).unsqueeze(1)
    y = CAP * torch.tanh(x / CAP) / t
    e = torch.exp(y - y.max(dim=1, keepdim=True).values)
    return e, e.sum(dim=1)


def _survivors64(case, x, settings):
    """probs [batch, capacity] of the TopK largest, in index order, and sums."""
    k = settings[1]
    probs = torch.zeros(x.shape[0], int(k.max()), dtype=torch.float64, device=x.device)
    sums = torch.zeros(x.shape[0], dtype=torch.float64, device=x.device)
    for r in range(x.shape[0]):
        at = torch.topk(x[r], int(k[r])).indices.sort().values
        e, s = _softmax64(case, x[r:r + 1, at].double(), [settings[0][r:r + 1]])
        probs[r, :len(at)] = e[0] / s
        sums[r] = s[0]
    return probs, sums


def exact(case, seed):
    kind = case["kind"]
    if kind in ("topk", "wide", "full"):
        if case["call"] == "sync":
            return None  # ids alone
        x = _logits(case, seed)[:, :case["vocab"]]
        sets = _settings(case, seed)
        if kind == "full":
            sums, probs = [], []
            for r in range(case["batch"]):
                e, s = _softmax64(case, x[r:r + 1].double(), [sets[0][r:r + 1]])
                sums.append(s)
                if case["probs"]:
                    probs.append(e / s)
            r = dict(count=None, argmax=None, ids=None, lsum=torch.cat(sums))
            if case["probs"]:
                r["probs"] = torch.cat(probs)
            return r
        probs, sums = _survivors64(case, x, sets)
        # which of several equal bf16 logits survive is the reference's heap order
        return dict(count=None, indices=None, argmax=None, ids=None, lsum=sums,
                    probs=probs if case["dtype"] == "f32" else None)
    w = _weights(case, seed)
    cols, n = case["cols"], case["vocab"]
    hidden = None
    if kind == "step":
        t = _tokens(case, seed).long()
        hidden = torch.cat([_rows64(w, cols, int(i), int(i) + 1) for i in t]) * _embed_scale(case)
        h = hidden.float().double()
    else:
        h = _hidden(case, seed).double()
    logits = torch.zeros(case["batch"], _stride(case), dtype=torch.float64, device=DEVICE)
    for lo in range(0, n, 16384):
        hi = min(n, lo + 16384)
        logits[:, lo:hi] = h @ _rows64(w, cols, lo, hi).T
    if kind == "lmhead":
        return logits
    sums = _survivors64(case, logits[:, :n], _settings(case, seed))[1]
    r = dict(count=None, indices=None, probs=None, argmax=None, ids=None, lsum=sums)
    if kind == "step":
        r["hidden"] = hidden
    if kind == "step" or case["logits"]:
        r["logits"] = logits
    return r

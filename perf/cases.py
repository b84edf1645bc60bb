"""The work this framework does for its users, as measurable passes: the mixers of the decoders it
serves, at the sizes of served steps, in the order of calls that the model classes make.

Kinds of case (``kind``):

  window   attention of a layer-list model over paged keys and values: norms, rotation and page
           append of a projected row, then attention.  ``form`` "softcap": rows convolved over time,
           softcapped softmax (Minerax); "sigmoid": projection bias, sliding window with kept first
           tokens, sigmoid weights (Nutitar).
  latent   attention whose pages hold one latent with a rotated key part for all heads: queries
           carried into the latent space, norm and append, attention with a softmax sink.  ``window``
           0 with an output gate per head (Nutitar), or a sliding window (Minerax).
  delta    the channel-wise gated delta rule behind activated convolutions (Bilolix, Minerax).
  gla      gated linear attention (Bilolix).
  wkv      token shift and wkv recurrence (Numalorn).
  llama    qkv projection with rotary append, then paged GQA attention (Llama-3, Mixtral).

``seqs`` lists the scheduled sequences of the step as "rows@context": rows of this step after
``context`` cached tokens.  One row per sequence is a decode step (the decode section of the engine's
step); otherwise the sequences are prompts or prompt chunks (its prefill section).  Heads, widths,
prompt and context lengths are those of the benchmark (``bench.py`` and ``--arch-compare``): models of
the 1b, 8b and 70b class, prompts of up to 2,048 tokens, up to 64 sequences decoding from some hundred
to two thousand tokens.
"""
from __future__ import annotations

import math

import torch

from replisense_rfq_amd import ops

DEV = "cuda"
BS = 32                     # tokens per page
EPS = 1e-5
UNIT_EPS = 1e-6             # unit vectors of the delta rule
RANK = 64                   # inner width of the low-rank decay and gate projections
TAPS = 4
CAP = 30.0                  # softcap of the scores
WINDOW, KEEP = 1024, 64
ROT = 64                    # rotated entries per head
ROT_BASE = 5e5
R_LAT = 512                 # latent width; its rotated key part is ROT wide
DIM = 128                   # head width of the attention layers
RDIM, VDIM = 64, 128        # state of a delta-rule / gla head
WDIM = 64                   # state of a wkv head: WDIM x WDIM
# (hidden, query heads, key/value heads) of the 1b, 8b and 70b class
CLASSES = ((2048, 16, 4), (4096, 32, 8), (8192, 64, 8))


# ----------------------------------------------------------------------------- cases
def _case(kind, seqs, d=4096, H=32, G=8, dtype="bfloat16", name=None, **more):
    c = {"kind": kind, "seqs": seqs, "d": d, "H": H, "G": G, "dtype": dtype, **more}
    if name is not None:
        c["name"] = name
    return c


def _ragged(n, lo, hi):
    """n contexts spread over lo .. hi, in no order: sequences of a running batch."""
    return [lo + (i * 7919 + 13) % (hi - lo + 1) for i in range(n)]


def listed():
    decode = ",".join(f"1@{c}" for c in _ragged(64, 300, 900))
    return [
        # one idle request decoding: the latency path's smallest call
        _case("window", "1@611", form="softcap", name="window_decode_one"),
        # a running batch of 64 documents, some hundred tokens into each
        _case("window", decode, form="softcap", name="window_decode_64"),
        # an admitted prompt of the full chunk and a short one beside it
        _case("window", "2048@0,600@0", form="softcap", name="window_prefill"),
        # prompts of odd lengths, one of them the second chunk of a long prompt; window, sigmoid
        _case("window", "1031@0,77@0,345@1701,1@0,613@0", form="sigmoid", name="window_prefill_ragged"),
        _case("latent", decode, window=0, name="latent_decode_64"),
        # the largest: four full prompts in one step
        _case("latent", "2048@0,2048@0,2048@0,2048@0", window=0, name="latent_prefill"),
        _case("delta", "2048@0,2048@0", H=32, G=32, name="delta_prefill"),
        _case("delta", decode, H=32, G=32, name="delta_decode_64"),
        # odd lengths and a continued prompt, a model served in full precision
        _case("gla", "1031@0,77@0,345@1701,1@0,613@0", H=32, G=32, dtype="float32", name="gla_prefill_ragged"),
        _case("wkv", "2048@0,2048@0", H=64, G=64, name="wkv_prefill"),
        # the headline model: a batch of short prompts (RFQ documents behind a cached prefix)
        _case("llama", "230@416,187@416,512@416,333@416,96@416,401@416,268@416,740@416", name="llama_prefill"),
        _case("llama", decode, name="llama_decode_64"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A step of any kind, class, number and length of sequences; ends where the listed ones end."""
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(("window", "latent", "delta", "gla", "wkv", "llama"))
        d, H, G = rng.choice(CLASSES)
        if rng.random() < 0.5:                       # decode
            n = _log_int(rng, 1, 64)
            top = _log_int(rng, 64, 2000)
            seqs = [(1, rng.randint(max(1, top // 3), top)) for _ in range(n)]
        else:                                        # prompts and prompt chunks
            n = _log_int(rng, 1, 8)
            seqs = [(_log_int(rng, 1, 2048), rng.choice((0, 0, 0, rng.randint(1, 2000)))) for _ in range(n)]
            if all(q == 1 for q, _ in seqs) or sum(q for q, _ in seqs) > 8192:
                continue
        c = _case(kind, ",".join(f"{q}@{p}" for q, p in seqs), d, H, G)
        if kind == "window":
            c["form"] = rng.choice(("softcap", "sigmoid"))
        elif kind == "latent":
            c["window"] = rng.choice((0, WINDOW))
        elif kind in ("delta", "gla"):
            c["H"] = c["G"] = d // 128
            c["dtype"] = rng.choice(("bfloat16", "bfloat16", "float32"))
        elif kind == "wkv":
            c["H"] = c["G"] = d // 64
            c["dtype"] = rng.choice(("bfloat16", "bfloat16", "float32"))
        # the longest run bounds a recurrence's time, the total everything else
        if kind in ("delta", "gla", "wkv") and sum(q for q, _ in seqs) > 4096:
            continue
        if _cost(c) <= most:
            return c


def _seqs(case):
    return [tuple(int(x) for x in s.split("@")) for s in case["seqs"].split(",")]


def _decode(case):
    return all(q == 1 for q, _ in _seqs(case)) and any(p > 0 for _, p in _seqs(case))


def _bytes_of(case):
    return 2 if case["dtype"] == "bfloat16" else 4


def _pairs(seqs, window=0, keep=0):
    """(query, key) pairs that are visible, and keys that some query sees."""
    pairs = seen = 0
    for q, p in seqs:
        for i in range(p, p + q):
            pairs += i + 1 if window == 0 else min(i + 1, window + min(keep, max(0, i + 1 - window)))
        seen += p + q if window == 0 else min(p + q, window + q - 1 + keep)
    return pairs, seen


def work(case):
    """Each input read once, each output written once; the products of the mixer."""
    seqs, kind, es = _seqs(case), case["kind"], _bytes_of(case)
    T, n = sum(q for q, _ in seqs), len(seqs)
    H, G, d = case["H"], case["G"], case["d"]
    live = sum(1 for _, p in seqs if p > 0)
    if kind == "window":
        N = (H + 2 * G) * DIM
        soft = case["form"] == "softcap"
        pairs, seen = _pairs(seqs) if soft else _pairs(seqs, WINDOW, KEEP)
        old = max(0, seen - T)
        nbytes = es * (T * N + old * 2 * G * DIM + T * 2 * G * DIM + T * H * DIM)
        nbytes += (n + live) * (TAPS - 1) * N * 4 if soft else 0
        return {"bytes": nbytes, "flops": 4.0 * DIM * H * pairs}
    if kind == "latent":
        E = R_LAT + ROT
        pairs, seen = _pairs(seqs, case["window"])
        N = H * (DIM + ROT) + E
        nbytes = es * (T * N + max(0, seen - T) * E + T * E + H * DIM * R_LAT + T * H * R_LAT)
        return {"bytes": nbytes, "flops": 2.0 * (E + R_LAT) * H * pairs + 2.0 * T * H * DIM * R_LAT}
    if kind in ("delta", "gla"):
        state = (n + live) * H * RDIM * VDIM * 4
        C = 2 * G * RDIM + H * VDIM
        inner = RANK * H * (RDIM + (VDIM if kind == "delta" else 0))
        row = C + RANK + H * VDIM + (RANK + H if kind == "delta" else H * VDIM)
        nbytes = es * (T * row + inner) + state + ((n + live) * (TAPS - 1) * C * 4 if kind == "delta" else 0)
        return {"bytes": nbytes, "flops": (10.0 if kind == "delta" else 6.0) * T * H * RDIM * VDIM + 2.0 * T * inner}
    if kind == "wkv":
        state = (n + live) * (H * WDIM * WDIM + d) * 4
        return {"bytes": T * d * 4 + es * T * d * 5 + es * T * H * WDIM * 6 + state, "flops": 6.0 * T * H * WDIM * WDIM}
    pairs, seen = _pairs(seqs)
    N = (H + 2 * G) * DIM
    nbytes = 2 * (T * d + N * d + max(0, seen - T) * 2 * G * DIM + T * 2 * G * DIM + T * H * DIM)
    return {"bytes": nbytes, "flops": 4.0 * DIM * H * pairs + 2.0 * T * N * d}


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 8e12, w["flops"] / 2.5e15)


def tolerance(case):
    """About four times the error against 64 bits: bf16 outputs 1.6e-3 .. 2.3e-3 (their own rounding; 3e-3
    behind the latent queries, which enter the products as bf16), fp32 models 6e-7 .. 1.1e-6."""
    if case["dtype"] == "float32":
        return {"rel": 5e-6}
    return {"rel": 1.2e-2 if case["kind"] == "latent" else 8e-3}


# ----------------------------------------------------------------------------- inputs
def _i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def __call__(self, *shape, mult=1.0, add=0.0, dtype=torch.float32):
        return (torch.randn(shape, generator=self.g, device=DEV) * mult + add).to(dtype)


def _rows(seqs):
    """Per-row arrays of the recurrent states (sequence i owns slot i) and the runs' first rows."""
    rs, rb, rf, pos, runs = [], [], [], [], []
    for i, (q, p) in enumerate(seqs):
        runs.append(len(rs))
        rs += [2 * i + i % 2] * q
        rb += range(q)
        rf += range(q - 1, -1, -1)
        pos += range(p, p + q)
    return {"row_state": _i32(rs), "row_back": _i32(rb), "row_fwd": _i32(rf), "pos": _i32(pos), "runs": _i32(runs)}


def _pages(seqs, seed):
    """Page tables over a pool in no order, the rows' slots and the work lists of the step."""
    need = [(q + p + BS - 1) // BS for q, p in seqs]
    total = sum(need) + 1
    perm = torch.randperm(total - 1, generator=torch.Generator().manual_seed(seed)).tolist()
    maxb, at, tables, slots, starts, t = max(need), 0, [], [], [], 0
    for (q, p), nb in zip(seqs, need):
        pages = perm[at:at + nb]
        tables.append(pages + [total - 1] * (maxb - nb))
        slots += [pages[i // BS] * BS + i % BS for i in range(p, p + q)]
        starts.append(t)
        t += q
        at += nb
    return {"blocks": total, "tables": _i32(tables), "slots": _i32(slots), "q_start": _i32(starts),
            "q_len": _i32([q for q, _ in seqs]), "kv_len": _i32([q + p for q, p in seqs]),
            "pos": _i32([i for q, p in seqs for i in range(p, p + q)])}


def _work_items(seqs, qblk):
    w = [(s, b) for s, (q, _) in enumerate(seqs) for b in range((q + qblk - 1) // qblk)]
    return _i32([x[0] for x in w]), _i32([x[1] for x in w])


def _inv_freq(n, base):
    return (base ** (-torch.arange(0, n, 2, dtype=torch.float64) / n)).float().to(DEV)


def prepare(case, seed):
    seqs, kind = _seqs(case), case["kind"]
    dt = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32
    rnd = _Rand(seed)
    H, G, d = case["H"], case["G"], case["d"]
    T, n = sum(q for q, _ in seqs), len(seqs)
    s = {"case": case, "dt": dt, "T": T, "decode": _decode(case), "seqs": seqs}
    if kind in ("window", "latent", "llama"):
        s["m"] = m = _pages(seqs, seed)
        nb = m["blocks"]
    if kind in ("window", "delta", "gla", "wkv"):
        s["rows"] = _rows(seqs)
    if kind == "window":
        N = (H + 2 * G) * DIM
        soft = case["form"] == "softcap"
        # in a softcapped layer the projected row also holds the delta rule's columns
        s["proj"] = rnd(T, N + (2 * H * RDIM + H * VDIM if soft else 0), mult=2.0 if soft else 0.7, dtype=dt)
        s["bias"] = None if soft else rnd(N, mult=0.3)
        s["qn"], s["kn"] = rnd(H * DIM, mult=0.2, add=1.0), rnd(G * DIM, mult=0.2, add=1.0)
        s["inv"], s["mult"] = _inv_freq(ROT, ROT_BASE), 1.0
        s["kc"] = rnd(nb, G, BS, DIM, dtype=dt)
        s["vc"] = rnd(nb, G, BS, DIM, dtype=dt)
        s["conv_w"] = rnd(TAPS, N, mult=0.5) if soft else None
        s["conv_state"] = rnd(2 * n, TAPS - 1, N, mult=2.0) if soft else None
        s["head_bias"] = None if soft else rnd(H, add=-3.0)
        s["work"] = _work_items(seqs, ops.KEEP_QBLK)
    elif kind == "latent":
        E = R_LAT + ROT
        gated = case["window"] == 0
        s["proj"] = rnd(T, H * (DIM + ROT) + E + (H if gated else H * DIM), dtype=dt)
        s["uk"] = rnd(H, DIM, R_LAT, mult=2.0 * R_LAT ** -0.5, dtype=dt)
        s["dkv_norm"], s["sink"] = rnd(R_LAT, mult=0.1, add=1.0), rnd(H)
        s["inv"], s["mult"] = _inv_freq(ROT, ROT_BASE), 0.1 * math.log(4.0) + 1.0
        s["pool"] = rnd(nb, 1, BS, E, dtype=dt)
        s["work"] = _work_items(seqs, ops.KEEP_QBLK)
    elif kind in ("delta", "gla"):
        C = 2 * G * RDIM + H * VDIM
        delta = kind == "delta"
        extra = {"x": C, "a1": RANK, **({"g1": RANK, "b": H} if delta else {"g": H * VDIM})}
        s["proj"], at = rnd(T, sum(extra.values()), mult=2.0 if delta else 1.0, dtype=dt), 0
        for key, w in extra.items():
            s[key] = s["proj"][:, at:at + w]
            at += w
        s["a2"] = rnd(H * RDIM, RANK, mult=RANK ** -0.5, dtype=dt)
        s["norm"] = rnd(VDIM, mult=0.1, add=1.0)
        s["S"] = rnd(2 * n, H, RDIM, VDIM, mult=0.3)
        if delta:
            s["conv_w"], s["conv_state"] = rnd(C, TAPS, mult=0.5), rnd(2 * n, TAPS - 1, C, mult=2.0)
            s["rate"], s["zbias"] = torch.exp(rnd(H, mult=0.5, add=-1.0)), rnd(H * RDIM, add=-1.0)
            s["g2"] = rnd(H * VDIM, RANK, mult=RANK ** -0.5, dtype=dt)
        else:
            s["rate"], s["zbias"] = torch.full((H,), 1.0 / 16.0, device=DEV), rnd(H * RDIM, add=2.0)
    elif kind == "wkv":
        HN = H * WDIM
        s["x"], s["mu"] = rnd(T, d), rnd(5, d, mult=0.25, add=0.5)
        s["prev"], s["S"] = rnd(2 * n, d), rnd(2 * n, H, WDIM, WDIM, mult=0.3)
        s["rkvg"] = rnd(4, T, HN, dtype=dt)
        s["zw"] = rnd(T, HN, mult=0.5, dtype=dt)
        s["w0"], s["u"] = rnd(HN, add=-2.0), rnd(H, WDIM, mult=0.5)
        s["norm"] = rnd(HN, mult=0.1, add=1.0)
    else:
        N = (H + 2 * G) * DIM
        s["x"], s["w"] = rnd(T, d, dtype=dt), rnd(N, d, mult=d ** -0.5, dtype=dt)
        s["kc"], s["vc"] = rnd(nb, G, BS, DIM, dtype=dt), rnd(nb, G, BS, DIM, dtype=dt)
        ang = torch.arange(4096, dtype=torch.float64)[:, None] * ROT_BASE ** (-torch.arange(0, DIM, 2, dtype=torch.float64) / DIM)
        s["cos_sin"] = torch.cat([ang.cos(), ang.sin()], -1).float().to(DEV)
        if s["decode"]:
            # the engine's split rule: enough (sequence, key/value head, split) work for the chip
            splits = 1
            while n * G * splits < 1024 and splits < 16:
                splits *= 2
            s["splits"] = max(1, min(splits, (max(p for _, p in seqs) + 1 + 255) // 256))
            s["tickets"] = torch.zeros(4096 * G, dtype=torch.int32, device=DEV) if H // G <= 4 else None
            s["work"] = _i32(range(n)), _i32([0] * n)
        else:
            s["work"] = _work_items(seqs, ops.prefill_qblk(H, G))
    return s


# ----------------------------------------------------------------------------- one pass
def _keep(s, q, kc, vc, vdim, bias, gate, out, scale, **more):
    m = s["m"]
    short = ops.TALK_DECODE_MAX_ROWS if s["decode"] else 0
    ops.attn_keep_window(q, kc, vc, vdim, m["tables"], m["q_start"], m["q_len"], m["kv_len"], *s["work"],
                         bias, gate, out, scale, short_rows=short, **more)


def _window(s):
    c, m, r = s["case"], s["m"], s["rows"]
    H, G, T = c["H"], c["G"], s["T"]
    q = torch.empty((T, H, DIM), dtype=torch.float32, device=DEV)
    out = torch.empty((T, H * DIM), dtype=s["dt"], device=DEV)
    soft = c["form"] == "softcap"
    conv = (s["conv_w"], s["conv_state"], r["row_state"], r["row_back"], r["row_fwd"]) if soft else None
    ops.qk_norm_rotary_append(s["proj"], s["bias"], s["qn"], s["kn"], True, DIM, EPS, m["pos"], s["inv"], s["mult"],
                              0, 0, m["slots"], s["kc"], s["vc"], H, G, DIM, DIM, DIM, 0, q, conv=conv)
    if soft:
        _keep(s, q, s["kc"], s["vc"], DIM, None, None, out, DIM ** -0.5, softcap=CAP, out_mult=0.6)
        return {"out": out, "k": s["kc"], "v": s["vc"], "conv": s["conv_state"]}
    _keep(s, q, s["kc"], s["vc"], DIM, s["head_bias"], None, out, DIM ** -0.5, window=WINDOW, keep_first=KEEP,
          sigmoid=True)
    return {"out": out, "k": s["kc"], "v": s["vc"]}


def _latent(s):
    c, m = s["case"], s["m"]
    H, T, E = c["H"], s["T"], R_LAT + ROT
    nq, gated = H * (DIM + ROT), c["window"] == 0
    q = torch.empty((T, H, E), dtype=torch.float32, device=DEV)
    qn = s["proj"][:, :nq].unflatten(1, (H, DIM + ROT))[:, :, :DIM].transpose(0, 1)
    ops.bmm_f32(qn, s["uk"], out=q[:, :, :R_LAT].transpose(0, 1))
    ops.qk_norm_rotary_append(s["proj"], None, None, s["dkv_norm"], False, R_LAT, EPS, m["pos"], s["inv"], s["mult"],
                              DIM, R_LAT, m["slots"], s["pool"], None, H, 1, DIM + ROT, E, 0, 2, q[:, :, R_LAT:],
                              neighbours=not gated)
    out = torch.empty((T, H * R_LAT), dtype=s["dt"], device=DEV)
    gate = s["proj"][:, nq + E:] if gated else None
    _keep(s, q, s["pool"], s["pool"], R_LAT, s["sink"], gate, out, (DIM + ROT) ** -0.5, window=c["window"])
    return {"out": out, "pool": s["pool"]}


def _recurrence(s):
    c, r = s["case"], s["rows"]
    H, G, T, delta = c["H"], c["G"], s["T"], c["kind"] == "delta"
    rows = (r["row_state"], r["row_back"], r["row_fwd"], r["pos"])
    nk = G * RDIM
    x = s["x"]
    if delta:
        x = torch.empty((T, x.shape[1]), dtype=torch.float32, device=DEV)
        ops.conv_act_heads(s["x"], s["conv_w"], s["conv_state"], *rows, 2 * G, RDIM, UNIT_EPS, x)
    z = ops.matmul_nt(s["a1"], s["a2"], out_dtype=torch.float32)
    gate = ops.matmul_nt(s["g1"], s["g2"]) if delta else s["g"]
    out = torch.empty((T, H * VDIM), dtype=s["dt"], device=DEV)
    ops.gated_linear_recurrence(
        x[:, :nk].unflatten(1, (G, RDIM)), x[:, nk:2 * nk].unflatten(1, (G, RDIM)),
        x[:, 2 * nk:].unflatten(1, (H, VDIM)), z, s["rate"], s["zbias"], 1.0 if delta else -1.0,
        s["b"] if delta else None, gate, delta, s["norm"], EPS, RDIM ** -0.5, s["S"], *rows, out, r["runs"])
    return {"out": out, "S": s["S"], **({"conv": s["conv_state"]} if delta else {})}


def _wkv(s):
    c, r = s["case"], s["rows"]
    T, HN = s["T"], c["H"] * WDIM
    rows = (r["row_state"], r["row_back"], r["row_fwd"], r["pos"])
    mixes = ops.token_shift_mix(s["x"], s["mu"], s["prev"], *rows, torch.empty((5, T, c["d"]), dtype=s["dt"], device=DEV))
    a = s["rkvg"]
    out = ops.wkv_recurrence(a[0], a[1], a[2], s["zw"], s["w0"], s["u"], a[3], s["norm"], EPS, s["S"], *rows,
                             torch.empty((T, HN), dtype=s["dt"], device=DEV), r["runs"])
    return {"mixes": mixes, "out": out, "prev": s["prev"], "S": s["S"]}


def _llama(s):
    c, m = s["case"], s["m"]
    H, G, T = c["H"], c["G"], s["T"]
    qkv = ops.qkv_rope(s["x"], s["w"], m["pos"], s["cos_sin"], m["slots"], s["kc"], s["vc"], H, G)
    out = torch.empty((T, H * DIM), dtype=s["dt"], device=DEV)
    meta = (m["tables"], m["q_start"], m["q_len"], m["kv_len"], *s["work"])
    if s["decode"]:
        k, po, pm = s["splits"], out, out
        if k > 1:
            po = torch.empty(T * H * k * DIM, device=DEV)
            pm = torch.empty(T * H * k * 2, device=DEV)
        ops.attn_decode(qkv, s["kc"], s["vc"], *meta, out, po, pm, H, G, DIM ** -0.5, k, 1 if 8 <= H // G <= 16 else 2,
                        s["tickets"])
    else:
        ops.attn_prefill(qkv, s["kc"], s["vc"], *meta, out, H, G, DIM ** -0.5, ops.prefill_qblk(H, G))
    return {"out": out, "k": s["kc"], "v": s["vc"]}


_RUN = {"window": _window, "latent": _latent, "delta": _recurrence, "gla": _recurrence, "wkv": _wkv, "llama": _llama}


def run(state):
    return _RUN[state["case"]["kind"]](state)


# ----------------------------------------------------------------------------- the same in 64 bits
def _stored(x, s):
    """A value that the framework keeps in the model's type between kernels."""
    return x.to(s["dt"]).double()


def _halves(i, n):
    """(row read, row written) of sequence i in a double-buffered state pool of n slots."""
    return (i % 2) * n + i, (1 - i % 2) * n + i


def _each(s):
    t = 0
    for i, (q, p) in enumerate(s["seqs"]):
        yield i, t, q, p
        t += q


def _conv64(s, x, w, pool):
    """Causal convolution of every sequence's rows (w [C, taps]) and the pool with its new halves."""
    out, new, n, K = [], pool.clone(), len(s["seqs"]), TAPS - 1
    for i, t, q, p in _each(s):
        rd, wr = _halves(i, n)
        head = pool[rd].double() if p > 0 else torch.zeros(K, x.shape[1], dtype=torch.float64, device=DEV)
        if 0 < p < K:
            head[:K - p] = 0.0
        full = torch.cat([head, x[t:t + q]])
        out.append(sum(w[:, j].double() * full[j:j + q] for j in range(TAPS)))
        new[wr] = torch.cat([pool[rd].double(), x[t:t + q]])[-K:].float()
    return torch.cat(out), new


def _rotate64(x, pos, inv, mult, off, neighbours):
    n = inv.numel()
    ang = pos.double()[:, None] * inv.double()
    c, s = (torch.cos(ang) * mult)[:, None], (torch.sin(ang) * mult)[:, None]
    a = slice(off, off + 2 * n, 2) if neighbours else slice(off, off + n)
    b = slice(off + 1, off + 2 * n, 2) if neighbours else slice(off + n, off + 2 * n)
    y = x.clone()
    y[..., a], y[..., b] = x[..., a] * c - x[..., b] * s, x[..., b] * c + x[..., a] * s
    return y


def _rms64(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _append64(pool, slots, rows):
    new = pool.clone()
    sl = slots.long()
    new[sl // BS, :, sl % BS] = rows.to(pool.dtype)
    return new


def _attend64(s, q, kc, vc, vdim, scale, window=0, keep=0, cap=0.0, sink=None, sig_bias=None):
    """q [T, H, E]; softmax over the visible keys (cap, sink) or sigmoid weights; [T, H, vdim]."""
    H, G = q.shape[1], kc.shape[1]
    rep = H // G
    out = torch.empty(q.shape[0], H, vdim, dtype=torch.float64, device=DEV)
    for i, t, n, p in _each(s):
        L = p + n
        pages = s["m"]["tables"][i, :(L + BS - 1) // BS].long()
        j, ii = torch.arange(L, device=DEV)[None], torch.arange(p, L, device=DEV)[:, None]
        ok = j <= ii
        if window > 0:
            ok &= (ii - j < window) | (j < keep)
        for g in range(G):
            k = kc[pages, g].reshape(-1, kc.shape[3])[:L].double()
            v = vc[pages, g].reshape(-1, vc.shape[3])[:L, :vdim].double()
            for h in range(g * rep, (g + 1) * rep):
                a = q[t:t + n, h] @ k.t() * scale
                if cap > 0:
                    a = cap * torch.tanh(a / cap)
                if sig_bias is not None:
                    w = torch.sigmoid(a + sig_bias[h].double()) * ok
                else:
                    a = a.masked_fill(~ok, -math.inf)
                    if sink is not None:
                        a = torch.cat([a, sink[h].double().expand(n, 1)], 1)
                    w = torch.softmax(a, -1)[:, :L]
                out[t:t + n, h] = w @ v
    return out


def _window64(s):
    c, m = s["case"], s["m"]
    H, G, T = c["H"], c["G"], s["T"]
    N, nq = (H + 2 * G) * DIM, H * DIM
    soft = c["form"] == "softcap"
    x, res = s["proj"][:, :N].double(), {}
    if soft:
        x, res["conv"] = _conv64(s, x, s["conv_w"].t(), s["conv_state"])
    else:
        x = x + s["bias"].double()
    q = (_rms64(x[:, :nq]) * s["qn"].double()).view(T, H, DIM)
    k = (_rms64(x[:, nq:nq + G * DIM]) * s["kn"].double()).view(T, G, DIM)
    q, k = (_rotate64(y, m["pos"], s["inv"], s["mult"], 0, False) for y in (q, k))
    kc = _append64(s["kc"], m["slots"], k)
    vc = _append64(s["vc"], m["slots"], x[:, nq + G * DIM:].reshape(T, G, DIM))
    if soft:
        o = 0.6 * _attend64(s, q, kc, vc, DIM, DIM ** -0.5, cap=CAP)
    else:
        o = _attend64(s, q, kc, vc, DIM, DIM ** -0.5, WINDOW, KEEP, sig_bias=s["head_bias"])
    return {"out": o.reshape(T, -1), "k": kc, "v": vc, **res}


def _latent64(s):
    c, m = s["case"], s["m"]
    H, T, E = c["H"], s["T"], R_LAT + ROT
    nq, gated = H * (DIM + ROT), c["window"] == 0
    x = s["proj"].double()
    q = x[:, :nq].view(T, H, DIM + ROT)
    lat = torch.stack([q[:, h, :DIM] @ s["uk"][h].double() for h in range(H)], 1)
    rot = _rotate64(q, m["pos"], s["inv"], s["mult"], DIM, not gated)[..., DIM:]
    row = x[:, nq:nq + E].clone()
    row[:, :R_LAT] = _rms64(row[:, :R_LAT]) * s["dkv_norm"].double()
    row = _rotate64(row[:, None], m["pos"], s["inv"], s["mult"], R_LAT, not gated)
    pool = _append64(s["pool"], m["slots"], row)
    o = _attend64(s, torch.cat([lat, rot], -1), pool, pool, R_LAT, (DIM + ROT) ** -0.5, c["window"], sink=s["sink"])
    if gated:
        o = o * torch.sigmoid(x[:, nq + E:])[:, :, None]
    return {"out": o.reshape(T, -1), "pool": pool}


def _scan64(s, pool, step, T, H, vdim):
    """Runs ``step(S, t) -> (S, o)`` over every sequence's tokens."""
    o = torch.empty(T, H, vdim, dtype=torch.float64, device=DEV)
    new, n = pool.clone(), len(s["seqs"])
    for i, t0, q, p in _each(s):
        rd, wr = _halves(i, n)
        S = pool[rd].double() if p > 0 else torch.zeros(pool.shape[1:], dtype=torch.float64, device=DEV)
        for t in range(t0, t0 + q):
            S, o[t] = step(S, t)
        new[wr] = S.float()
    return o, new


def _recurrence64(s):
    c, T = s["case"], s["T"]
    H, G, delta = c["H"], c["G"], c["kind"] == "delta"
    x, res, nk = s["x"].double(), {}, G * RDIM
    if delta:
        y, res["conv"] = _conv64(s, x, s["conv_w"], s["conv_state"])
        x = y * torch.sigmoid(y)
        u = x[:, :2 * nk].view(T, 2 * G, RDIM)
        x = torch.cat([(u / torch.sqrt((u * u).sum(-1, keepdim=True) + UNIT_EPS)).view(T, -1), x[:, 2 * nk:]], 1)
    q, k, v = x[:, :nk].view(T, G, RDIM), x[:, nk:2 * nk].view(T, G, RDIM), x[:, 2 * nk:].view(T, H, VDIM)
    q, k = q.repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1)
    z = s["a1"].double() @ s["a2"].double().t() + s["zbias"].double()
    sp = torch.nn.functional.softplus(z if delta else -z, threshold=1000.0).view(T, H, RDIM)
    a = torch.exp(-s["rate"].double()[:, None] * sp)[..., None]
    b = torch.sigmoid(s["b"].double())[..., None] if delta else None
    kT, qT = k[:, :, :, None], q[:, :, None, :] * RDIM ** -0.5

    def step(S, t):
        S = S * a[t]
        w = v[t]
        if delta:
            w = b[t] * (w - (kT[t].transpose(1, 2) @ S)[:, 0])
        S = S + kT[t] * w[:, None]
        return S, (qT[t] @ S)[:, 0]

    o, S = _scan64(s, s["S"], step, T, H, VDIM)
    g = _stored(s["g1"].double() @ s["g2"].double().t(), s) if delta else s["g"].double()
    act = torch.sigmoid(g) if delta else g * torch.sigmoid(g)
    y = _rms64(o) * s["norm"].double() * act.view(T, H, VDIM)
    return {"out": y.reshape(T, -1), "S": S, **res}


def _wkv64(s):
    c, T, n = s["case"], s["T"], len(s["seqs"])
    H = c["H"]
    x = s["x"].double()
    before, prev = torch.zeros_like(x), s["prev"].clone()
    for i, t, q, p in _each(s):
        rd, wr = _halves(i, n)
        before[t + 1:t + q] = x[t:t + q - 1]
        if p > 0:
            before[t] = s["prev"][rd].double()
        prev[wr] = s["x"][t + q - 1]
    mixes = x[None] + (before - x)[None] * s["mu"].double()[:, None]
    r, k, v, g = (y.double().view(T, H, WDIM) for y in s["rkvg"])
    w = torch.exp(-torch.exp(s["zw"].double() + s["w0"].double())).view(T, H, WDIM)[..., None]
    u = s["u"].double()[..., None]

    def step(S, t):
        kv = k[t][..., None] * v[t][:, None]
        return w[t] * S + kv, (r[t][:, None] @ (S + u * kv))[:, 0]

    o, S = _scan64(s, s["S"], step, T, H, WDIM)
    y = _rms64(o).reshape(T, -1) * s["norm"].double() * (g * torch.sigmoid(g)).reshape(T, -1)
    return {"mixes": mixes, "out": y, "prev": prev, "S": S}


def _llama64(s):
    c, m = s["case"], s["m"]
    H, G, T = c["H"], c["G"], s["T"]
    qkv = _stored(s["x"].double() @ s["w"].double().t(), s).view(T, H + 2 * G, DIM)
    cs = s["cos_sin"][m["pos"].long()].double()[:, None]
    a, b, h = qkv[:, :H + G, :DIM // 2], qkv[:, :H + G, DIM // 2:], DIM // 2
    qk = _stored(torch.cat([a * cs[..., :h] - b * cs[..., h:], b * cs[..., :h] + a * cs[..., h:]], -1), s)
    kc, vc = _append64(s["kc"], m["slots"], qk[:, H:]), _append64(s["vc"], m["slots"], qkv[:, H + G:])
    return {"out": _attend64(s, qk[:, :H], kc, vc, DIM, DIM ** -0.5).reshape(T, -1), "k": kc, "v": vc}


_EXACT = {"window": _window64, "latent": _latent64, "delta": _recurrence64, "gla": _recurrence64, "wkv": _wkv64,
          "llama": _llama64}


def exact(case, seed):
    return _EXACT[case["kind"]](prepare(case, seed))

"""Recurrences in chunks of 16 tokens (csrc/kernels/mix_chunk.hip) against the token-by-token
reference: run lengths around the chunk, head sizes around the tiles, decays from none to total,
non-finite values."""
import pytest
import torch

from replisense_rfq_amd import ops
from replisense_rfq_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"
LENS = [1, 5, 15, 16, 17, 32, 33, 49, 150]       # 318 rows in 9 runs


def _rows(lens, start):
    rs, rb, rf, pos, runs = [], [], [], [], []
    for i, n in enumerate(lens):
        runs.append(len(rs))
        rs += [2 * i + i % 2] * n
        rb += list(range(n))
        rf += list(range(n - 1, -1, -1))
        p = start if i % 3 else 0                # some runs go on from a state, some begin
        pos += list(range(p, p + n))
    t = [torch.tensor(x, dtype=torch.int32) for x in (rs, rb, rf, pos, runs)]
    return t[:4], torch.cat([t[4][:2], torch.tensor([-1], dtype=torch.int32), t[4][2:]])   # -1: padding


def _close(got, want, tol):
    got, want = got.double().cpu(), want.double()
    assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    ok = torch.isfinite(want)
    scale = want[ok].square().mean().sqrt()
    assert float((got[ok] - want[ok]).abs().max()) <= tol * max(1.0, float(scale)) * 8
    assert float((got[ok] - want[ok]).square().mean().sqrt()) <= tol * float(scale)


def _linrec(mode, H, Hq, dim, vdim, dtype, shift, lens=LENS, spoil=None, pad=3, keys=None, spare=0,
            sizes=(1.0, 1.0, 1.0, 1.0)):
    g = torch.Generator().manual_seed(H * 1000 + dim + vdim)
    T = sum(lens)
    wide = torch.randn(T, 2 * Hq * dim + H * vdim + pad, generator=g)              # columns of wider rows
    qk = wide[:, :2 * Hq * dim].unflatten(1, (2 * Hq, dim))
    qk /= qk.square().sum(-1, keepdim=True).sqrt() / (2.0 if mode == "gla" else 1.0)   # unit vectors: delta rule
    if keys is not None:
        keys(qk[:, Hq:], wide[:, 2 * Hq * dim:])
    for part, size in zip((qk[:, :Hq], qk[:, Hq:], wide[:, 2 * Hq * dim:]), sizes):
        part *= size
    if spoil is not None:
        wide[spoil[0], 2 * Hq * dim + spoil[1]] = float(spoil[2])
    wide = wide.to(dtype)
    z = torch.randn(T, H * dim, generator=g) * 2
    rate, zb = torch.rand(H, generator=g) + 0.1, torch.randn(H * dim, generator=g) + shift
    beta = torch.randn(T, H, generator=g).to(dtype) if mode == "delta" else None
    gate = torch.randn(T, H * vdim, generator=g).to(dtype)
    nw = torch.randn(vdim, generator=g)
    st = torch.randn(2 * len(lens), H, dim, vdim, generator=g) * (0.3 * sizes[3])
    rows, runs = _rows(lens, 23)
    runs = torch.cat([runs, torch.full((spare,), -1, dtype=torch.int32)])

    def call(dev, f, w, zz, s, **more):
        out = torch.empty(T, H * vdim, dtype=dtype, device=dev)
        m = lambda x: None if x is None else x.to(dev)  # noqa: E731
        q, k = (w[:, i * Hq * dim:(i + 1) * Hq * dim].unflatten(1, (Hq, dim)) for i in (0, 1))
        v = w[:, 2 * Hq * dim:2 * Hq * dim + H * vdim].unflatten(1, (H, vdim))
        f(q, k, v, zz, m(rate), m(zb), 1.0, m(beta), m(gate), mode == "delta", m(nw), 1e-5, dim ** -0.5, s,
          *(m(r) for r in rows), out, **more)
        return out, s

    want = call("cpu", ref.gated_linear_recurrence, wide, z.clone(), st.clone())
    zd = z.to(DEV)
    assert dim <= ops.CHUNK_DIM
    got = call(DEV, ops.gated_linear_recurrence, wide.to(DEV), zd, st.to(DEV), run_rows=runs.to(DEV))
    assert torch.equal(zd.cpu(), z)              # the chunks read the logits, they do not replace them
    return got, want


# fp32: sums of up to 64 + 16 products and a few hundred decays, each to 2^-24: 1e-5 of the rms is
# ten times what the longest run shows; bf16 outputs are one rounding (2^-9) of the same sums
@pytest.mark.parametrize("shift", [-3.0, 0.0, 60.0])      # decays near one, ordinary, all but zero
@pytest.mark.parametrize("H,Hq,dim,vdim", [(2, 2, 64, 64), (4, 2, 64, 128), (3, 3, 40, 24), (1, 1, 7, 5), (2, 2, 32, 80)])
@pytest.mark.parametrize("mode", ["gla", "delta"])
def test_linear_recurrence_in_chunks(mode, H, Hq, dim, vdim, shift):
    (out, st), (out_w, st_w) = _linrec(mode, H, Hq, dim, vdim, torch.float32, shift)
    _close(out, out_w, 1e-5)
    _close(st, st_w, 1e-5)


@pytest.mark.parametrize("mode", ["gla", "delta"])
def test_linear_recurrence_in_chunks_bf16(mode):
    (out, st), (out_w, st_w) = _linrec(mode, 2, 2, 64, 128, torch.bfloat16, 0.0)
    _close(out, out_w, 2.0 ** -8)
    _close(st, st_w, 1e-5)


@pytest.mark.parametrize("mode", ["gla", "delta"])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_a_non_finite_value_stays_out_of_earlier_tokens(mode, value):
    """Row 9 of the run of 49 (rows 119 ..), in the middle of its first chunk."""
    first = sum(LENS[:7])
    (out, _), (out_w, _) = _linrec(mode, 2, 2, 64, 64, torch.float32, 0.0, spoil=(first + 9, 3, value))
    out, out_w = out.cpu(), out_w
    _close(out[:first + 9], out_w[:first + 9], 1e-5)
    assert not torch.isfinite(out[first + 9, :64]).all()      # the head's norm spreads it over its row
    _close(out[sum(LENS[:8]):], out_w[sum(LENS[:8]):], 1e-5)  # and no other run sees it


def _wkv(dtype, shift, spoil=None, lens=LENS, sizes=(1.0, 1.0, 1.0, 1.0), H=3):
    N = 64
    g = torch.Generator().manual_seed(5)
    T = sum(lens)
    r, k, v, zw, gate = (torch.randn(T, H * N, generator=g) for _ in range(5))
    r, k, v = (x * size for x, size in zip((r, k, v), sizes))
    if spoil is not None:
        v[spoil[0], spoil[1]] = spoil[2]
    r, k, v, zw, gate = (x.to(dtype) for x in (r, k, v, zw, gate))
    w0, u = torch.randn(H * N, generator=g) + shift, torch.randn(H, N, generator=g)
    nw, st = torch.randn(H * N, generator=g), torch.randn(2 * len(lens), H, N, N, generator=g) * (0.3 * sizes[3])
    rows, runs = _rows(lens, 23)

    def call(dev, f, s, **more):
        out = torch.empty(T, H * N, dtype=dtype, device=dev)
        m = [x.to(dev) for x in (r, k, v, zw, w0, u, gate, nw)]
        f(*m, 1e-5, s, *(x.to(dev) for x in rows), out, **more)
        return out, s

    return call(DEV, ops.wkv_recurrence, st.to(DEV), run_rows=runs.to(DEV)), call("cpu", ref.wkv_recurrence, st.clone())


@pytest.mark.parametrize("shift", [-6.0, -2.0, 5.0])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_wkv_in_chunks(dtype, shift):
    (out, st), (out_w, st_w) = _wkv(dtype, shift)
    _close(out, out_w, 1e-5 if dtype == torch.float32 else 2.0 ** -8)
    _close(st, st_w, 1e-5)


def test_wkv_non_finite_value_stays_out_of_earlier_tokens():
    first = sum(LENS[:7])
    (out, _), (out_w, _) = _wkv(torch.float32, -2.0, (first + 9, 3, float("inf")))
    _close(out[:first + 9], out_w[:first + 9], 1e-5)
    _close(out[sum(LENS[:8]):], out_w[sum(LENS[:8]):], 1e-5)


def _cut(mode, H, vdim, lens, waves=8):
    """The host lets the step's runs be cut (the list of runs has an entry of -1 more); waves of the kernel before the
    recurrence's that share a segment."""
    kind = {"wkv": 0, "gla": 1, "delta": 2}[mode]
    got = torch.ops.rfq_mix.recurrence_segments(kind, sum(lens), len(lens) + 1, H, 64, vdim)
    return got[0] > len(lens) + 1 and got[1] == (1 if mode == "delta" else waves)


# 1e-5 is for sums of up to 150 tokens; where decays are near one, roundings add up with the root of their number, in the
# reference (one sum a token) as here
def _tol(lens, shift):
    return 1e-5 * max(1.0, max(lens) / 150) ** 0.5 if shift < 0 else 1e-5


# Runs in segments of 128 tokens, which is what the device takes for SEGMENTS and as few heads as here (a state's way into a
# segment is one more sum and product a segment): ends just before, at and behind a segment's end, runs that begin and that
# go on, states of several segments back; rows of wider tensors that a segment's loads of four fit (a pad of 4) and that they
# do not (3: whole runs).  WHOLE: too short, on the average, for the host to cut.
SEGMENTS = [1535, 256, 513, 129, 127]
WHOLE = [700, 1, 129, 128, 255, 257, 400]


def test_which_steps_are_cut():
    for H, vdim in ((2, 64), (4, 128)):
        assert _cut("gla", H, vdim, SEGMENTS) and not _cut("gla", H, vdim, WHOLE)
    assert _cut("wkv", 3, 64, SEGMENTS) and not _cut("wkv", 3, 64, WHOLE)
    assert not _cut("gla", 2, 96, SEGMENTS) and not _cut("delta", 2, 64, SEGMENTS)
    got = torch.ops.rfq_mix.recurrence_segments(1, 2070, 8, 32, 64, 128)
    assert got[0] == 0                                        # as many entries as segments fit: runs stay whole


@pytest.mark.parametrize("shift", [-6.0, 0.0, 60.0])      # decays near one over segments, ordinary, all but zero
@pytest.mark.parametrize("H,Hq,vdim,pad", [(2, 2, 64, 4), (4, 2, 128, 0), (2, 2, 64, 3)])
@pytest.mark.parametrize("lens", [SEGMENTS, WHOLE])
def test_linear_recurrence_in_segments(lens, H, Hq, vdim, pad, shift):
    (out, st), (out_w, st_w) = _linrec("gla", H, Hq, 64, vdim, torch.float32, shift, lens=lens, pad=pad)
    _close(out, out_w, _tol(lens, shift))
    _close(st, st_w, _tol(lens, shift))


@pytest.mark.parametrize("lens", [SEGMENTS, WHOLE, [4096 + 40]])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_wkv_in_segments(dtype, lens):
    tol = 1e-5 * (max(lens) / 150) ** 0.5                    # as above, whatever the decays
    for shift in (-6.0, -2.0, 5.0):
        (out, st), (out_w, st_w) = _wkv(dtype, shift, lens=lens)
        _close(out, out_w, tol if dtype == torch.float32 else 2.0 ** -8)
        _close(st, st_w, tol)


# Sixteen waves to a segment (heads are many, runs long): segments of 1,280 rows, whose last ones are shorter
@pytest.mark.parametrize("mode,H,vdim,lens,dtype", [
    ("wkv", 64, 64, [4136], torch.bfloat16), ("wkv", 40, 64, [3333, 2900], torch.float32),
    ("gla", 64, 128, [4136], torch.bfloat16), ("gla", 40, 64, [3333, 2900], torch.float32)])
def test_segments_of_sixteen_waves(mode, H, vdim, lens, dtype):
    assert _cut(mode, H, vdim, lens, 16)
    for shift in (-6.0, 0.0):
        (out, st), (out_w, st_w) = (_wkv(dtype, shift, lens=lens, H=H) if mode == "wkv" else
                                    _linrec(mode, H, H, 64, vdim, dtype, shift, lens=lens, pad=4))
        tol = 1e-5 * (max(lens) / 150) ** 0.5
        if dtype == torch.float32:
            _close(out, out_w, tol)
        else:
            # 34 million values up to 10 times the rms: where two sums round to different sides, the neighbouring bf16 value,
            # up to 2^-7 of the value away; the sums' own difference is 8 tol of the rms as in fp32
            got, want = out.cpu().double(), out_w.double()
            rms = float(want.square().mean().sqrt())
            assert bool(((got - want).abs() <= 2.0 ** -7 * want.abs() + 8 * tol * max(1.0, rms)).all())
            assert float((got - want).square().mean().sqrt()) <= 2.0 ** -8 * rms
        _close(st, st_w, tol)


@pytest.mark.parametrize("mode,H,vdim,lens", [("gla", 2, 128, SEGMENTS), ("gla", 2, 64, SEGMENTS),
                                              ("delta", 2, 128, [1500, 33, 700])])
def test_linear_recurrence_in_segments_bf16(mode, H, vdim, lens):
    assert _cut(mode, H, vdim, lens)
    (out, st), (out_w, st_w) = _linrec(mode, H, H, 64, vdim, torch.bfloat16, 0.0, lens=lens, pad=4)
    _close(out, out_w, 2.0 ** -8)
    _close(st, st_w, 1e-5)


@pytest.mark.parametrize("lens,other", [(SEGMENTS, 1535), (WHOLE, 700)])
def test_a_non_finite_value_stays_out_of_earlier_segments(lens, other):
    (out, _), (out_w, _) = _linrec("gla", 2, 2, 64, 64, torch.float32, 0.0, lens=lens, spoil=(300, 3, float("inf")), pad=4)
    _close(out[:300], out_w[:300], 1e-5)
    _close(out[other:], out_w[other:], 1e-5)


# The delta rule's segments are whole chunks, as many as the chip has room for: runs of several, of one, of less than one
# and of a chunk, a single long one, all of them whole (the first list); states carried through turns of 64 x 64
@pytest.mark.parametrize("shift", [-6.0, 0.0, 60.0])
@pytest.mark.parametrize("H,Hq,vdim,lens", [(2, 2, 128, [1500, 33, 16, 700]), (2, 2, 128, [1500, 33, 700]), (2, 2, 128, [1600, 16]),
                                            (4, 2, 128, [2100]), (1, 1, 256, [513, 1024])])
def test_delta_rule_in_segments(H, Hq, vdim, lens, shift):
    assert _cut("delta", H, vdim, lens) == (len(lens) < 4)
    (out, st), (out_w, st_w) = _linrec("delta", H, Hq, 64, vdim, torch.float32, shift, lens=lens)
    tol = _tol(lens, shift)
    _close(out, out_w, tol)
    _close(st, st_w, tol)


# As many entries as the chip has room for segments: whole runs, however many of the entries are empty (the one that every
# list here has and `spare`).  Cut into segments all the same, three of five runs, or every one, would begin from states
# that no kernel had made.
@pytest.mark.parametrize("mode,H,lens,spare", [("gla", 32, [1031, 77, 345, 1, 613], 2), ("gla", 64, [700, 800], 1),
                                               ("delta", 16, [600] * 4, 11), ("delta", 32, [1300, 900], 5)])
def test_empty_entries_leave_runs_whole(mode, H, lens, spare):
    # decays near one: what a segment begins from stays in its rows
    (out, st), (out_w, st_w) = _linrec(mode, H, H, 64, 128, torch.float32, -6.0, lens=lens, pad=4, spare=spare)
    tol = 1e-5 * (max(lens) / 150) ** 0.5                    # as for wkv above
    _close(out, out_w, tol)
    _close(st, st_w, tol)


def test_segments_beside_other_work():
    """Workgroups that begin late, between others that are done, read the same: products on another stream hold CUs meanwhile.
    Decays near one, and other inputs in between, so that a state from elsewhere would show."""
    steps = []
    for seed, lens in ((1, [1500, 900]), (2, [2400])):
        g = torch.Generator().manual_seed(seed)
        T, H = sum(lens), 16
        q, k = (torch.nn.functional.normalize(torch.randn(T, H, 64, generator=g), dim=-1).to(DEV) for _ in range(2))
        v, z = torch.randn(T, H, 128, generator=g).to(DEV), torch.randn(T, H * 64, generator=g).to(DEV)
        beta, gate = torch.randn(T, H, generator=g).to(DEV), torch.randn(T, H * 128, generator=g).to(DEV)
        rows, runs = _rows(lens, 23)
        st = torch.randn(2 * len(lens), H, 64, 128, generator=g).to(DEV)
        steps.append((q, k, v, z, beta, gate, st, [r.to(DEV) for r in rows], runs.to(DEV)))

    def call(q, k, v, z, beta, gate, st, rows, runs):
        out, st = torch.empty_like(gate), st.clone()
        rate, zb = torch.full((16,), 0.01, device=DEV), torch.full((16 * 64,), -4.0, device=DEV)
        ops.gated_linear_recurrence(q, k, v, z, rate, zb, 1.0, beta, gate, True, torch.ones(128, device=DEV), 1e-5, 0.125, st, *rows,
                                    out, run_rows=runs)
        return out, st

    alone = [call(*s) for s in steps]
    side, m = torch.cuda.Stream(), torch.randn(2048, 2048, device=DEV)
    torch.cuda.synchronize()
    for i in range(12):
        with torch.cuda.stream(side):
            for _ in range(1 + i % 4):
                m @ m
        for s, want in zip(steps, alone):
            got = call(*s)
            assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), i
    torch.cuda.synchronize()


@pytest.mark.parametrize("size,row,vdim", [(3.0, 2100, 128), (1e20, 1000, 128), (3.0, 700, 256)])
def test_delta_rule_turns_that_grow(size, row, vdim):
    """Keys that turn a state into a larger one, or a state of zeros into what no fp32 holds, leave segments to be done in
    sequence.  Few keys are not zero, so that the growth is not undone; the large one meets a channel that holds nothing."""
    def keys(k, v):
        keep = torch.zeros(len(k), dtype=torch.bool)
        keep[::97] = True
        k[~keep] = 0.0
        k[:1500, :, 0] = 0.0
        k[row], v[row] = 0.0, 0.0
        k[row, :, 0] = size

    (out, st), (out_w, st_w) = _linrec("delta", 2, 2, 64, vdim, torch.float32, -9.0, lens=[1500, 900], keys=keys)
    # a norm of size^2 on a difference: 9 times the roundings of the state it reads
    _close(out, out_w, 1e-4)
    _close(st, st_w, 1e-4)


@pytest.mark.parametrize("mode", ["gla", "delta"])
def test_many_long_runs_share_workgroups_of_128_channels(mode):
    (out, st), (out_w, st_w) = _linrec(mode, 8, 4, 64, 192, torch.float32, 0.0, lens=[81 + i % 7 for i in range(24)] + [3, 16])
    _close(out, out_w, 1e-5)
    _close(st, st_w, 1e-5)


# Entries of queries, keys and states, values and states whose second and third parts bf16 does not hold: the precision is
# that of others, relative to what comes out (of about 1e-36: fp32 itself ends at 2^-149, 1e-9 of it)
@pytest.mark.parametrize("sizes", [(1e-36, 1.0, 1.0, 1.0), (1.0, 1e-36, 1.0, 1e-36), (1.0, 1.0, 1e-36, 1e-36)])
@pytest.mark.parametrize("mode,H,vdim,lens", [("gla", 2, 64, LENS), ("delta", 2, 64, LENS), ("gla", 8, 128, [2100]),
                                              ("delta", 8, 128, [2100]), ("wkv", 3, 64, LENS), ("wkv bf16", 3, 64, LENS)])
def test_small_operands(mode, H, vdim, lens, sizes):
    if mode[:3] == "wkv":
        (out, st), (out_w, st_w) = _wkv(torch.float32 if mode == "wkv" else torch.bfloat16, -2.0, sizes=sizes)
    else:
        (out, st), (out_w, st_w) = _linrec(mode, H, H, 64, vdim, torch.float32, 0.0, lens=lens, pad=4, sizes=sizes)
    for got, want in ((out, out_w), (st, st_w)):
        new = want.double().square().mean().sqrt()
        _close(got.double() / float(new), want.double() / float(new), 1e-5 if got.dtype == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("mode", ["gla", "delta"])
def test_small_operands_that_decays_leave(mode):
    """Sixteen tokens without values read a state that decays take to 1e-37 of itself, each row to the precision of the first.
    (Delta rule: without keys too, so that the rule leaves the state alone.)"""
    g, H = torch.Generator().manual_seed(3), 2
    q, k, v = torch.randn(16, H, 64, generator=g), torch.randn(16, H, 64, generator=g), torch.zeros(16, H, 64)
    if mode == "delta":
        k *= 0.0
    z, st = torch.full((16, H * 64), 5.3), torch.randn(2, H, 64, 64, generator=g)
    rows, runs = _rows([16], 23)
    rows[3][:] += 23                                         # the run goes on from the state
    beta = torch.zeros(16, H) if mode == "delta" else None

    def call(dev, f, **more):
        m = lambda x: None if x is None else x.to(dev)  # noqa: E731
        out, s = torch.empty(16, H * 64, device=dev), m(st.clone())
        f(m(q), m(k), m(v), m(z), m(torch.ones(H)), m(torch.zeros(H * 64)), 1.0, m(beta), m(torch.ones(16, H * 64)), mode == "delta",
          m(torch.ones(64)), 1e-5, 1.0, s, *(m(r) for r in rows), out, **more)
        return out.cpu().double()

    got, want = call(DEV, ops.gated_linear_recurrence, run_rows=runs.to(DEV)), call("cpu", ref.gated_linear_recurrence)
    # sixteen decays of e^-5.3, each to 2^-21 (exponent and exponential): 1e-5; the last row's 6e-37 ends at 2^-149
    assert bool(((got - want).norm(dim=1) <= 2e-5 * want.norm(dim=1)).all())


@pytest.mark.parametrize("value", [3.395e38, 1e-37])         # a part of three would round to infinity; parts below 2^-126
@pytest.mark.parametrize("mode", ["gla", "delta"])
def test_states_at_the_ends_of_fp32(mode, value):
    first = sum(LENS[:7])
    (_, st), (_, st_w) = _linrec(mode, 2, 2, 64, 64, torch.float32, 0.0, spoil=(first + 9, 3, value))
    assert torch.equal(torch.isfinite(st.cpu()), torch.isfinite(st_w))
    for i in range(len(LENS)):                               # every run against its own size
        if i != 7 or value < 1:
            _close(st[i::len(LENS)], st_w[i::len(LENS)], 1e-5)


def test_products_that_end_just_below_the_range():
    """(2^64 - 2^55)^2 is a number of fp32, the square of what it rounds to in bf16 is not: a key's entry and a value in the
    last row of the longest run."""
    def keys(k, v):
        k[-1], v[-1] = 0.0, 0.0
        k[-1, :, 0] = v[-1, 3] = 2.0 ** 64 - 2.0 ** 55

    (_, st), (_, st_w) = _linrec("gla", 2, 2, 64, 64, torch.float32, 0.0, keys=keys)
    assert bool(torch.isfinite(st_w).all())
    _close(st, st_w, 1e-5)


# 40 rows: chunks; 6: token by token; 200 without a list of runs: the scan
@pytest.mark.parametrize("n", [40, 6, 200])
@pytest.mark.parametrize("mode", ["gla", "delta"])
def test_decays_and_steps_keep_32_bits(mode, n):
    """One write, one decay, no reads: the state is beta_0 a_0 and known to a few units in the last place.
    Arguments of the exponentials are whole numbers, or a tiny softplus times a rate that fp32 holds."""
    dim, H = 64, 2
    T, off = n, torch.arange(dim, dtype=torch.float32)
    z = torch.full((T, H, dim), -200.0)                      # softplus and, times any rate, the logarithm 0
    z[1, 0], z[1, 1] = 20.0 + off, -off                      # decays e^-20 .. e^-83; softplus(0 .. -63)
    rate = torch.tensor([1.0, 2.0 ** 10])
    q, v = torch.zeros(T, H, dim), torch.zeros(T, H, dim)
    k, v[0] = q.clone(), 1.0
    k[0] = 1.0 if mode == "gla" else dim ** -0.5
    beta = torch.zeros(T, H)
    beta[0] = torch.tensor([-27.0, -51.0])
    rows, runs = _rows([n], 0)
    state = torch.zeros(2, H, dim, dim)
    m = lambda x: x.to(DEV)  # noqa: E731
    out, st = torch.empty(T, H * dim, device=DEV), m(state)
    ops.gated_linear_recurrence(m(q), m(k), m(v), m(z.view(T, -1)), m(rate), torch.zeros(H * dim, device=DEV), 1.0,
                                m(beta) if mode == "delta" else None, torch.zeros(T, H * dim, device=DEV), True,
                                torch.ones(dim, device=DEV), 1e-5, 1.0, st, *(m(r) for r in rows), out,
                                run_rows=m(torch.tensor([0], dtype=torch.int32)) if n < 200 else None)
    a = torch.exp(-rate.double()[:, None] * torch.log1p(torch.exp(z[1].double())))
    want = a * k[0].double() * (torch.sigmoid(beta[0].double())[:, None] if mode == "delta" else 1.0)
    got = st[1].double().cpu()                               # row_state 0: slot 0, written half 1
    # a unit in the last place (2^-23) for each of exponential, logarithm and quotient, their products'
    # roundings; head 1's argument passes its own three on to the exponential, times itself
    x = rate.double()[:, None] * torch.log1p(torch.exp(z[1].double()))
    tol = torch.stack([torch.full_like(x[0], 6.0), 6.0 + 4.0 * x[1]]) * 2.0 ** -23
    seen = want > 1e-30
    err = ((got - want[:, :, None]).abs() / want[:, :, None])[seen]
    assert bool(seen[0].any()) and bool(seen[1].any())
    assert bool((err <= tol[seen][:, None]).all()), float((err / tol[seen][:, None]).max())


def test_wkv_decays_and_gates_keep_32_bits():
    """The same for wkv: e^z is known to a unit or two in its last place, which the decay takes times itself;
    every value is read alike, so that the norm leaves one and the gate shows."""
    T, H, N = 40, 2, 64
    z, zero = torch.full((T, H, N), -200.0), torch.zeros(T, H * N)
    z[1] = torch.linspace(-4.0, 4.0, H * N).view(H, N)
    k, v, r = zero.clone(), zero.clone(), zero.clone()
    k[0], v[0], r[1] = 1.0, 1.0, 1.0
    gate = torch.linspace(-60.0, 60.0, T * H * N).view(T, -1)
    rows, runs = _rows([T], 0)
    st, out = torch.zeros(2, H, N, N, device=DEV), torch.empty(T, H * N, device=DEV)
    m = lambda x: x.to(DEV)  # noqa: E731
    ops.wkv_recurrence(m(r), m(k), m(v), m(z.view(T, -1)), m(zero[0]), m(zero[0].view(H, N)), m(gate),
                       torch.ones(H * N, device=DEV), 0.0, st, *(m(x) for x in rows), out,
                       run_rows=torch.zeros(1, dtype=torch.int32, device=DEV))
    x = torch.exp(z[1].double())
    err = (st[1].double().cpu() * torch.exp(x)[:, :, None] - 1).abs()
    assert bool((err <= (4 + 3 * x[:, :, None]) * 2.0 ** -23).all()), float((err / (4 + 3 * x[:, :, None])).max() * 2 ** 23)
    g = gate[1].double()
    want = g * torch.sigmoid(g)
    err = (out[1].double().cpu() - want).abs() / want.abs()
    assert bool((err <= 8 * 2.0 ** -23).all()), float(err.max() * 2 ** 23)      # and the norm's square root and quotient

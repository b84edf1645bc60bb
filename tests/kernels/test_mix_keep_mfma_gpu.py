"""attn_keep_window on MFMA tiles: decode rows with the pages split over waves
(csrc/kernels/mix_keep_split.hip) and prompt rows (mix_keep_attn_mfma.hip).  Contexts around pages and
waves, head groups around columns and workgroups, every option."""
import pytest
import torch

from replisense_rfq_amd import ops
from replisense_rfq_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV, BS = "cuda", 32
# (cached tokens, rows): shorter than a page, page edges, one piece per wave and one more, a short
# extend, a padding sequence without rows
SEQS = [(1, 1), (31, 1), (32, 1), (33, 1), (129, 1), (257, 1), (300, 5), (40, 0), (700, 1), (70, 33)]


def _check(H, G, E, vd, shared, seqs=SEQS, spoil=None, prompt=False, spare=0, rising=0.0, **opt):
    g = torch.Generator().manual_seed(H + E + vd)
    need = [(n + BS - 1) // BS for n, _ in seqs]
    perm = torch.randperm(sum(need), generator=g).tolist()
    tables, at = [], 0
    for nb in need:
        tables.append(perm[at:at + nb] + [sum(need)] * (max(need) - nb))
        at += nb
    nb = sum(need) + 1
    k = torch.randn(nb, G, BS, E, generator=g).bfloat16()
    for t in tables if rising else ():           # later pages' scores are larger
        k[t] = (k[t].float() * (1 + rising * torch.arange(len(t))[:, None, None, None])).bfloat16()
    v = k if shared else torch.randn(nb, G, BS, vd, generator=g).bfloat16()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)  # noqa: E731
    ql, kl, bt = i32([r for _, r in seqs]), i32([n for n, _ in seqs]), i32(tables)
    for i, (n, r) in enumerate(seqs):            # what was never written may be anything
        if n % BS:
            for x in (k, v):
                x[tables[i][n // BS], :, n % BS:] = float("nan")
        if spoil is not None and n > spoil and opt.get("window"):
            for x in (k, v):                     # a key that no row sees any more
                x[tables[i][spoil // BS], :, spoil % BS] = float("inf")
    qs, T = torch.cumsum(ql, 0).int() - ql, int(ql.sum())
    q = torch.randn(T, H, E, generator=g) * 2
    q = q.bfloat16().float() if rising else q    # large scores: no part of what is compared is their queries' rounding
    gate = opt.pop("gate", None)
    gate = None if gate is None else torch.randn(T, H * (vd if gate == "output" else 1), generator=g).bfloat16()
    bias = torch.randn(H, generator=g) - 1 if opt.pop("bias", False) else None
    out = torch.zeros(T, H * vd, dtype=torch.bfloat16)
    args = lambda d: (vd, *(x.to(d) for x in (bt, qs, ql, kl)))  # noqa: E731
    kc, vc = (torch.nan_to_num(x.float(), nan=0.0, posinf=0.0).bfloat16() for x in (k, v))
    ref.attn_keep_window(q, kc, vc, *args("cpu"), bias, gate, out, E ** -0.5, opt.get("window", 0),
                         opt.get("keep_first", 0), opt.get("sigmoid", False), opt.get("softcap", 0.0),
                         opt.get("out_mult", 1.0))
    if spare:                                    # a captured step's rows beyond those of its sequences
        q = torch.cat([q, torch.full((spare, H, E), float("nan"))])
        out = torch.cat([out, torch.full((spare, H * vd), 7.0, dtype=torch.bfloat16)])
        gate = None if gate is None else torch.cat([gate, gate[:1].expand(spare, -1)])
    got = torch.full_like(out, 7.0).to(DEV)
    kd = k.to(DEV)
    m = lambda x: None if x is None else x.to(DEV)  # noqa: E731
    items = [(i, b) for i, (_, r) in enumerate(seqs) for b in range((r + 31) // 32)] + [(-1, 0)]   # -1: padding
    ws, wq = (i32([x[j] for x in items]).to(DEV) for j in (0, 1))
    ops.attn_keep_window(q.to(DEV), kd, kd if shared else v.to(DEV), *args(DEV), ws, wq, m(bias), m(gate), got,
                         E ** -0.5, short_rows=0 if prompt else max(r for _, r in seqs), **opt)
    # both sides round to bf16, whose neighbouring values are up to 2^-7 of the value apart: where the
    # fp32 results lie on two sides of a tie they end one spacing apart.  Queries of keys wider than
    # 320 entries enter the products as bf16: four times that.
    tol = 2.0 ** -7 if E <= 320 else 2.0 ** -5
    err = (got.cpu().float() - out.float()).abs()
    assert float(err.max()) <= tol * max(1.0, float(out.float().abs().max()))
    assert float((err / out.float().abs().clamp_min(0.25)).mean()) <= tol


@pytest.mark.parametrize("H,G", [(4, 4), (6, 2), (32, 8), (32, 2), (17, 1), (40, 1)])
def test_head_groups_around_the_columns(H, G):
    _check(H, G, 128, 128, False, softcap=30.0, out_mult=0.6)


@pytest.mark.parametrize("E,vd", [(32, 32), (64, 128), (96, 64), (128, 32)])
def test_plain_sizes(E, vd):
    _check(8, 2, E, vd, False, bias=True, gate="output")


@pytest.mark.parametrize("E,vd,H", [(96, 64, 8), (128, 64, 4), (128, 96, 16), (160, 128, 8), (192, 128, 20),
                                    (320, 256, 16), (576, 512, 32), (576, 512, 5)])
def test_shared_sizes(E, vd, H):
    _check(H, 1, E, vd, True, bias=True, gate="head")


@pytest.mark.parametrize("sigmoid", [False, True])
@pytest.mark.parametrize("window,keep", [(1, 0), (33, 0), (64, 5), (100, 64), (512, 40)])
def test_windows_and_kept_tokens(window, keep, sigmoid):
    _check(32, 8, 128, 128, False, window=window, keep_first=keep, sigmoid=sigmoid, bias=True)
    _check(16, 1, 576, 512, True, window=window, keep_first=keep, bias=True)


def test_many_sequences_take_four_waves():
    _check(32, 8, 128, 128, False, seqs=[(1 + 37 * i % 400, 1) for i in range(40)], softcap=20.0)


def test_a_key_outside_the_window_may_hold_infinities():
    seqs = [(200, 1), (333, 1), (129, 1)]
    _check(32, 8, 128, 128, False, seqs=seqs, spoil=20, window=64, keep_first=4)
    _check(16, 1, 576, 512, True, seqs=seqs, spoil=20, window=64, keep_first=4)


# a row a sequence on the average: pages around the streams of one and of several workgroups
STREAMS = [(1, 1), (32, 1), (33, 1), (128, 1), (129, 1), (300, 2), (40, 0), (512, 1), (513, 1), (700, 1), (1500, 1)]


@pytest.mark.parametrize("H,G", [(17, 1), (32, 1), (33, 1), (64, 1), (48, 2)])
def test_wide_rows_in_streams(H, G):
    _check(H, G, 576, 512, True, seqs=STREAMS, bias=True, gate="head")
    _check(H, G, 576, 512, True, seqs=STREAMS, softcap=20.0, out_mult=0.6, gate="output")
    _check(H, G, 576, 512, True, seqs=STREAMS[5:], window=100, keep_first=40, spoil=50, bias=True)   # no row sees 50
    _check(H, G, 576, 512, True, seqs=STREAMS, window=64, keep_first=5, sigmoid=True, bias=True)
    _check(H, G, 576, 512, True, seqs=STREAMS[4:5], sigmoid=True, softcap=15.0, bias=True)
    _check(H, G, 576, 512, True, seqs=STREAMS[-1:])


# as many rows as sequences, and fewer, but several of one sequence: an extend beside padding in a captured step
EXTENDS = [(300, 1), (40, 0), (700, 16), (64, 1), (33, 5), (90, 0), (161, 2)] + [(40, 0)] * 20


@pytest.mark.parametrize("H,G", [(17, 1), (32, 1), (64, 1), (48, 2)])
def test_wide_rows_of_one_sequence_in_streams(H, G):
    _check(H, G, 576, 512, True, seqs=EXTENDS, bias=True, gate="head")
    _check(H, G, 576, 512, True, seqs=EXTENDS, softcap=20.0, gate="output", spare=2)
    _check(H, G, 576, 512, True, seqs=EXTENDS, window=620, keep_first=5, sigmoid=True, bias=True, spare=1)
    _check(H, G, 576, 512, True, seqs=[(40, 0)] * 63 + [(700, 32)], spare=9)


def _time(n, rows, kv, width):
    """us of a call in a captured graph, so that the host has no part in it: n sequences of rows[i] rows in kv tokens
    each, 32 heads of 576, a table of `width` pages."""
    H, E, vd = 32, 576, 512
    g = torch.Generator().manual_seed(0)
    used = (kv + BS - 1) // BS
    k = torch.randn(n * used, 1, BS, E, generator=g).bfloat16().to(DEV)
    q = torch.randn(sum(rows), H, E, generator=g).to(DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    tables = torch.zeros(n, width, dtype=torch.int32)
    tables[:, :used] = torch.randperm(n * used, generator=g).int().view(n, used)
    out = torch.empty(sum(rows), H * vd, dtype=torch.bfloat16, device=DEV)
    meta = (vd, tables.to(DEV), i32([sum(rows[:i]) for i in range(n)]), i32(rows), i32([kv] * n), i32(range(n)), i32([0] * n))

    def call():
        ops.attn_keep_window(q, k, k, *meta, None, None, out, E ** -0.5, short_rows=32)

    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(10):
            call()
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    best = float("inf")
    for _ in range(8):
        ev[0].record()
        graph.replay()
        ev[1].record()
        torch.cuda.synchronize()
        best = min(best, ev[0].elapsed_time(ev[1]) * 100)
    return best


def test_wide_rows_of_one_sequence_side_by_side():
    """Sixteen rows of one sequence beside padding take about what a row each of sixteen sequences takes (17 us more a
    row when they follow one another)."""
    assert _time(16, [16] + [0] * 15, 700, 22) <= 3 * _time(16, [1] * 16, 700, 22)


@pytest.mark.parametrize("H,G", [(17, 1), (64, 1), (48, 2)])
def test_wide_rows_in_streams_with_a_window(H, G):
    """Windows of 21 pages and more, rows of one page and of one workgroup's pages beside long ones."""
    for padding in (0, 20, 50):                  # the fewer sequences, the more workgroups a row
        seqs = STREAMS + [(40, 0)] * padding
        _check(H, G, 576, 512, True, seqs=seqs[9:], window=641, keep_first=0, spoil=50, bias=True, gate="head")  # no row sees 50
        _check(H, G, 576, 512, True, seqs=seqs, window=700, keep_first=40, softcap=20.0, gate="output")
        _check(H, G, 576, 512, True, seqs=seqs, window=610, keep_first=70, sigmoid=True, bias=True)


@pytest.mark.parametrize("H,G,n", [(64, 1, 64), (32, 1, 128), (17, 1, 85)])
def test_wide_rows_in_streams_of_many_turns(H, G, n):
    """Two or three workgroups a row, up to eight turns of four pages each; the maximum moves in most of them."""
    seqs = [(2016, 1), (1999, 1), (1300, 1), (257, 2), (33, 1)]
    seqs += [(40, 0)] * (n - len(seqs))
    _check(H, G, 576, 512, True, seqs=seqs, rising=0.1, bias=True, gate="head")
    _check(H, G, 576, 512, True, seqs=seqs, rising=0.05, softcap=20.0, gate="output")
    _check(H, G, 576, 512, True, seqs=seqs, window=1000, keep_first=70, sigmoid=True, bias=True)


@pytest.mark.parametrize("H,G,n", [(33, 1, 100), (64, 1, 128), (48, 1, 90), (128, 2, 40)])
def test_wide_rows_of_64_heads_together(H, G, n):
    """Two workgroups a row only where 64 heads share one: one to six pages a workgroup, a last tile without heads."""
    seqs = [(353, 1), (352, 1), (32, 1), (33, 1), (65, 1), (300, 2), (97, 1), (450, 1), (1, 1)]
    seqs += [(40, 0)] * (n - len(seqs))
    _check(H, G, 576, 512, True, seqs=seqs + [(700, 0)], rising=0.1, bias=True, gate="head")
    _check(H, G, 576, 512, True, seqs=seqs + [(700, 0)], softcap=20.0, gate="output", out_mult=0.6)
    _check(H, G, 576, 512, True, seqs=seqs[1:] + [(800, 1)], window=700, keep_first=70, sigmoid=True, bias=True)


@pytest.mark.parametrize("H,G,n", [(64, 1, 128), (128, 2, 40)])
def test_wide_rows_of_eight_pages_and_nine(H, G, n):
    """Where 64 heads share a page, rows of up to eight pages are one workgroup's, longer ones two's; a window's pages count."""
    seqs = [(256, 1), (257, 1), (224, 1), (288, 1), (289, 1), (255, 2)]
    seqs += [(40, 0)] * (n - len(seqs))
    _check(H, G, 576, 512, True, seqs=seqs + [(700, 0)], rising=0.1, bias=True, gate="output")
    _check(H, G, 576, 512, True, seqs=[(800, 1), (815, 1), (832, 1)] + seqs[3:] + [(1000, 0)], window=650, keep_first=33, softcap=20.0)


# Shares of one page and more from fourteen pages to see on
@pytest.mark.parametrize("kv", [417, 448, 449, 480])
def test_wide_rows_of_few_pages_in_streams(kv):
    _check(32, 1, 576, 512, True, seqs=[(kv, 1), (1, 1), (64, 1), (65, 1), (129, 1), (40, 0)], bias=True, gate="head")


def test_few_pages_under_a_wide_table():
    """Workgroups without a page cost nothing: 20 tokens take about as long where the table has room for 8,192 (14.5
    us both; 21.5 when all of them took part)."""
    assert _time(16, [1] * 16, 20, 256) <= 1.25 * _time(16, [1] * 16, 20, 1)


PROMPTS = [(1, 1), (31, 31), (32, 32), (33, 33), (100, 70), (300, 45), (40, 0), (161, 97)]


@pytest.mark.parametrize("H,G,E,vd,shared", [(4, 4, 128, 128, False), (6, 3, 64, 32, False), (8, 2, 96, 128, False),
                                             (3, 1, 32, 64, False), (8, 1, 96, 64, True), (6, 1, 128, 96, True),
                                             (5, 1, 160, 128, True), (4, 1, 192, 128, True), (8, 1, 320, 256, True),
                                             (6, 1, 576, 512, True), (3, 1, 576, 512, True), (16, 1, 576, 512, True)])
def test_prompt_rows(H, G, E, vd, shared):
    _check(H, G, E, vd, shared, seqs=PROMPTS, prompt=True, bias=True, gate="head")
    _check(H, G, E, vd, shared, seqs=PROMPTS, prompt=True, softcap=20.0, out_mult=0.6, gate="output")
    _check(H, G, E, vd, shared, seqs=PROMPTS, prompt=True, window=37, keep_first=5, sigmoid=True, bias=True)
    _check(H, G, E, vd, shared, seqs=PROMPTS, prompt=True, window=64, keep_first=40)


@pytest.mark.parametrize("H,G,E,vd,shared", [(2, 1, 128, 128, False), (24, 4, 64, 64, False), (12, 2, 32, 128, False),
                                             (6, 1, 96, 64, True), (3, 1, 192, 128, True), (4, 2, 160, 128, True)])
def test_prompt_rows_of_small_groups(H, G, E, vd, shared):
    """Both sides of where groups of one and two heads change kernels: three pages and four, 1,024 workgroups."""
    for n in (96, 97):
        seqs = [(n, n), (1, 1), (33, 33), (40, 7), (40, 0)]
        _check(H, G, E, vd, shared, seqs=seqs, prompt=True, bias=True, gate="head")
        _check(H, G, E, vd, shared, seqs=seqs, prompt=True, softcap=20.0, window=37, keep_first=5)
        _check(H, G, E, vd, shared, seqs=seqs, prompt=True, sigmoid=True, bias=True, gate="output")
    per = H // 2 if H // G % 2 == 0 else H
    for items in (1023 // per - 1, 1024 // per):             # one more item is padding
        seqs = [(70, 70)] * (items // 3) + [(32, 32)] * (items % 3)
        _check(H, G, E, vd, shared, seqs=seqs, prompt=True, sigmoid=True, bias=True)
        _check(H, G, E, vd, shared, seqs=seqs, prompt=True, sigmoid=True, bias=True, softcap=20.0)


@pytest.mark.parametrize("H,G,E,vd,shared", [(4, 1, 128, 128, False), (2, 1, 64, 64, False), (1, 1, 32, 32, False),
                                             (4, 1, 96, 64, True), (2, 1, 192, 128, True), (4, 1, 576, 512, True)])
def test_long_chains_of_pages(H, G, E, vd, shared):
    """More pages than any buffer holds, odd and even numbers of them, short blocks beside long ones."""
    seqs = [(1100, 40), (991, 33), (640, 64), (97, 97)]
    _check(H, G, E, vd, shared, seqs=seqs, prompt=True, softcap=20.0)
    _check(H, G, E, vd, shared, seqs=seqs, prompt=True, window=400, keep_first=70, sigmoid=True, bias=True)


@pytest.mark.parametrize("H,G", [(32, 8), (24, 6), (16, 4)])
def test_blocks_whose_heads_are_turned(H, G):
    """More than 8 MB of queries: the heads of a block begin where its number says."""
    seqs = [(33, 33), (64 * 512 // H // 2, 64 * 512 // H // 2), (90, 17)]          # sigmoid weights only
    _check(H, G, 128, 128, False, seqs=seqs, prompt=True, softcap=20.0, gate="head")
    _check(H, G, 128, 128, False, seqs=seqs, prompt=True, window=100, keep_first=40, sigmoid=True, bias=True)


@pytest.mark.parametrize("H,G,E,vd,shared", [(16, 4, 128, 128, False), (8, 2, 64, 32, False), (4, 1, 192, 128, True)])
def test_short_rows_of_four_heads(H, G, E, vd, shared):
    """Both sides of where four heads a workgroup change kernels: pages, and 192 and 256 workgroups."""
    for n in (64, 65, 128, 129):
        seqs = [(n, n), (1, 1), (33, 33), (40, 7), (40, 0)]
        _check(H, G, E, vd, shared, seqs=seqs, prompt=True, sigmoid=True, bias=True, gate="output")
    for wgs in (192, 193, 256, 257):
        items = -(-wgs // (H // 4)) - 1                      # one more item is padding
        for n, opt in ((64, {}), (65, {"softcap": 20.0}), (256, {"sigmoid": True, "bias": True}),
                       (257, {"sigmoid": True, "bias": True, "softcap": 20.0})):
            left = items - (n + 31) // 32
            _check(H, G, E, vd, shared, seqs=[(n, n)] + [(32, 5)] * left, prompt=True, window=90, keep_first=40, **opt)


@pytest.mark.parametrize("H,G", [(4, 1), (16, 2), (5, 1)])
def test_latent_prompt_rows(H, G):
    """Waves of scores and waves of values: one page and up to six, blocks of one row, eight rows and nine, whole ones,
    gates of either kind, all weights, the maximum moving at every page."""
    seqs = [(1, 1), (8, 8), (9, 9), (32, 32), (33, 33), (70, 8), (97, 41), (160, 9), (161, 40), (40, 0)]
    _check(H, G, 576, 512, True, seqs=seqs, prompt=True, rising=0.3, bias=True, gate="head")
    _check(H, G, 576, 512, True, seqs=seqs, prompt=True, rising=0.3, softcap=20.0, out_mult=0.6, gate="output")
    _check(H, G, 576, 512, True, seqs=seqs, prompt=True, window=37, keep_first=5, sigmoid=True, bias=True)
    _check(H, G, 576, 512, True, seqs=seqs, prompt=True, window=64, keep_first=40, sigmoid=True, softcap=15.0, bias=True)


def test_prompt_rows_with_rising_scores():
    """Every page moves the maximum by far: the accumulators are rescaled each time."""
    for shared, E, vd in ((False, 128, 128), (True, 576, 512)):
        g = torch.Generator().manual_seed(1)
        n, nb = 160, 6
        k = torch.randn(nb, 1, BS, E, generator=g)
        k *= (torch.arange(nb * BS).view(nb, 1, BS, 1) // BS + 1)
        k = k.bfloat16()
        v = k if shared else torch.randn(nb, 1, BS, vd, generator=g).bfloat16()
        q = torch.randn(n, 4, E, generator=g) * 3
        i32 = lambda x: torch.tensor(x, dtype=torch.int32)  # noqa: E731
        meta = (vd, i32([[0, 1, 2, 3, 4]]), i32([0]), i32([n]), i32([n]))
        out = torch.zeros(n, 4 * vd, dtype=torch.bfloat16)
        qb = q.bfloat16().float() if shared else q      # wide queries enter the products as bf16
        ref.attn_keep_window(qb, k, v, *meta, None, None, out, 0.5, 0, 0, False)
        got = torch.empty_like(out).to(DEV)
        kd = k.to(DEV)
        ops.attn_keep_window(qb.to(DEV), kd, kd if shared else v.to(DEV), vd, *(x.to(DEV) for x in meta[1:]),
                             i32([0] * 5).to(DEV), i32(list(range(5))).to(DEV), None, None, got, 0.5)
        err = (got.cpu().float() - out.float()).abs()
        # scores of some hundreds, their bf16 hi + lo products to 2^-16: weights to about 1 %
        assert float(err.mean()) <= 0.02 * float(out.float().abs().mean())

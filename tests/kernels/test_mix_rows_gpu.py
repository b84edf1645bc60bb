"""Row kernels that take several channels a lane or several rows a thread (csrc/kernels/mix_par.hip,
mix_wkv.hip, mix_keep_attn.hip) against the row-by-row reference: runs that begin and end inside a
thread's rows, runs shorter than the taps, head sizes, the last rows and columns of a grid."""
import pytest
import torch

from replisense_rfq_amd import ops
from replisense_rfq_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rows(lens, start=23):
    rs, rb, rf, pos = [], [], [], []
    for i, n in enumerate(lens):
        rs += [-1 if i % 5 == 4 else 2 * i + i % 2] * n              # some without a state
        rb += list(range(n))
        rf += list(range(n - 1, -1, -1))
        p = (start, 0, 1)[i % 3]                                     # going on, beginning, one token old
        pos += list(range(p, p + n))
    return [torch.tensor(x, dtype=torch.int32) for x in (rs, rb, rf, pos)]


def _lens(total):
    lens = [1, 2, 3, 8, 1, 9, 15, 1, 1, 4]
    return lens + [total - sum(lens)]


# 8,192 (rows x columns of 1,024 channels) and more are taken eight rows together, fewer singly
@pytest.mark.parametrize("together", [False, True])
@pytest.mark.parametrize("taps,dim,heads,n_unit", [(2, 16, 3, 2), (3, 32, 40, 40), (4, 64, 64, 32), (4, 128, 32, 16),
                                                   (2, 256, 16, 3), (4, 128, 3, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_convolution_by_groups_of_lanes(dtype, taps, dim, heads, n_unit, together):
    g = torch.Generator().manual_seed(dim + taps)
    T = 8192 // -(-heads * dim // 1024) + 3 if together else 50
    C, lens = heads * dim, _lens(T)
    wide = torch.randn(T, C + 8, generator=g).to(dtype)
    w = torch.randn(C, taps, generator=g)
    state = torch.randn(2 * len(lens), taps - 1, C, generator=g)
    rows = _rows(lens)
    got_s, want_s = state.to(DEV), state.clone()
    got, want = torch.empty(T, C, device=DEV), torch.empty(T, C)
    ops.conv_act_heads(wide.to(DEV)[:, 8:], w.to(DEV), got_s, *(r.to(DEV) for r in rows), n_unit, dim, 1e-6, got)
    ref.conv_act_heads(wide[:, 8:], w, want_s, *rows, n_unit, dim, 1e-6, want)
    # up to four products of at most 25 and their sum to 2^-24 each: 100 * 5 * 2^-24 = 3e-5; a unit
    # vector's sum of 256 squares adds less
    torch.testing.assert_close(got.cpu(), want, atol=3e-5, rtol=1e-5)
    assert torch.equal(got_s.cpu(), want_s)


def test_convolution_at_the_ends_of_the_range():
    """What a sigmoid makes of infinities, NaN and where its exponential ends."""
    x = torch.tensor([float("inf"), -float("inf"), float("nan"), 3e38, -3e38, 86.9, -86.9, -87.1, -88.5, -104.0, 0.0, 1e-40,
                      20.0, -20.0, 5.0, -1e-5]).repeat(4)[None].contiguous()
    w, state, i = torch.zeros(64, 4), torch.zeros(2, 3, 64), torch.zeros(1, dtype=torch.int32)
    w[:, 3] = 1.0
    got, want = torch.empty(1, 64, device=DEV), torch.empty(1, 64)
    ops.conv_act_heads(x.to(DEV), w.to(DEV), state.to(DEV), *(r.to(DEV) for r in (i, i, i, i)), 0, 16, 1e-6, got)
    ref.conv_act_heads(x, w, state, i, i, i, i, 0, 16, 1e-6, want)
    # below -88.7 zero for less than 88.7 e^-88.7 = 3e-37; four roundings of 2^-24, 20 of them in the reference's exponential
    torch.testing.assert_close(got.cpu(), want, atol=2e-36, rtol=2e-6, equal_nan=True)


def test_convolution_of_far_negative_sums():
    """Results are normal numbers down to -88.7, where the exponential ends, in all three kernels: heads of whole groups of
    lanes, in fours, and any."""
    for dim, C in ((16, 64), (20, 40), (3, 6)):
        x = -torch.linspace(86.5, 88.7, C).clone()[None].contiguous()
        x[0, 1] = 7.0                                        # beside one in the middle of the range
        w, state, i = torch.zeros(C, 4), torch.zeros(2, 3, C), torch.zeros(1, dtype=torch.int32)
        w[:, 3] = 1.0
        got, want = torch.empty(1, C, device=DEV), x.double() / (1 + torch.exp(-x.double()))
        ops.conv_act_heads(x.to(DEV), w.to(DEV), state.to(DEV), *(r.to(DEV) for r in (i, i, i, i)), 0, dim, 1e-6, got)
        # an exponential begins with the product of -x and log2 e, between 64 and 128 and so rounded by up to 2^-18, of which
        # ln 2 are the result's, 2.6e-6; the other four roundings, 2^-24 each, make less than the rest of 2^-18, 3.8e-6
        assert float((got.cpu().double() / want - 1).abs().max()) <= 2.0 ** -18


# the last three: four rows a thread; the last: past the caches
@pytest.mark.parametrize("T,d", [(47, 4), (50, 2052), (1371, 2052), (4099, 64), (3301, 4100)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_token_shift_four_channels_a_lane(dtype, T, d):
    g = torch.Generator().manual_seed(d)
    lens = _lens(T)
    x, mu, prev = torch.randn(T, d, generator=g), torch.randn(5, d, generator=g), torch.randn(2 * len(lens), d, generator=g)
    rows = _rows(lens)
    got_p, want_p = prev.to(DEV), prev.clone()
    got, want = torch.empty(5, T, d, dtype=dtype, device=DEV), torch.empty(5, T, d, dtype=dtype)
    ops.token_shift_mix(x.to(DEV), mu.to(DEV), got_p, *(r.to(DEV) for r in rows), got)
    ref.token_shift_mix(x, mu, want_p, *rows, want)
    # a + (b - a) mu with terms up to 50, two roundings of 2^-24; bf16: the neighbouring value
    torch.testing.assert_close(got.cpu(), want, atol=1e-5, rtol=2.0 ** -7 if dtype == torch.bfloat16 else 1e-6)
    assert torch.equal(got_p.cpu(), want_p)


# 256 rows: a thread per chunk of a row and a wave for the sines; 257: blocks of 256 threads
@pytest.mark.parametrize("T", [256, 257])
@pytest.mark.parametrize("H,G,dim", [(2, 1, 16), (40, 8, 128), (72, 8, 128), (3, 1, 10)])
@pytest.mark.parametrize("taps,norm_all", [(0, True), (0, False), (1, True), (4, False), (4, True), (6, True)])
def test_norm_and_rotation_by_number_of_rows(taps, norm_all, H, G, dim, T):
    g = torch.Generator().manual_seed(H + taps)
    W, lens, page = (H + 2 * G) * dim, _lens(T), 32
    proj, state = torch.randn(T, W, generator=g), torch.randn(2 * len(lens), max(taps - 1, 0), W, generator=g)
    qn, kn = (torch.randn(n * dim if norm_all else dim, generator=g) for n in (H, G))
    w, freq = torch.randn(max(taps, 1), W, generator=g), 1000.0 ** -torch.linspace(0, 1, dim // 2)
    rows = _rows(lens)
    slots = torch.randperm(9 * page, generator=g)[:T].to(torch.int32)
    slots[5] = -1

    def call(dev, f, st):
        m = lambda x: x.to(dev)  # noqa: E731
        q, kc, vc = torch.empty(T, H, dim, device=dev), *(torch.full((9, G, page, dim), 7.0, device=dev) for _ in range(2))
        rs, rb, rf, pos = (m(r) for r in rows)
        f(m(proj), None, m(qn), m(kn), norm_all, dim, 1e-5, pos, m(freq), 1.5, 0, 0, m(slots), kc, vc, H, G, dim, dim,
          dim, 0, q, conv=(m(w), st, rs, rb, rf) if taps else None)
        return q, kc, vc, st

    got, want = call(DEV, ops.qk_norm_rotary_append, state.to(DEV)), call("cpu", ref.qk_norm_rotary_append, state.clone())
    # a normed entry times weight and sine, up to 30, after some ten roundings of 2^-24; values: sums
    # of up to six products of at most 25
    for a, b in zip(got, want):
        torch.testing.assert_close(a.cpu(), b, atol=3e-5, rtol=1e-5)


# Several rows a workgroup, two chunks a thread or one: rows that its groups do not divide, runs that begin and end inside
# a group, rotated parts behind plain ones, rows of one wave's chunks and of ten, columns that no thread has alone
@pytest.mark.parametrize("T", [1, 66, 1030, 2101])
@pytest.mark.parametrize("H,G,dim,nrot,off", [(2, 1, 64, 16, 32), (20, 3, 64, 32, 0), (64, 8, 128, 32, 64), (5, 5, 40, 0, 0)])
@pytest.mark.parametrize("conv", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_norm_and_rotation_of_rows_one_after_another(dtype, conv, H, G, dim, nrot, off, T):
    g = torch.Generator().manual_seed(T + H)
    W, lens, page = (H + 2 * G) * dim, _lens(T) if T > 45 else [T], 32
    wide, state = torch.randn(T, W + 8, generator=g).to(dtype), torch.randn(2 * len(lens), 3, W, generator=g)
    qn, kn, bias = (torch.randn(n, generator=g) for n in (H * dim, G * dim, W))
    w, freq = torch.randn(4, W, generator=g), 1000.0 ** -torch.linspace(0, 1, nrot)
    rows, pages = _rows(lens), T // page + 2
    slots = torch.randperm(pages * page, generator=g)[:T].to(torch.int32)
    if T > 5:
        slots[5] = -1

    def call(dev, f, st):
        m = lambda x: x.to(dev)  # noqa: E731
        q = torch.empty(T, H, dim, device=dev)
        kc, vc = (torch.full((pages, G, page, dim), 7.0, device=dev, dtype=dtype) for _ in range(2))
        rs, rb, rf, pos = (m(r) for r in rows)
        f(m(wide)[:, 8:], None if conv else m(bias), m(qn), m(kn), True, dim, 1e-5, pos, m(freq), 1.5, off, off, m(slots), kc,
          vc, H, G, dim, dim, dim, 0, q, conv=(m(w), st, rs, rb, rf) if conv else None)
        return q, kc, vc, st

    got, want = call(DEV, ops.qk_norm_rotary_append, state.to(DEV)), call("cpu", ref.qk_norm_rotary_append, state.clone())
    # as above; angles of up to 2,100 radians round by 1.2e-4 of them: 30 times the sine's error of 2^-13; bf16 pages: the
    # neighbouring value, up to 2^-7 away
    for a, b, rel in zip(got, want, (0.0, 2.0 ** -7, 2.0 ** -7, 0.0)):
        torch.testing.assert_close(a.cpu().float(), b.float(), atol=3e-5 if T < 100 else 4e-3, rtol=1e-5 + (rel if dtype == torch.bfloat16 else 0.0))


# Runs of one to seven rows everywhere: workgroups that begin at any row of a run, with and without a state
@pytest.mark.parametrize("T,H,G,dim", [(2101, 20, 3, 64), (1030, 40, 8, 128), (300, 64, 8, 128), (1030, 56, 8, 128), (1030, 64, 8, 128), (2060, 56, 8, 128)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_convolved_rows_of_short_runs(monkeypatch, dtype, T, H, G, dim):
    lens = [1 + i % 7 for i in range(T // 4)]
    lens = lens[:next(i for i in range(len(lens)) if sum(lens[:i + 1]) >= T - 7) + 1]
    monkeypatch.setitem(globals(), "_lens", lambda total: lens + [total - sum(lens)] * (total > sum(lens)))
    test_norm_and_rotation_of_rows_one_after_another(dtype, True, H, G, dim, 32, 0, T)


# More rows than one round of workgroups takes in sixteens: two rounds of eight or nine
@pytest.mark.parametrize("T", [4096, 4104])
def test_norm_and_rotation_of_rows_in_rounds(T):
    test_norm_and_rotation_of_rows_one_after_another(torch.bfloat16, False, 64, 8, 128, 32, 64, T)


# The same without values: the rotated ends of query heads, one key of which only the leading entries are normed
@pytest.mark.parametrize("T", [3, 1030])
@pytest.mark.parametrize("neighbours", [False, True])
@pytest.mark.parametrize("H,qw,latent,rot", [(5, 48, 96, 16), (32, 192, 512, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rotated_ends_and_a_partly_normed_key(dtype, H, qw, latent, rot, neighbours, T):
    g = torch.Generator().manual_seed(T + H)
    E, page, pages = latent + rot, 32, T // 32 + 2
    proj = torch.randn(T, H * qw + E + 8, generator=g).to(dtype)
    kn, freq = torch.randn(latent, generator=g), 1000.0 ** -torch.linspace(0, 1, rot // 2)
    pos, slots = torch.arange(7, T + 7, dtype=torch.int32), torch.randperm(pages * page, generator=g)[:T].to(torch.int32)
    slots[1] = -1

    def call(dev, f):
        m = lambda x: x.to(dev)  # noqa: E731
        q, pool = torch.full((T, H, E), 3.0, device=dev), torch.full((pages, 1, page, E), 7.0, device=dev, dtype=dtype)
        f(m(proj), None, None, m(kn), False, latent, 1e-5, m(pos), m(freq), 1.5, qw - rot, latent, m(slots), pool, None, H, 1,
          qw, E, 0, 2, q[:, :, latent:], neighbours=neighbours)
        return q, pool

    # as above
    for a, b, rel in zip(call(DEV, ops.qk_norm_rotary_append), call("cpu", ref.qk_norm_rotary_append), (0.0, 2.0 ** -7)):
        torch.testing.assert_close(a.cpu().float(), b.float(), atol=3e-5 if T < 100 else 4e-3, rtol=1e-5 + (rel if dtype == torch.bfloat16 else 0.0))


def test_rotations_of_wide_heads_in_long_steps():
    """512 sines a row of a step with sixteen rows a workgroup: they leave room for fewer."""
    H, w, T, page = 8, 1024, 3850, 32
    g = torch.Generator().manual_seed(1)
    W, pages, slots = (H + 2) * w, T // page + 1, torch.arange(T, dtype=torch.int32)
    proj, freq, pos = torch.randn(T, W, generator=g).bfloat16(), 1000.0 ** -torch.linspace(0, 1, w // 2), torch.arange(T, dtype=torch.int32) % 100

    def call(dev, f):
        m = lambda x: x.to(dev)  # noqa: E731
        q = torch.empty(T, H, w, device=dev)
        kc, vc = (torch.zeros(pages, 1, page, w, device=dev, dtype=torch.bfloat16) for _ in range(2))
        f(m(proj), None, None, None, False, w, 1e-5, m(pos), m(freq), 1.0, 0, 0, m(slots), kc, vc, H, 1, w, w, w, 0, q, neighbours=True)
        return q, kc, vc

    # as above, angles of up to 100 radians
    for a, b, rel in zip(call(DEV, ops.qk_norm_rotary_append), call("cpu", ref.qk_norm_rotary_append), (0.0, 2.0 ** -7, 2.0 ** -7)):
        torch.testing.assert_close(a.cpu().float(), b.float(), atol=3e-4, rtol=1e-5 + rel)

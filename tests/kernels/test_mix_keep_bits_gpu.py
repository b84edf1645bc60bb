"""attn_keep_window on MFMA tiles against 64-bit attention: options together, and the precision of
queries, scores and weights, seen through values that cancel."""
import pytest
import torch

from replisense_rfq_amd import ops

pytestmark = pytest.mark.gpu
DEV, BS = "cuda", 32


def _exact(q, k, v, bias, scale, window, keep_first, sigmoid, softcap):
    """q [T, H, E], k [L, G, E], v [L, G, vd]; the rows are the sequence's last T.  64 bits."""
    T, H, L, rep = q.shape[0], q.shape[1], k.shape[0], q.shape[1] // k.shape[1]
    k, v = (x.double().repeat_interleave(rep, 1) for x in (k, v))
    i, j = torch.arange(L - T, L)[:, None], torch.arange(L)[None]
    ok = (j <= i) & ((i - j < window) | (j < keep_first) if window else True)
    s = torch.stack([q.double()[:, h] @ k[:, h].t() for h in range(H)]) * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    b = None if bias is None else bias.double()[:, None, None]
    if sigmoid:
        w = torch.sigmoid(s + b) * ok
    else:
        s = s.masked_fill(~ok, float("-inf"))
        w = torch.softmax(s if b is None else torch.cat([s, b.expand(H, T, 1)], -1), -1)[..., :L]
    return torch.stack([w[h] @ v[:, h] for h in range(H)], 1)


def _both(q, k, v, prompt, bias=None, scale=1.0, window=0, keep_first=0, sigmoid=False, softcap=0.0):
    """(ops.attn_keep_window, 64 bits), [T, H, vd]; v None: the keys' leading entries."""
    T, H, E = q.shape
    L, G = k.shape[:2]
    nb = (L + BS - 1) // BS
    pages = lambda x: torch.cat([x, torch.zeros(nb * BS - L, *x.shape[1:], dtype=x.dtype)]) \
        .view(nb, BS, G, -1).transpose(1, 2).flip(0).contiguous().to(DEV)  # noqa: E731
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    kd = pages(k)
    vd = E - 64 if v is None else v.shape[2]
    out = torch.empty(T, H * vd, dtype=torch.bfloat16, device=DEV)
    blocks = range((T + 31) // 32)
    ops.attn_keep_window(q.to(DEV), kd, kd if v is None else pages(v), vd, i32(*range(nb - 1, -1, -1))[None], i32(0),
                         i32(T), i32(L), i32(*[0 for _ in blocks]), i32(*blocks), None if bias is None else bias.to(DEV),
                         None, out, scale, window=window, keep_first=keep_first, sigmoid=sigmoid, softcap=softcap,
                         short_rows=0 if prompt else T)
    want = _exact(q, k, k[..., :vd] if v is None else v, bias, scale, window, keep_first, sigmoid, softcap)
    return out.view(T, H, vd).double().cpu(), want


@pytest.mark.parametrize("prompt", [True, False])
@pytest.mark.parametrize("H,G,E,vd", [(8, 2, 128, 128), (3, 3, 64, 32), (8, 1, 320, 0), (4, 1, 576, 0)])
def test_sigmoid_weights_of_capped_scores(H, G, E, vd, prompt):
    """The cap binds: scores of 6 rms under a cap of 4, weights of some hundred keys."""
    g = torch.Generator().manual_seed(E + H)
    T, L = (70, 150) if prompt else (2, 150)
    q, k = torch.randn(T, H, E, generator=g) * 6, torch.randn(L, G, E, generator=g).bfloat16()
    v = torch.randn(L, G, vd, generator=g).bfloat16() if vd else None
    got, want = _both(q, k, v, prompt, torch.randn(H, generator=g) - 1, E ** -0.5, 90, 5, True, 4.0)
    # half a bf16 step of the result, and of the wide queries: 2^-9 of scores of 6, whose weights
    # of 150 keys add up in quadrature
    err, rms = (got - want).abs(), want.square().mean().sqrt()
    assert bool((err <= 2.0 ** -8 * want.abs() + 2.0 ** -5 * rms).all())


def _cancelling(T, L, H, G, E, vd, step, seed):
    """Queries of 4,108 and a little more (``step``: of 4,096 and a multiple of it), keys +-1 in pairs
    that cancel: the scores are the differences of the small parts."""
    g = torch.Generator().manual_seed(seed)
    small = torch.randn(T, H, E, generator=g)
    small = (small * 4).round() * step if step else 12.0 + small / 4
    s = torch.randint(0, 2, (L, G, E // 2), generator=g) * 2.0 - 1.0
    k = torch.stack([s, -s], -1).reshape(L, G, E).bfloat16()
    v = torch.randn(L, G, vd, generator=g).bfloat16() if vd else None
    return 4096.0 + small, k, v


def _near(got, want, part):
    """Half a bf16 step of the value, and ``part`` of the results' rms."""
    err, rms = (got - want).abs(), want.square().mean().sqrt()
    assert bool((err <= 2.0 ** -8 * want.abs() + part * rms).all()), float(((err - 2.0 ** -8 * want.abs()) / rms).max())


@pytest.mark.parametrize("H,E", [(4, 576), (6, 576), (3, 576), (8, 320)])
def test_wide_prompt_queries_enter_as_they_are(H, E):
    """Queries that bf16 holds exactly are not rounded again, whatever the scale."""
    q, k, _ = _cancelling(70, 150, H, 1, E, 0, 32, E)
    _near(*_both(q, k, None, True, scale=(2 * E) ** -0.5 / 32.0), 2.0 ** -8)


@pytest.mark.parametrize("H,G,E", [(3, 1, 576), (5, 1, 320), (14, 2, 320), (9, 3, 576), (2, 1, 576), (3, 3, 320)])
def test_wide_prompts_of_heads_that_leave_waves_idle(H, G, E):
    """Groups of 3, 5, 7, 3, 2 and 1 heads: nothing is written past a group's last one."""
    g = torch.Generator().manual_seed(H)
    q, k = torch.randn(70, H, E, generator=g), torch.randn(150, G, E, generator=g).bfloat16()
    got, want = _both(q.bfloat16().float(), k, None, True, torch.randn(H, generator=g), E ** -0.5)
    _near(got, want, 2.0 ** -9)


@pytest.mark.parametrize("prompt", [True, False])
@pytest.mark.parametrize("H,G,E,vd", [(8, 2, 128, 128), (16, 1, 128, 128), (4, 1, 576, 0), (16, 1, 576, 0)])
@pytest.mark.parametrize("opt", [{}, {"sigmoid": True}, {"softcap": 20.0}])
def test_a_query_that_is_no_number_shows(H, G, E, vd, prompt, opt):
    g = torch.Generator().manual_seed(3)
    q, k = torch.randn(1, H, E, generator=g), torch.randn(150, G, E, generator=g).bfloat16()
    v = torch.randn(150, G, vd, generator=g).bfloat16() if vd else None
    q[0, 1, 5] = float("nan")
    for bias in (torch.zeros(H), None)[:1 if opt.get("sigmoid") else 2]:
        got, _ = _both(q, k, v, prompt, bias, E ** -0.5, **opt)
        assert bool(got[0, 1].isnan().all()) and bool(got[0, [0, *range(2, H)]].isfinite().all())


# Fewer than 16 heads share a key head: fp32 queries, weights and scores.
GROUPS = [(8, 2, 128, 128), (3, 3, 64, 32), (15, 1, 96, 64), (4, 1, 320, 0), (15, 1, 576, 0), (5, 1, 576, 0)]


@pytest.mark.parametrize("H,G,E,vd", GROUPS)
def test_decode_weights_keep_32_bits(H, G, E, vd):
    """Values that cancel in neighbouring keys, scores of rms 2^-12: the results are differences of
    nearly equal weights.  Weights to 2^-24: 2^-12 of the results each way; to 16 bits: 2^-6."""
    g = torch.Generator().manual_seed(E + 1)
    L = 160
    k, q = torch.randn(L, G, E, generator=g).bfloat16(), torch.randn(2, H, E, generator=g)
    if vd:
        v = torch.randn(L // 2, G, vd, generator=g).bfloat16()
        v = torch.stack([v, -v], 1).view(L, G, vd)
    else:                                       # the keys are the values: they differ in the last 64 entries
        v = None
        k[1::2, :, :E - 64] = -k[0::2, :, :E - 64]
        q[..., :E - 64] = 0.0
    n = 64 if v is None else E
    got, want = _both(q, k, v, False, scale=2.0 ** -12 * n ** -0.5)
    _near(got[1:], want[1:], 2.0 ** -8)         # the last row: an even number of keys


@pytest.mark.parametrize("H,G,E,vd", GROUPS)
def test_an_infinite_query_under_a_cap(H, G, E, vd):
    """The head's scores are +-cap, whatever the other entries."""
    g = torch.Generator().manual_seed(E + 3)
    q, k = torch.randn(1, H, E, generator=g), torch.randn(150, G, E, generator=g).bfloat16()
    v = torch.randn(150, G, vd, generator=g).bfloat16() if vd else None
    q[0, 1, 3] = float("inf")
    _near(*_both(q, k, v, False, scale=E ** -0.5, softcap=3.0), 2.0 ** -9)


@pytest.mark.parametrize("H,G,E,vd", GROUPS)
def test_decode_scores_under_a_wide_cap(H, G, E, vd):
    """A cap far above the scores leaves them as they are."""
    g = torch.Generator().manual_seed(E + 2)
    q, k = torch.randn(2, H, E, generator=g) * 2, torch.randn(150, G, E, generator=g).bfloat16()
    v = torch.randn(150, G, vd, generator=g).bfloat16() if vd else None
    _near(*_both(q, k, v, False, scale=E ** -0.5, softcap=2.0 ** 17), 2.0 ** -9)


# prompts, and decode rows of 16 heads a key head or more: weights in two parts, 16 bits
@pytest.mark.parametrize("H,G,E,vd,prompt", [(8, 2, 128, 128, True), (4, 4, 64, 32, True), (6, 1, 192, 0, True), (8, 1, 320, 0, True),
                                             (4, 1, 576, 0, True), (32, 2, 128, 128, False), (16, 1, 192, 0, False),
                                             (20, 1, 320, 0, False), (16, 1, 576, 0, False)])
def test_weights_keep_16_bits(H, G, E, vd, prompt):
    """The values of neighbouring keys cancel, scores of rms 2^-6: the results are 2^-6 of what goes in.  Two
    parts of a weight, 2^-17: 2^-11 of the results; one, 2^-9: an eighth of them.  The last row has an even
    number of keys."""
    g = torch.Generator().manual_seed(E + 7)
    T, L = (34, 160) if prompt else (2, 160)
    k, q = torch.randn(L, G, E, generator=g).bfloat16(), torch.randn(T, H, E, generator=g).bfloat16().float()
    if vd:
        v = torch.randn(L // 2, G, vd, generator=g).bfloat16()
        v, n = torch.stack([v, -v], 1).view(L, G, vd), E
    else:                                       # the keys are the values: they differ in the last 64 entries
        v, n = None, 64
        k[1::2, :, :E - 64] = -k[0::2, :, :E - 64]
        q[..., :E - 64] = 0.0
    got, want = _both(q, k, v, prompt, scale=2.0 ** -6 * n ** -0.5)
    _near(got[-1:], want[-1:], 2.0 ** -7)

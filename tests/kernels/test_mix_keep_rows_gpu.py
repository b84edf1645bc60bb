"""attn_keep_window, decode rows of many sequences or many rows: wide latents on the prompts' kernel, its
columns heads of a row; fewer waves to a workgroup; workgroups that take several rows one after another."""
import pytest
import torch

from replisense_rfq_amd import ops
from tests.kernels.test_mix_keep_bits_gpu import _both, _near
from tests.kernels.test_mix_keep_mfma_gpu import _check

pytestmark = pytest.mark.gpu


# more than 256 (row, 16 heads): one, two and four heads' blocks a workgroup, a group that ends inside a wave's
# columns and inside a workgroup's waves
@pytest.mark.parametrize("H,T", [(128, 33), (128, 160), (72, 60), (40, 90), (64, 65), (17, 130), (16, 260)])
@pytest.mark.parametrize("E", [576, 320])
@pytest.mark.parametrize("opt", [{}, {"softcap": 4.0}, {"sigmoid": True, "window": 40, "keep_first": 5},
                                 {"sigmoid": True, "softcap": 4.0}, {"window": 33}])
def test_wide_rows(H, T, E, opt):
    g = torch.Generator().manual_seed(H + E)
    q, k = (torch.randn(T, H, E, generator=g) * 4).bfloat16().float(), torch.randn(T + 20, 1, E, generator=g).bfloat16()
    bias = torch.randn(H, generator=g) if opt.get("sigmoid") or "window" in opt else None
    got, want = _both(q, k, None, False, bias, E ** -0.5, **opt)
    _near(got, want, 2.0 ** -9)


LATENTS = [(16, 280), (72, 60), (128, 40)]


@pytest.mark.parametrize("H,n", LATENTS)
def test_wide_rows_of_many_sequences(H, n):
    """Contexts around pages, sequences without rows and with more rows than their neighbours."""
    seqs = [(1 + 13 * i % 100, 0 if i % 17 == 16 else 1) for i in range(n)] + [(70, 9), (33, 33)]
    _check(H, 1, 576, 512, True, seqs=seqs, bias=True, gate="head")
    _check(H, 1, 320, 256, True, seqs=seqs, softcap=20.0, out_mult=0.6, gate="output")
    out_of_sight = [(60 + 13 * i % 100, 1) for i in range(n)] + [(70, 9)]
    _check(H, 1, 576, 512, True, seqs=out_of_sight, spoil=20, window=30, keep_first=4)


@pytest.mark.parametrize("rows", [1, 2, 4])
@pytest.mark.parametrize("H,G,E,vd,shared", [(32, 2, 128, 128, False), (40, 1, 96, 64, True)])
def test_many_sequences_of_large_groups(H, G, E, vd, shared, rows):
    """Four, two and one waves to a workgroup."""
    seqs = [(rows + 13 * i % 100, rows) for i in range(260 // G)]
    _check(H, G, E, vd, shared, seqs=seqs, window=50, keep_first=3, bias=True)


def test_many_rows_of_few_sequences():
    """Column tiles side by side beyond four, and one after another."""
    for H, G, E, vd, shared in ((32, 8, 128, 128, False), (20, 1, 192, 128, True), (4, 1, 576, 512, True)):
        _check(H, G, E, vd, shared, seqs=[(90, 32), (33, 1), (40, 20)], softcap=20.0)
    _check(32, 8, 128, 128, False, seqs=[(33, 1)] * 70 + [(90, 32)])


def test_more_column_tiles_than_a_grid_holds():
    """One sequence of 33,000 rows with 32 heads, as a decode section and as a prompt."""
    T, H, E, BS = 33000, 32, 32, 32
    g = torch.Generator().manual_seed(1)
    q = torch.randn(T, H, E, generator=g).cuda()
    nb = (T + BS - 1) // BS
    k, v = (torch.randn(nb, 1, BS, E, generator=g).bfloat16().cuda() for _ in range(2))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    blocks = list(range((T + 31) // 32))
    out = []
    for short in (T, 0):
        out.append(torch.zeros(T, H * E, dtype=torch.bfloat16, device="cuda"))
        ops.attn_keep_window(q, k, v, E, i32([list(range(nb))]), i32([0]), i32([T]), i32([T]), i32([0] * len(blocks)),
                             i32(blocks), None, None, out[-1], E ** -0.5, window=40, short_rows=short)
    # both round the same sums to bf16: neighbouring values at a tie
    torch.testing.assert_close(out[0].float(), out[1].float(), atol=1e-3, rtol=2.0 ** -7)

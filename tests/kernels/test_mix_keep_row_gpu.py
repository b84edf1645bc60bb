"""attn_keep_window, decode rows of groups of up to eight heads with the parts of queries and weights in MFMA columns
(csrc/kernels/mix_keep_row.hip): groups around four and eight heads, contexts around pages and waves, sequences without
rows and with more than one, rows of captured steps that no sequence has, pages read through the caches and past them, all of fp32's bits."""
import pytest
import torch

from replisense_rfq_amd import ops
from tests.kernels.test_mix_keep_bits_gpu import _both, _near
from tests.kernels.test_mix_keep_mfma_gpu import _check

pytestmark = pytest.mark.gpu
# no more rows than sequences; one of seven rows and one without any between others
SEQS = [(1, 1), (31, 1), (32, 1), (33, 1), (40, 0), (129, 1), (257, 1), (290, 1), (70, 7), (700, 1)] + [(9, 0)] * 5


@pytest.mark.parametrize("H,G", [(8, 2), (4, 4), (6, 2), (5, 1), (16, 2), (7, 1)])
@pytest.mark.parametrize("E", [64, 128])
@pytest.mark.parametrize("opt", [{}, {"softcap": 30.0, "out_mult": 0.6, "gate": "output"}, {"bias": True, "gate": "head"},
                                 {"bias": True, "sigmoid": True, "window": 64, "keep_first": 5}, {"window": 33},
                                 {"bias": True, "sigmoid": True, "softcap": 20.0}])
def test_groups_around_the_columns(H, G, E, opt):
    _check(H, G, E, E, False, seqs=SEQS, **opt)


@pytest.mark.parametrize("H,G", [(32, 8), (3, 1), (2, 1), (4, 4), (40, 8)])
@pytest.mark.parametrize("E", [64, 128])
def test_extends_in_captured_steps(H, G, E):
    """As many rows as sequences, several of them a sequence's: rows that share columns and rows on their own, from any
    row of the step on, more than 64 sequences, rows beyond the last one's."""
    for opt in ({"softcap": 30.0}, {"window": 64, "keep_first": 5, "bias": True}):
        _check(H, G, E, E, False, seqs=[(600, 12), (1, 1), (33, 2)] + [(1, 0)] * 14, spare=2, **opt)
        _check(H, G, E, E, False, seqs=[(40, 1), (290, 7), (70, 32), (9, 3)] + [(1, 0)] * 70 + [(257, 5)], spare=27, **opt)


def test_extends_cost_no_more_than_their_rows():
    """Sixteen rows of three sequences, pages of 600 tokens, against a row of sixteen each: rows that went one after
    another took nine times as long, side by side they take as long."""
    g = torch.Generator().manual_seed(3)
    k, v = (torch.randn(305, 8, 32, 128, generator=g).bfloat16().cuda() for _ in range(2))
    q, out = torch.randn(16, 32, 128, generator=g).cuda(), torch.zeros(16, 4096, dtype=torch.bfloat16, device="cuda")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    bt, zero, ids = i32([[19 * s + i for i in range(19)] for s in range(16)]), i32([0] * 16), i32(range(16))

    def least(rows):
        ql = i32(rows)
        args = bt, (torch.cumsum(ql, 0) - ql).int(), ql, i32([600] * 16), ids, zero
        ops.attn_keep_window(q, k, v, 128, *args, None, None, out, 128 ** -0.5, short_rows=32)
        took = []
        for _ in range(20):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            torch.cuda.synchronize()
            torch.cuda._sleep(200_000)                       # the calls are queued before the first one starts
            a.record()
            for _ in range(8):
                ops.attn_keep_window(q, k, v, 128, *args, None, None, out, 128 ** -0.5, short_rows=32)
            b.record()
            torch.cuda.synchronize()
            took.append(a.elapsed_time(b))
        return min(took)

    assert least([12, 3, 1] + [0] * 13) <= 4 * least([1] * 16)


@pytest.mark.parametrize("H,G,E", [(8, 2, 128), (16, 2, 64)])
def test_infinities_out_of_sight(H, G, E):
    _check(H, G, E, E, False, seqs=[(n + 60, r) for n, r in SEQS], spoil=20, window=30, keep_first=4)


@pytest.mark.parametrize("H,G", [(32, 8), (64, 8)])
def test_pages_past_the_caches(H, G):
    """Tables with room for more than 96 MB: four waves to a workgroup, and eight."""
    _check(H, G, 128, 128, False, seqs=[(200 + 37 * i % 700, 1) for i in range(40)], softcap=30.0)
    _check(H, G, 128, 128, False, seqs=[(9600, 1), (100, 1), (33, 1)], window=1024, keep_first=64)


@pytest.mark.parametrize("H,G,E", [(8, 2, 128), (3, 3, 64), (16, 2, 128), (5, 1, 64)])
def test_weights_keep_32_bits(H, G, E):
    """Values that cancel in neighbouring keys, scores of rms 2^-12: the results are differences of nearly equal
    weights.  Weights to 2^-24: 2^-12 of the results each way; to 16 bits: 2^-6."""
    g = torch.Generator().manual_seed(E + 1)
    k, q = torch.randn(160, G, E, generator=g).bfloat16(), torch.randn(1, H, E, generator=g)
    v = torch.randn(80, G, E, generator=g).bfloat16()
    _near(*_both(q, k, torch.stack([v, -v], 1).view(160, G, E), False, scale=2.0 ** -12 * E ** -0.5), 2.0 ** -8)

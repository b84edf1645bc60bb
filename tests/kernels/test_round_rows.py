"""When qkv_rope takes two library products for one (ops._round_rows): the rule alone, without a GPU."""
import pytest
import torch

from replisense_rfq_amd import ops


@pytest.fixture
def chip(monkeypatch):
    """256 CUs; tensors count as on the GPU."""
    monkeypatch.setattr(ops, "_gpu", lambda t: True)
    monkeypatch.setattr(ops, "_cus", lambda index: 256)
    ops.reset_plans()
    yield monkeypatch
    ops.reset_plans()


def _pair(M, N, K, dtype=torch.bfloat16):
    return torch.empty((M, K), dtype=dtype, device="meta"), torch.empty((N, K), dtype=dtype, device="meta")


class _Rows:
    """A step of M rows of which nothing but the number may be asked."""
    def __init__(self, M):
        self.shape = (M,)


@pytest.mark.parametrize("M", [0, 1, 16, 64, 1024])
def test_few_rows_ask_nothing_else(M):
    assert ops._round_rows(_Rows(M), None) == 0


# 6,144 columns: rounds of 10 x 24 tiles; 10,240: of 6 x 40; 4,096: of 16 x 16; 8,704: of 7 x 34, too few for 256 CUs
@pytest.mark.parametrize("M,N,K,head", [
    (2560, 6144, 4096, 0), (2561, 6144, 4096, 2560), (2816, 6144, 4096, 2560), (2817, 6144, 4096, 0),
    (2561, 6144, 3072, 2560), (2561, 6144, 3071, 0), (2561, 6144, 2048, 0), (4097, 4096, 2048, 4096),
    (4097, 4096, 2047, 0), (5377, 3072, 2048, 5376), (1793, 8704, 4096, 0), (1025, 14336, 4096, 0), (1537, 10240, 16384, 1536),
    (1537, 10240, 16512, 0), (5121, 6144, 4096, 0), (3072, 10240, 8192, 0), (3073, 10240, 8192, 3072),
    (3993, 10240, 8192, 3072), (3994, 10240, 8192, 0), (3073, 10240, 8191, 0), (3073, 10240, 9217, 0),
    (5530, 10240, 8192, 0), (6145, 10240, 8192, 0),          # 25 x 40 tiles fit four rounds
    (6401, 10240, 8192, 6144), (7681, 10240, 8192, 0), (5121, 6144, 8192, 0), (2561, 6100, 4096, 0), (8193, 2048, 4096, 8192)])
def test_bounds(chip, M, N, K, head):
    assert ops._round_rows(*_pair(M, N, K)) == head


def test_plans_copies_types_and_derivatives_have_the_word(chip):
    x, w = _pair(2561, 6144, 4096)
    assert ops._round_rows(x, w) == 2560
    assert ops._round_rows(*_pair(2561, 6144, 4096, torch.float16)) == 0
    assert ops._round_rows(x.t().contiguous().t(), w) == 0
    assert ops._round_rows(x, w.detach().requires_grad_()) == 0
    ops._SPLIT_PLAN[(6144, 4096)] = (256, [])
    assert ops._round_rows(x, w) == 0
    ops._SPLIT_PLAN.clear()
    chip.setattr(ops, "tiled_only", lambda t: True)
    assert ops._round_rows(x, w) == 0


def test_autocast_has_the_word(chip):
    """Under autocast to another type one product would give rows of that type, which the append refuses."""
    x, w = _pair(2561, 6144, 4096)
    assert ops._round_rows(x, w) == 2560
    chip.setattr(torch, "is_autocast_enabled", lambda device: device == "cuda")      # no GPU, no autocast
    assert ops._round_rows(x, w) == 0

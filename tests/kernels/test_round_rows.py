"""When qkv_rope takes two library products for one (ops._round_rows): the rule alone, without a GPU."""
import pytest

from replisense_rfq_amd import ops


class _Rows:
    """A step of M rows of which nothing but the number may be asked."""
    def __init__(self, M):
        self.shape = (M,)


@pytest.mark.parametrize("M", [0, 1, 16, 64, 1024])
def test_few_rows_ask_nothing_else(M):
    assert ops._round_rows(_Rows(M), None) == 0

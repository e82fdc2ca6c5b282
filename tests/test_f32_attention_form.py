"""Which kernel a 32-bit prompt goes to: by its widths alone, however many waves its rows get."""
import pytest

from transformer_amd import kernels
from ctypes import c_int


def _form(batch, longest, tokens, heads, kv, dk, dv):
    """(widths, waves for 16 rows); widths 0: 128 and 128, 1: 64 and 64, 2: both up to 64, 3: any."""
    return divmod(kernels.library().ta_attention_f32_form(*map(c_int, (batch, longest, tokens, heads, kv, dk, dv))), 8)


@pytest.mark.parametrize("batch,longest,tokens,waves", [(1, 40, 40, 4), (1, 1500, 1500, 2), (2, 1000, 1500, 2), (1, 9000, 9000, 1), (64, 200, 9000, 1)])
def test_narrow_heads_go_to_the_narrow_kernel(batch, longest, tokens, waves):
    for dk, dv, widths in ((128, 128, 0), (64, 64, 1), (16, 16, 2), (48, 64, 2), (64, 32, 2), (80, 16, 3), (64, 128, 3), (128, 64, 3)):
        assert _form(batch, longest, tokens, 8, 4, dk, dv) == (widths, waves), (dk, dv)


def test_many_sequences_of_the_narrowest_heads_get_one_wave():
    assert _form(8, 300, 2400, 8, 8, 16, 16) == (2, 1) and _form(1, 1021, 1021, 8, 8, 16, 16) == (2, 4) and _form(8, 200, 1600, 8, 8, 16, 32) == (2, 2)


def test_rows_past_a_grid_get_one_wave():
    assert _form(1, 70000, 70000, 32, 1, 64, 64) == (1, 1)
    assert _form(1, 5, 5, 6, 4, 64, 64) == (0, 0)          # heads that do not divide

"""The rule that picks the postscan's form: register counters only where they
were measured no slower on uniform, sorted and skewed keys, for calls on user
input and for digit passes."""
import pytest

from test_emu_cpu import emu  # noqa: F401


@pytest.mark.parametrize("log_b,kv,n,starts,digit_pass,reg", [
    # calls without bucket starts: from the size on where no key distribution loses
    (1, 1, (1 << 24) - 1, 0, 0, 0), (1, 1, 1 << 24, 0, 0, 1), (3, 1, 9_500_000, 0, 0, 0),
    (4, 1, 20_000_000, 0, 0, 0), (4, 1, 1 << 25, 0, 0, 1), (2, 0, 13_500_000, 0, 0, 0),
    (3, 0, 50_000_000, 0, 0, 0), (3, 0, 1 << 26, 0, 0, 1), (4, 0, 1 << 27, 0, 0, 0),
    # 32 buckets of pairs: sorted keys lose more than uniform ones gain
    (5, 1, 1 << 26, 0, 0, 0), (5, 1, 1 << 27, 1, 0, 0),
    # calls with starts
    (1, 0, 2_300_000, 1, 0, 1), (3, 0, 9_500_000, 1, 0, 1), (4, 1, 8_500_000, 1, 0, 1),
    (8, 0, (9 << 20) - 1, 1, 0, 1), (8, 0, 9 << 20, 1, 0, 0), (8, 1, (7 << 20) - 1, 1, 0, 1),
    (8, 1, 7 << 20, 1, 0, 0), (9, 1, 3_000_000, 1, 0, 0),
    # digit passes: never key-only, pairs where the loads stream
    (3, 0, 1 << 25, 0, 1, 0), (3, 0, 1 << 27, 0, 1, 0), (2, 0, 1 << 26, 0, 1, 0),
    (4, 1, 1 << 25, 0, 1, 0), (3, 1, 1 << 25, 0, 1, 0), (4, 1, 1 << 26, 0, 1, 1),
    (5, 1, 1 << 27, 0, 1, 0), (8, 1, 3_000_000, 0, 1, 0)])
def test_form(emu, log_b, kv, n, starts, digit_pass, reg):  # noqa: F811
    assert emu.gms_emu_reg_rank(log_b, kv, n, starts, digit_pass) == reg

"""Which models' tokens run as one launch: host arithmetic of the library, no GPU call."""
import pytest

from deepj_amd._native import library


def groups(kind=0, vocab=1000, max_seq=64, d=256, heads=8, layers=2, dff=688, groups=0):
    return library().deepj_hip_token_plan_shape_groups(kind, vocab, max_seq, d, heads, layers, dff, groups)


def test_a_shape_takes_the_groups_asked_for_or_none():
    for g in range(1, 9):
        assert groups(groups=g, dff=1000) == g
    assert groups(groups=9) == 0 and groups(groups=-1) == 0
    assert groups(heads=2, d=64, groups=4) == 0                      # a head for every group
    assert groups(dff=130, groups=4) == 0                            # .. and 64 hidden units
    assert groups(kind=1) == 0 and groups(d=250) == 0 and groups(heads=4, d=64) == 0
    assert groups(d=8192, heads=64) == 0 and groups(dff=1 << 30) == 0


@pytest.mark.parametrize("kind", [0, 2])
def test_the_choice_follows_the_weights_of_a_block(kind):
    assert groups(kind) == 1
    assert groups(kind, vocab=32000, d=2048, heads=16, layers=16, dff=8192) == 8
    assert groups(kind, d=640, heads=5, dff=2000, layers=12, vocab=30000) == 4


@pytest.mark.parametrize("hd", [32, 64, 128])
def test_a_head_s_rows_are_reached_with_32_bits(hd):
    """A key's byte offset in its head's rows is a 32-bit number in the kernel: past 2^32 bytes a new row would land on an early
    key."""
    most = (1 << 32) // (4 * hd)
    assert groups(max_seq=most, d=hd, heads=1, layers=1) == 1
    assert groups(max_seq=most + 1, d=hd, heads=1, layers=1) == 0


def test_heads_and_tags_are_counted_with_32_bits():
    assert groups(vocab=(1 << 28) - 16, groups=8, dff=1000) == 8
    assert groups(vocab=(1 << 28) - 15, groups=8, dff=1000) == 0 and groups(vocab=(1 << 31) - 1) == 0
    assert groups(layers=(1 << 21) - 1, max_seq=1, d=32, heads=1) == 1
    assert groups(layers=1 << 21, max_seq=1, d=32, heads=1) == 0

"""Which kernel a launch takes, at the places where both sides were measured (256 compute units)."""

import pytest

from tests.dispatch import scan_plan, sweep_columns


@pytest.mark.parametrize(
    "N, H, V, longest, chunks, layout, columns",
    [
        (4, 16, 128, 64, 256, "rows", 64),
        (2, 16, 128, 32, 64, "rows", 32),
        (11, 16, 128, 99, 512, "packed", 64),
        (21, 16, 128, 32, 51, "packed", 32),   # one sequence of 2000 tokens, 20 of 64
        (1, 16, 128, 63, 512, "packed", 32),   # one of 4000 tokens in a row of 32768: the rest of the row is nobody's
        (2, 32, 128, 63, 78, "packed", 32),    # 4000 and 1000 tokens
        # left-padded, only one row of them full as far as the host knows: whether its chains fit an XCD side by side
        (6, 16, 128, 64, 6 * 64, "padded", 64),
        (26, 5, 128, 32, 26 * 32, "padded", 64),
        (32, 4, 128, 32, 32 * 32, "padded", 32),
        (8, 16, 64, 32, 8 * 32, "padded", 64),
        (16, 8, 64, 32, 16 * 32, "padded", 32),
        (43, 3, 256, 32, 43 * 32, "padded", 64),
        (48, 2, 256, 32, 48 * 32, "padded", 32),
        (7, 14, 128, 4, 7 * 64, "padded", 64),  # rows of 4096 tokens, none of which uses more than 256
        (2, 16, 128, 4, 2 * 64, "padded", 32),
        (4, 16, 96, 64, 256, "rows", 32),      # whole slices of 64 columns only
    ],
)
def test_width_of_the_sweeps(N, H, V, longest, chunks, layout, columns):
    assert sweep_columns(N, H, V, longest, chunks, layout == "packed", layout == "padded") == columns


@pytest.mark.parametrize(
    "K, rows, H, T, V, packed, direct",
    [
        (128, 20, 16, 64, 128, False, False), (128, 20, 16, 65, 128, False, True), (128, 20, 16, 255, 128, False, True), (128, 20, 16, 256, 128, False, False),
        (128, 12, 32, 200, 256, False, True), (128, 48, 16, 200, 128, False, True), (128, 49, 16, 200, 128, False, False), (128, 100, 16, 112, 128, False, True), (128, 100, 16, 113, 128, False, False),
        (128, 100, 16, 128, 128, False, False), (64, 40, 16, 65, 128, False, True), (64, 40, 16, 128, 128, False, False), (128, 60, 16, 200, 128, True, False),
        (128, 8, 16, 65, 128, False, False), (256, 40, 16, 65, 512, False, False),  # two slices, half slices
    ],
)  # fmt: skip
def test_who_stores_the_output_of_four_slices(K, rows, H, T, V, packed, direct):
    assert scan_plan(K, rows * H, T, V, packed).direct == direct


def _cases_of(test):
    return next(m for m in test.pytestmark if m.name == "parametrize").args[1]


def test_the_cases_of_the_scans_take_the_scans_they_are_of():
    """At 256 compute units: a rule that is moved moves no test to another kernel unnoticed."""
    from tests import test_chunk_gpu as chunk

    for T, V, _, H in _cases_of(chunk.test_split_keys_at_the_edges_of_chunks):
        assert scan_plan(256, 2 * H, T, V).split_keys, (T, V, H)
    for T, V, _, H in _cases_of(chunk.test_half_slices_of_256_keys_at_the_edges_of_chunks):
        assert not scan_plan(256, 4 * H, T, V).split_keys, (T, V, H)
    for T in _cases_of(chunk.test_four_slices_at_the_edges_of_chunks):
        plan = scan_plan(64, 9 * 16, T, 128)
        assert plan.nw == 4 and plan.direct == (T == 65), T
    for T in _cases_of(chunk.test_four_slices_of_two_chunks_through_the_loaders):
        plan = scan_plan(64, 9 * 16, T, 128)
        assert plan.nw == 4 and not plan.direct, T


def test_the_cases_of_the_sweeps_have_the_width_they_are_of():
    from tests.test_sweeps_gpu import CASES

    wide = 0
    for layout, lens, K, V, _, H in CASES:
        if K == 128:
            rows, longest = len(lens), -(-max(lens) // 64)
            chunks = sum(lens) // 64 if layout == "packed" else rows * longest
            columns = sweep_columns(rows, H, V, longest, chunks, layout == "packed", layout == "padded")
            assert columns == (64 if H >= 8 else 32), (layout, lens, H)
            wide += columns == 64
    assert wide == 10

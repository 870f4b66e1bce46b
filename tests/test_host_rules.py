"""The rules that choose a dispatch's kernels, as the runtime calls them
(peregrine_amd/csrc/host_rules.h), at both sides of every bound."""
import pytest


@pytest.mark.parametrize("w4,D,I,rows", [
    (1, 96, 64, 48), (1, 2048, 1280, 48),          # one expert's weights: up to 4e6 bytes
    (1, 2048, 1344, 40), (1, 5120, 1536, 40),      # up to 12e6
    (1, 4096, 2048, 32), (1, 7168, 2048, 32),
    (0, 96, 64, 24), (0, 2048, 640, 24),           # int8: up to 4e6
    (0, 2048, 704, 16), (0, 5120, 1600, 16),       # up to 25e6
    (0, 5120, 1664, 8), (0, 6144, 2048, 8),
])
def test_gemv_pays_bounds(host_rules, w4, D, I, rows):
    assert host_rules.gemv_pays_c(D, I, w4, w4, 1) and host_rules.gemv_pays_c(D, I, w4, w4, rows)
    assert not host_rules.gemv_pays_c(D, I, w4, w4, rows + 1) and not host_rules.gemv_pays_c(D, I, w4, w4, 14216)


def test_gemv_pays_mixed_formats(host_rules):
    """One projection in int8: the int8 bounds."""
    for a, b in ((1, 0), (0, 1)):
        assert host_rules.gemv_pays_c(96, 64, a, b, 24) and not host_rules.gemv_pays_c(96, 64, a, b, 25)


@pytest.mark.parametrize("w4,D,I,n,R", [
    (1, 5120, 1536, 160, 24 * 160),     # K of 2017 on: 24 rows per expert
    (1, 2017, 8192, 8, 24 * 8),
    (1, 2016, 8192, 8, 64 * 8),         # shorter K: 64
    (0, 5120, 1536, 160, 24 * 160),
    (0, 1536, 2048, 128, 24 * 128),     # int8, short K, many items: 24
    (0, 96, 1024, 40, 64 * 40),         # int8, short K, under 512 items: 64
])
def test_row_groups_rows_per_expert(host_rules, w4, D, I, n, R):
    assert host_rules.row_groups_c(D, I, w4, 1, 1, R, n, 0)
    assert not host_rules.row_groups_c(D, I, w4, 1, 1, R - 1, n, 0)


@pytest.mark.parametrize("w4,items", [(1, 256), (0, 128)])
def test_row_groups_items_fill_the_chip(host_rules, w4, items):
    """One expert of R rows: (R / 128 + 1) leading tiles x 4 slabs."""
    R = (items // 4 - 1) * 128
    assert host_rules.row_groups_c(4096, 512, w4, 1, 1, R, 1, 0)
    assert not host_rules.row_groups_c(4096, 512, w4, 1, 1, R - 1, 1, 0)


def test_row_groups_needs_per_row_weights_and_activations(host_rules):
    args = (14216, 160)
    assert host_rules.row_groups_c(5120, 1536, 1, 1, 1, *args, 0)
    assert host_rules.row_groups_c(5120, 1536, 1, 1, 0, *args, 0) and host_rules.row_groups_c(5120, 1536, 1, 0, 1, *args, 0)
    assert not host_rules.row_groups_c(5120, 1536, 1, 1, 1, *args, 32)
    assert not host_rules.row_groups_c(5120, 1536, 1, 0, 0, *args, 0)

"""The decode launch's own partitions: what :func:`decode_split` and
:func:`decode_balanced` may return over the sizes a launch takes."""

from __future__ import annotations

import itertools

import pytest

from flashattntile_amd.autotune import decode_balanced, decode_split


@pytest.mark.parametrize("mfma", [False, True])
@pytest.mark.parametrize("token_bytes", [64, 256, 512, 2048])
def test_decode_split_stays_in_range(token_bytes, mfma):
    for items, longest, ragged in itertools.product((1, 4, 8, 31, 127, 128, 200, 255, 256, 257, 300, 1000, 20000),
                                                    (1, 63, 128, 256, 257, 1024, 5000, 40000, 10 ** 6), (1.0, 1.3, 30.0)):
        split, waves = decode_split(items, longest, longest / ragged, token_bytes, mfma)
        assert 1 <= split <= 64 and waves in (None, 4, 8)
        assert split == 1 or longest / split >= 64  # no partitions shorter than a kernel's blocks
        assert waves != 8 or items * split <= 256
        if longest <= 256:
            assert split == 1


def test_decode_split_fills_the_cus():
    assert decode_split(8, 4096, 4096, 512)[0] * 8 >= 128
    assert decode_split(8, 100000, 100000, 512)[0] * 8 == 256
    assert decode_split(1000, 2000, 2000, 512)[0] == 1
    assert 300 * decode_split(300, 2000, 2000, 512)[0] > 512  # not two rounds, the second nearly empty


def test_decode_balanced_takes_large_ragged_batches():
    assert decode_balanced(16000, 8000, 500_000_000, 4)
    assert not decode_balanced(16000, 15000, 500_000_000, 4)  # uniform
    assert not decode_balanced(16000, 8000, 50_000_000, 4)  # short
    assert not decode_balanced(16000, 8000, 500_000_000, 17)  # more rows than its merge takes


@pytest.mark.parametrize("rows", [1, 4, 16, 32])
@pytest.mark.parametrize("mfma", [False, True])
def test_decode_split_of_very_ragged_batches_stays_in_range(mfma, rows):
    """Around the lines of its rule: four and twelve times the mean, and the
    bytes from which it applies."""
    for items, longest, ratio, waves in itertools.product((1, 16, 64, 255, 256, 257, 800, 1024, 4096, 100000),
                                                          (63, 257, 800, 1999, 2001, 16000, 65536, 10 ** 6),
                                                          (3.9, 4.0, 11.9, 12.0, 60.0, 1000.0), (None, 4, 8)):
        split, chosen = decode_split(items, longest, longest / ratio, 512, mfma, rows=rows, waves=waves)
        assert 1 <= split <= 64 and chosen in (None, 4, 8)
        assert split == 1 or longest / split >= 64
        if ratio < 4.0:
            assert split == decode_split(items, longest, longest / ratio, 512, mfma)[0]
        if longest <= 256:
            assert split == 1


def test_decode_split_of_very_ragged_batches():
    # many long sequences share their CUs: partitions of less than a CU's share
    assert decode_split(1024, 16000, 16000 / 6, 512, True, rows=8)[0] >= 3
    assert decode_split(1024, 16000, 16000 / 6, 512, False)[0] > decode_split(1024, 16000, 16000 / 2, 512, False)[0]
    # one long sequence among short ones, 32 rows per workgroup
    assert decode_split(64, 100000, 1759, 512, True, rows=32)[0] >= 16
    # rows of many sequences: the partials of a partition are large
    assert decode_split(1024, 30000, 1900, 512, True, rows=32)[0] <= 4
    # whole sequences already fill the CUs many times over
    assert decode_split(4096, 4096, 800, 512, True, rows=8)[0] == 1


def test_decode_balanced_leaves_many_short_items_to_partitions():
    items, mean = 2048, 1310
    assert not decode_balanced(8000, mean, items * mean * 512, 4, items, 512, False)
    assert not decode_balanced(8000, mean, items * mean * 256, 2, items, 256, True)
    assert decode_balanced(8000, mean, 800 * mean * 256, 2, 800, 256, True)  # fewer, on the MFMA kernel
    assert decode_balanced(8000, 8000 / 2, items * mean * 512, 4, items, 512, False)  # lengths within a factor
    assert decode_balanced(30000, 1900, 1024 * 1900 * 512, 4, 1024, 512, False)  # a few long ones
    assert not decode_balanced(16000, 3000, 512 * 3000 * 256, 4, 512, 256, False)  # head_dim 64 on the VALU kernel
    assert decode_balanced(16000, 3000, 512 * 3000 * 512, 4, 512, 512, False)

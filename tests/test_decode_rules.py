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

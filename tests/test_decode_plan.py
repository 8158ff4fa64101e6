"""The decode attention's split plan (kernels.decode_plan) against decode_splits: it differs only where
halved splits leave less of the last round of workgroups empty; what it returns always covers the block
table with at most 32 splits of the planned context, and does not depend on the contexts."""

from __future__ import annotations

import pytest

from miniserve_amd import kernels


@pytest.mark.parametrize("num_seqs,planned,want", [
    (3, 32768, 1024),  # a round and a half of 2048-key splits
    (6, 16000, 1024),
    (4, 32768, 2048),  # whole rounds
    (31, 4096, 2048),
    (16, 4000, 2048),  # one round
    (2, 40960, 2048),  # 1024-key splits would be more than 32
    (3, 32784, 2048),
    (32, 32768, 4096),  # 256 pairs: one split up to 4096 keys
    (1, 1100, 64),
])
def test_decode_plan_rounds(num_seqs, planned, want):
    width = -(-planned // 16)
    assert kernels.decode_plan(num_seqs, 8, width, 4, planned) == (want, -(-width * 16 // want))
    assert kernels.decode_plan(num_seqs, 8, width, 4) == kernels.decode_plan(num_seqs, 8, width, 4, 16 * width)


def test_decode_plan_covers_and_only_halves():
    for pairs in (1, 2, 4, 8):
        for num_seqs in (1, 2, 3, 5, 8, 13, 24, 31, 40, 100):
            for planned in (16, 100, 1000, 2048, 5000, 9999, 16384, 20000, 32768, 33000, 50000):
                width = -(-planned // 16)
                base = kernels.decode_splits(num_seqs, pairs, width, 4, planned)
                part, parts = kernels.decode_plan(num_seqs, pairs, width, 4, planned)
                assert part * parts >= width * 16
                assert (part, parts) == base or (part * 2 == base[0] == 2048 and parts <= 32)

"""The fast hard forward's block count on the CPU: 1024-thread blocks run one
per CU, so a launch has at most 256 of them or whole rounds of 256, and no
histogram copy counts more voxels than its 11-bit field."""

from __future__ import annotations

import itertools

import pytest

from test_geometry import _geometry, geo  # noqa: F401  (the harness fixture)


@pytest.mark.parametrize("c,vec", [(2, 4), (3, 4), (4, 2)])
def test_whole_rounds(geo, c, vec) -> None:  # noqa: F811
    for b, k in itertools.product([1, 2, 3, 5], [2, 20, 50]):
        for n in [1000, 128 ** 3 // 3 * 2 - 5, 128 ** 3 - 7, 128 ** 3, 128 ** 3 + 1, 3_932_160, 7_864_320, 7_864_321,
                  191 * 223 * 207, 15_728_641, 33_030_144, 33_030_145, 70_000_001]:
            nt, v, lds, _, nblk = _geometry(geo, b, c, n, k, 0, 1, 1024)
            assert (nt, v) == (1024, vec)
            total = b * n
            # 64 copies count 2047 voxels each: 63 (31) steps of 1024 lanes a block
            rounds = -(-total // (256 * 1024 * vec * (2047 // (16 * vec))))
            assert nblk <= 256 * rounds, (b, n, k, nblk, rounds)
            assert nblk * 1024 * vec * (2047 // (16 * vec)) >= total
            assert lds <= 160 * 1024

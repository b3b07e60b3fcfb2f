"""GPU: layout conversion is a lossless byte permutation; the device generator equals the CPU one."""
import numpy as np
import pytest

from helpers import random_blocks, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,k", [(32, 128), (1, 128), (33, 256), (4096, 4096), (100, 14336)])
def test_tile_untile_roundtrip(q8, rows, k):
    rng = np.random.default_rng(rows + k)
    w = random_blocks(rng, rows, k)
    t = q8.tile(to_dev(w), rows, k)
    assert t.numel() == ((rows + 31) // 32) * (k // 128) * 4352
    assert np.array_equal(to_host(q8.untile(t, rows, k)), w)


def test_tiled_layout_definition(q8):
    # spot-check the documented address formula against a host-side permutation
    rows, k = 64, 256
    rng = np.random.default_rng(1)
    w = random_blocks(rng, rows, k).reshape(rows, k // 32, 34)
    t = to_host(q8.tile(to_dev(w.reshape(-1)), rows, k))
    groups = k // 128
    for row, b, q in [(0, 0, 0), (5, 3, 17), (37, 6, 31), (63, 7, 15), (32, 4, 16)]:
        macro = ((row // 32) * groups + b // 4) * 4352
        lane = row % 32 + 32 * (q // 16)
        assert t[macro + (b % 4) * 1024 + 16 * lane + q % 16] == w[row, b, 2 + q]
        assert t[macro + 4096 + 8 * (row % 32) + 2 * (b % 4)] == w[row, b, 0]
        assert t[macro + 4096 + 8 * (row % 32) + 2 * (b % 4) + 1] == w[row, b, 1]


def test_device_generator_matches_cpu(q8, oracle):
    for seed, n, k, first in [(0, 64, 4096, 0), (12345, 3, 96, 77), (2**63 + 5, 16, 128, 10**9)]:
        got = to_host(q8.fill_weight_blocks(seed, n, k, first_block=first))
        assert np.array_equal(got, oracle.fill_weights(seed, n, k, first_block=first))
        x = to_host(q8.fill_activations(seed, 4097))
        assert np.array_equal(x, oracle.fill_activations(seed, 4097))


@pytest.mark.parametrize("rows", [1, 31, 32, 65])
@pytest.mark.parametrize("groups", [1, 3, 4, 5, 9])  # a wave takes a group, a workgroup four: full, short and single
def test_tile_is_the_documented_permutation(q8, rows, groups):
    rng = np.random.default_rng(rows * 16 + groups)
    w = random_blocks(rng, rows, groups * 128)
    strips = (rows + 31) // 32
    padded = np.zeros((strips * 32, groups, 4, 34), dtype=np.uint8)  # rows past the last are zero blocks
    padded[:rows] = w.reshape(rows, groups, 4, 34)
    by_strip = padded.reshape(strips, 32, groups, 4, 34).transpose(0, 2, 3, 1, 4)  # strip, group, tile, row, bytes
    quants = by_strip[..., 2:].reshape(strips, groups, 4, 32, 2, 16).transpose(0, 1, 2, 4, 3, 5).reshape(strips, groups, 4096)
    scales = by_strip[..., :2].transpose(0, 1, 3, 2, 4).reshape(strips, groups, 256)
    want = np.concatenate([quants, scales], axis=2).reshape(-1)
    assert np.array_equal(to_host(q8.tile(to_dev(w), rows, groups * 128)), want)

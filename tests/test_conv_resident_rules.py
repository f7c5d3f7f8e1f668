"""Which convolutions run with their filter resident in LDS, and how they are divided (csrc/conv_resident_rules.hpp), compiled without
device code."""
import itertools
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    binary = str(tmp_path_factory.mktemp("host_checks") / "conv_resident_rules")
    cmd = ["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17",
           os.path.join(ROOT, "tests", "host_checks", "conv_resident_rules.cpp"), "-o", binary]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return lambda *q: [int(v) for v in subprocess.run([binary, *map(str, q)], capture_output=True, text=True, check=True).stdout.split()]


def test_plans_cover_the_product_and_fit_lds(ask):
    for positions, columns, channels, kh, kw in itertools.product((30000, 32768, 32801, 529000), (1, 32, 33, 65, 130, 400), (8, 9, 64, 100, 512), (1, 3, 7), (3, 5)):
        per_row, units, pairs, chunk, tn, blocks_n, tiles, wvk, per_block, lds = ask("plan", positions, columns, channels, kh, kw)
        assert 8 * per_row >= channels > 8 * (per_row - 1) and units == kh * per_row and 2 * pairs >= units > 2 * (pairs - 1)
        assert 1 <= chunk <= pairs and tn in (1, 2) and 32 * tn * blocks_n >= columns > 32 * tn * blocks_n - 64
        assert 32 * tiles >= positions > 32 * (tiles - 1)
        # table, runs, and a step more of the filter than is multiplied; two wavefronts on a tile hand their sums over where it lay
        assert (pairs + 4) * 16 + 8 * 48 * 96 + max((chunk * kw + 1) * tn * 3072, 4 * (tn * 1024 + 64) * 4 * (wvk - 1)) <= lds <= 160 * 1024 - 64
        assert (wvk == 2) == ((tiles + 3) // 4 * blocks_n <= 256 and pairs * kw * tn >= 18)
        if wvk == 2:  # one tile for every pair of wavefronts, one round of workgroups
            assert 4 * per_block >= tiles > 4 * (per_block - 1) and per_block * blocks_n <= 256
        else:
            assert 8 * (per_block - 1) < tiles and (per_block == 1 or per_block * blocks_n <= 256)


def test_elements_of_a_tile(ask):
    """32 positions from any place of rows of any length: the rows they touch, with kw - 1 more elements each, fit 48 where the kernel is taken."""
    for row, kw in itertools.product(range(1, 70), (3, 5)):
        touched = max((start + 31) // row + 1 for start in range(row))
        taken = ask("takes", 30000, 3, row, 8, 8, 3, kw, 1)
        assert taken == [int(32 + (kw - 1) * touched <= 48)] * 2, (row, kw)


def test_filters_beyond_lds(ask):
    """Filters whose table of units nearly fills LDS by itself are declined in both directions, at any number of positions; the largest
    that leave room for one pair of units have a plan."""
    for columns, channels, kh, kw in ((64, 4096, 22, 5), (33, 4096, 23, 5), (65, 4096, 31, 3), (64, 4096, 25, 5), (32, 2904, 31, 5), (64, 4096, 31, 5)):
        for batch in (1, 16):
            for same in (0, 1):
                assert ask("takes", batch, 45, 45, channels, columns, kh, kw, same) == [0, 0]
                assert ask("takes", batch, 45, 45, columns, channels, kh, kw, same)[1] == 0
    for columns, kw in itertools.product((32, 64), (3, 5)):
        step, chunks = (columns // 32) * 3072, {}
        for pairs in range(5000, 8200):
            room = 160 * 1024 - 64 - (pairs + 4) * 16 - 8 * 48 * 96
            if room // step - 1 >= kw:
                chunks["last"] = pairs
            else:
                chunks.setdefault("none", pairs)
        for pairs, planned in ((chunks["last"], True), (chunks["none"], False)):
            plan = ask("plan", 529000, columns, 16 * pairs, 1, kw)
            assert (plan[3] >= 1) == planned and (not planned or plan[2] == pairs and plan[9] <= 160 * 1024 - 64)


def test_which_convolutions_of_one_round(ask):
    """Up to 128 positions a CU short reductions stay with the tiled kernels, and input gradients from whole 32s of filters with the ring."""
    for batch, beyond in ((118, 0), (128, 0), (129, 1)):  # 30208, 32768 and 33024 positions
        for want, *shape in (([beyond, beyond], 8, 16, 1, 5), ([beyond, beyond], 16, 16, 2, 3), ([1, 1], 16, 24, 3, 3), ([1, 1], 24, 40, 3, 3), ([1, 1], 8, 8, 5, 5),
                             ([1, beyond], 64, 64, 3, 3), ([1, beyond], 64, 64, 1, 3), ([1, 0], 16, 32, 3, 3), ([1, 1], 64, 40, 3, 3)):
            assert ask("takes", batch, 16, 16, *shape, 1) == want, (batch, shape)
    assert ask("takes", 117, 16, 16, 24, 40, 3, 3, 1) == [0, 0]


def test_which_convolutions(ask):
    for want, *shape in (([1, 0], 100, 25, 25, 32, 64, 3, 3, 0),     # an input gradient onto 32 channels of 62500 positions stays with the ring
                         ([1, 1], 1000, 13, 13, 32, 64, 3, 3, 0),
                         ([0, 0], 100, 13, 13, 32, 64, 3, 3, 0),     # too few positions
                         ([1, 0], 125, 16, 16, 48, 80, 3, 3, 1),     # 80 -> 48 channels: three chunks
                         ([0, 0], 1000, 13, 13, 4, 7, 3, 3, 0),      # less than a unit of channels
                         ([0, 0], 1000, 13, 13, 32, 64, 3, 4, 0),
                         ([0, 0], 1000, 13, 13, 32, 64, 32, 3, 1),
                         ([0, 1], 60, 24, 24, 7, 50, 3, 3, 1),
                         ([0, 0], 30000, 60, 60, 8, 8, 3, 3, 1)):    # a tensor beyond 2 GiB
        assert ask("takes", *shape) == want, shape


def test_every_variant_has_a_product_in_the_parity_tests(ask):
    """Tiles of a workgroup x width x wavefronts a tile in both directions, and chunks with one round of tiles and with a second, ragged one; and
    what those tests say of which products run here is what the rule says."""
    source = open(os.path.join(ROOT, "tests", "test_gpu_parity.py")).read()
    at = source.index("RESIDENT_CONVOLUTIONS = [")
    shapes = eval(source[at + 24:source.index("]\n", at) + 1])
    variants, rounds = set(), set()
    for batch, height, width, channels, filters, (kh, kw), pad, taken in shapes:
        if isinstance(pad, str):
            assert ask("takes", batch, height, width, channels, filters, kh, kw, int(pad == "same")) == list(taken)
            oh, ow = (height, width) if pad == "same" else (height - kh + 1, width - kw + 1)
        else:
            oh, ow = height + pad[0] + pad[1] - kh + 1, width + pad[2] + pad[3] - kw + 1
        for direction, positions, columns, k in ((0, batch * oh * ow, filters, channels), (1, batch * height * width, channels, filters)):
            if taken[direction]:
                _, _, pairs, chunk, tn, blocks_n, tiles, wvk, per_block, _ = ask("plan", positions, columns, k, kh, kw)
                variants.add((direction, tn, kw, wvk))
                if chunk < pairs:
                    rounds.add((tn, wvk, tiles * wvk > 8 * per_block))
    assert variants == set(itertools.product((0, 1), (1, 2), (3, 5), (1, 2)))
    assert rounds >= {(1, 1, True), (2, 1, True), (2, 2, False)}

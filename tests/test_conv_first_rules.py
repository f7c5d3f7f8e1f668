"""Which first layers have kernels of their own and how these divide them (csrc/conv_first_rules.hpp), compiled without device code."""
import itertools
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    binary = str(tmp_path_factory.mktemp("host_checks") / "conv_first_rules")
    cmd = ["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17",
           os.path.join(ROOT, "tests", "host_checks", "conv_first_rules.cpp"), "-o", binary]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return lambda *q: [int(v) for v in subprocess.run([binary, *map(str, q)], capture_output=True, text=True, check=True).stdout.split()]


def test_every_position_lies_in_one_segment_of_one_wavefront(ask):
    for rows, wo, room in itertools.product((1, 3, 8, 100, 2600, 4096, 4097, 676000), (1, 15, 16, 17, 33, 398, 4088), (32, 100, 1024)):
        segments, length, per_wave, parts = ask("cut", rows, wo, room)
        assert length % 16 == 0 and (segments - 1) * length < wo <= segments * length
        assert 4 * parts * per_wave >= rows * segments > 4 * (parts - 1) * per_wave
        assert parts <= room


@pytest.mark.parametrize("rows,wo", [(8, 4088), (64, 2040), (100, 504), (64, 1016), (128, 504), (2, 2048)])
def test_few_long_rows_are_spread_over_the_chip(ask, rows, wo):
    """A wavefront walks at most twice the positions that an even division over 4096 wavefronts would leave it, or one trip of 16."""
    segments, length, per_wave, _ = ask("cut", rows, wo, 1024)
    assert min(length, wo) * per_wave <= max(16, 2 * rows * wo / 4096 + 16)


def test_many_rows_stay_whole(ask):
    assert ask("cut", 2600, 26, 1024) == [1, 32, 1, 650]
    assert ask("cut", 26000, 26, 1024)[:3] == [1, 32, 7]


def test_many_taps_onto_many_filters_stay_with_the_tiled_kernels(ask):
    for kh, kw, cin, cout, want in ((4, 4, 4, 192, 1), (4, 4, 4, 196, 0), (4, 4, 4, 256, 0), (4, 4, 3, 512, 0), (3, 3, 4, 344, 0), (5, 5, 2, 256, 0), (8, 8, 1, 512, 0),
                                    (4, 4, 2, 512, 0), (3, 3, 3, 512, 1), (3, 3, 1, 1400, 1), (7, 4, 1, 700, 1), (3, 3, 3, 50, 0), (9, 8, 1, 32, 0), (3, 3, 5, 32, 0)):
        assert ask("forward", kh, kw, cin, cout) == [want], (kh, kw, cin, cout)


def test_two_tiles_of_filters_where_a_wavefront_can_gather_again(ask):
    for taps, cout, want in ((9, 64, 2), (18, 128, 2), (4, 96, 2), (20, 256, 2), (9, 16, 1), (9, 32, 2), (9, 48, 3), (9, 56, 4), (9, 80, 4), (27, 64, 4), (32, 128, 4)):
        assert ask("tiles", taps, cout, 0) == [want], (taps, cout)
    assert ask("tiles", 9, 64, 1) == [4]

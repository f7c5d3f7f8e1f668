"""Host-side rules of the split products (csrc/split_launch.hpp, csrc/common.hpp), compiled without device code: what the
kernels are given to read, and which tile a product takes."""
import itertools
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    binary = str(tmp_path_factory.mktemp("host_checks") / "split_rules")
    cmd = ["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17",
           os.path.join(ROOT, "tests", "host_checks", "split_rules.cpp"), "-o", binary]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return lambda *q: [int(v) for v in subprocess.run([binary, *map(str, q)], capture_output=True, text=True, check=True).stdout.split()]


def test_split_convolutions_hold_four_values_of_every_image_they_read(ask):
    """The masked loaders clamp a vector of four to [0, total - 4]: a tensor of one to three values would be read in front of
    its start.  One-row batches and 1 x 1 images reach such sizes; one value more and the kernels may take them."""
    seen = {False: 0, True: 0}
    for n, side, cin, cout, kw in itertools.product((1, 2, 3, 4), (1, 2), (1, 2, 3, 4), (1, 2, 3, 4, 5), (1, 2, 4)):
        pad = (kw - 1) // 2
        forward, input_gradient, filter_gradient = ask("conv", n, side, side, cin, side, side, cout, kw, kw, 1, 1, pad, pad)
        x, dy, w = n * side * side * cin, n * side * side * cout, kw * kw * cin * cout
        assert forward == (x >= 4 and w >= 4 and cout >= 4)
        assert input_gradient == (dy >= 4 and w >= 4 and kw * cout >= 4)
        assert filter_gradient == (x >= 4 and dy >= 4 and cout >= 4 and kw * cin >= 4)
        seen[bool(forward)] += 1
    assert min(seen.values()) > 100


def test_split_convolutions_stay_inside_32_bit_offsets(ask):
    assert ask("conv", 1023, 32, 32, 128, 32, 32, 128, 3, 3, 1, 1, 1, 1) == [1, 1, 1]
    # (n + 1) images of 2^21 bytes reach 2^31
    assert ask("conv", 4095, 32, 32, 128, 32, 32, 128, 3, 3, 1, 1, 1, 1) == [0, 0, 0]


def test_a_sum_that_the_optimizer_cannot_take_is_priced_as_a_launch(ask):
    """The choice of tile and splits charges 1 us for partial sums that the optimizer's launch adds and 4.5 for a launch of
    their own: only sums that launch takes are the cheap kind.  The 3 x 3 x 3 x 48 filter of a colour image's first layer has
    1296 values and is not, whatever its caller asked for."""
    assert [ask("defers", m, n, 1)[0] for m, n in ((27, 48), (32, 128), (63, 65), (33, 125), (64, 65), (432, 80))] == [0, 1, 0, 0, 1, 1]
    assert ask("defers", 432, 80, 0) == [0] and ask("defers", 1 << 15, 1 << 15, 1) == [0]
    cheap, dear = ask("choose", 27, 48, 6000, 3, 1), ask("choose", 27, 48, 6000, 3, 0)
    assert cheap[3] >= dear[3]


def test_many_positions_with_few_columns_stay_off_the_split_kernels(ask):
    for m, n, k, c, want in ((378450, 16, 72, 8, 1), (40000, 32, 216, 24, 1), (39999, 16, 72, 8, 0), (378450, 33, 72, 8, 0), (378450, 16, 90, 10, 0),
                             (378450, 8, 288, 32, 0)):
        assert ask("float32", m, n, k, c) == [want]


def test_the_split_count_is_one_the_stages_reach(ask):
    """Partial results are written by ceil(stages / per workgroup) splits and read by as many: the chosen count is that one,
    and a long reduction onto one or two tiles fills the chip whatever its number of stages is."""
    for m, n, k in ((72, 48, 31232), (72, 8, 32076), (432, 8, 8232), (288, 8, 118800), (30, 30, 65537), (700, 770, 1003), (5, 2000, 333)):
        for deferred in (0, 1):
            bm, bn, bk, splits = ask("choose", m, n, k, 3, deferred)
            stages = -(-k // bk)
            assert -(-stages // -(-stages // splits)) == splits
            if k > 8000:
                assert splits * -(-m // bm) * -(-n // bn) >= 200


def test_every_tile_has_a_product_in_the_parity_tests(ask):
    source = open(os.path.join(ROOT, "tests", "test_gpu_parity.py")).read()
    for name, planes, count in (("TILE_SHAPES", 3, 6), ("TILE_SHAPES_BF16", 1, 5)):
        at = source.index(f"\n{name} = ") + len(name) + 4
        shapes = eval(source[at:source.index("}", at) + 1])
        assert len(shapes) == count
        for tile, (rows, hidden, features) in shapes.items():
            assert tuple(ask("choose", rows, hidden, features, planes, 0)[:3]) == tile


def test_every_tile_of_one_plane_is_some_products(ask):
    """Products of the sizes classifiers have reach every tile that is built for one plane, and no other."""
    seen = set()
    for m, n, k in itertools.product((16, 100, 700, 2001, 8192), (17, 330, 1500, 4097), (33, 600, 1501, 4099)):
        for deferred in (0, 1):
            seen.add(tuple(ask("choose", m, n, k, 1, deferred)[:3]))
    assert seen == {(128, 128, 32), (64, 64, 32), (64, 64, 64), (64, 32, 64), (32, 64, 64)}

"""Which filter gradients run on split products straight from the tensors, and how they are divided (csrc/conv_wgrad_split_rules.hpp),
compiled without device code."""
import itertools
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    binary = str(tmp_path_factory.mktemp("host_checks") / "conv_wgrad_split_rules")
    cmd = ["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17",
           os.path.join(ROOT, "tests", "host_checks", "conv_wgrad_split_rules.cpp"), "-o", binary]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return lambda *q: [int(v) for v in subprocess.run([binary, *map(str, q)], capture_output=True, text=True, check=True).stdout.split()]


def _narrow(positions, cin, cout, kh, kw):
    """Tiles of 32 per filter row against tiles of 64 over all rows, each of whole vectors of four."""
    packed = kh * 4 * -(-kw * cin // 4)
    ratio = kh * 32 * -(-kw * cin // 32) / (32 if packed <= 32 else 64 * -(-packed // 64))
    if ratio < 1.5 or kh * kw * cin * cout <= 512:
        return False
    return ratio >= 2.25 or positions >= 32768 and not (cout <= 64 and kh <= 5 and 3 * ratio <= 5)


def test_plans_cover_the_product_and_fit_the_workspace(ask):
    for n, cin, cout, kernel, same in itertools.product((30, 311), (8, 33, 96, 512), (1, 33, 64, 300), ((1, 1), (3, 3), (15, 15)), (0, 1)):
        shape = (n, 16, 17, cin, cout, *kernel, 1, same)
        size, length = kernel[0] * kernel[1] * cin * cout, kernel[1] * cin
        for room in (-1, size, 3 * size):
            taken, tm, tn, groups_m, groups_n, chunks, parts, padded, workspace, reserve = ask(*shape, room)
            assert (tm, tn) in ((1, 1), (1, 2), (1, 3), (2, 1), (2, 2), (3, 1), (3, 2))
            assert 32 * tm * groups_m >= length > 32 * tm * (groups_m - 1) and 32 * tn * groups_n >= cout > 32 * tn * (groups_n - 1)
            assert padded == int(same and kernel != (1, 1))
            positions = n * (16 * 17 if same else (17 - kernel[0]) * (18 - kernel[1]))
            narrow = _narrow(positions, cin, cout, *kernel)
            groups = kernel[0] * groups_m * groups_n
            if room < 0:
                places = -(-groups * parts // 256) * 256
                idle = places - groups * parts
                short = cout > 64 and (20 * idle > places if places > 256 else 5 * idle > places and positions * kernel[0] * length * cout >= 2e10)
            assert 16 * chunks >= positions > 16 * (chunks - 1) and 1 <= parts <= chunks and taken == int(positions >= 4096 and not narrow and not short)
            assert reserve == taken * workspace  # set aside only where it runs
            assert parts * size <= (workspace if room < 0 else room) and (parts == 1 or groups * parts <= 256)
        assert ask(*shape, size - 1)[6] == 0  # no room for one partial result: left to the general path


def test_narrow_runs(ask):
    """Filter rows of a few values leave their tiles of 32 empty, but for results of at most 512 values: how far, at 22500 and 62500 positions."""
    for few, many, cin, cout, kh, kw in ((0, 0, 8, 32, 5, 1), (0, 0, 12, 64, 5, 1), (0, 0, 8, 16, 9, 1), (0, 0, 8, 64, 3, 1), (0, 0, 8, 40, 4, 1),
                                         (1, 1, 8, 8, 5, 1), (1, 1, 8, 8, 7, 1), (1, 1, 10, 16, 3, 1),  # 320, 448 and 480 values
                                         (1, 0, 12, 40, 7, 3), (1, 0, 10, 16, 6, 2), (1, 0, 9, 64, 4, 1), (1, 0, 8, 64, 2, 1), (1, 0, 11, 65, 3, 3), (1, 0, 17, 100, 5, 2),
                                         (1, 1, 11, 64, 3, 3), (1, 1, 12, 16, 3, 1), (1, 1, 17, 64, 5, 2),
                                         (1, 1, 14, 100, 3, 3), (1, 1, 21, 64, 3, 1), (1, 1, 21, 300, 6, 1),  # one vector more than whole tiles of 64
                                         (1, 1, 8, 64, 1, 1), (1, 1, 16, 16, 5, 1), (1, 1, 14, 16, 7, 3), (1, 1, 8, 16, 3, 3), (1, 1, 32, 64, 7, 1), (1, 1, 10, 64, 4, 4)):
        for positions, want in ((22500, few), (62500, many)):
            assert ask(positions // 625, 25, 25, cin, cout, kh, kw, 1, 1, -1)[0] == want == int(not _narrow(positions, cin, cout, kh, kw)), (cin, cout, kh, kw)
        if few and not many:  # room for the smaller batches that run it
            assert ask(100, 25, 25, cin, cout, kh, kw, 1, 1, -1)[9] == ask(50, 25, 25, cin, cout, kh, kw, 1, 1, -1)[8] > 0


def test_large_results(ask):
    """More than 64 filters, and a last round of workgroups short of full: not behind a first round, nor in the only one of a large product."""
    for want, batch, cin, cout, kh, kw in ((1, 128, 256, 256, 3, 3), (0, 200, 256, 256, 3, 3), (0, 1000, 128, 512, 3, 3), (1, 200, 128, 128, 3, 3),
                                           (0, 22, 512, 512, 3, 3), (1, 64, 256, 512, 3, 3), (0, 128, 256, 512, 3, 3), (1, 300, 384, 384, 3, 3),
                                           (0, 22, 256, 256, 5, 5), (0, 64, 512, 80, 5, 5), (1, 64, 1024, 64, 5, 5), (1, 150, 512, 64, 5, 5),
                                           (1, 64, 512, 1024, 2, 2), (1, 64, 2048, 1024, 1, 1), (0, 64, 2048, 2048, 1, 1), (1, 300, 192, 192, 3, 3)):
        assert ask(batch, 14, 14, cin, cout, kh, kw, 1, 1, -1)[0] == want, (batch, cin, cout, kh, kw)


def test_which_filter_gradients(ask):
    for want, *shape in ((1, 100, 25, 25, 32, 64, 3, 3, 1, 0),
                         (0, 100, 25, 25, 7, 64, 3, 3, 1, 0),       # a run that leaves most of a tile empty
                         (0, 100, 25, 25, 32, 64, 16, 3, 1, 1),     # a row of the filter for every bit
                         (1, 100, 25, 25, 32, 64, 15, 15, 1, 1),
                         (0, 16, 16, 15, 32, 64, 3, 3, 1, 1),       # 3840 positions
                         (1, 16, 16, 16, 32, 64, 3, 3, 1, 1),
                         (0, 30000, 60, 60, 8, 8, 3, 3, 1, 1)):     # a tensor beyond 2 GiB
        assert ask(*shape, -1)[0] == want, shape

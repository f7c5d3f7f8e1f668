"""Workspace rules of the batch normalisation's reductions (csrc/batchnorm_rules.hpp), compiled without device code."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    binary = str(tmp_path_factory.mktemp("host_checks") / "batchnorm_rules")
    cmd = ["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17",
           os.path.join(ROOT, "tests", "host_checks", "batchnorm_rules.cpp"), "-o", binary]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return lambda *q: [int(v) for v in subprocess.run([binary, *map(str, q)], capture_output=True, text=True, check=True).stdout.split()]


@pytest.mark.parametrize("cols,batch", [(1024, 8275), (512, 16500), (256, 33000), (1000, 9000), (48, 70000), (32, 700000), (12, 5000), (4, 9000), (5, 9000),
                                        (1028, 9000)])
def test_a_workspace_for_the_batch_takes_every_smaller_pass(ask, cols, batch):
    """The workspace is sized for the model's batch; a pass of fewer rows asks for no more."""
    room, asked = ask("room", cols, batch)
    assert asked <= room


@pytest.mark.parametrize("cols", [4, 5, 12, 32, 48, 256, 1000, 1024, 1028])
def test_a_reduction_writes_no_more_slices_than_it_asks_for(ask, cols):
    for rows in (1, 2, 63, 64, 65, 1000, 8192, 8275, 33000, 700001):
        asked, written = ask("written", cols, rows)
        assert 1 <= written <= asked


@pytest.mark.parametrize("cols", [4, 12, 100, 132, 256, 260, 388, 516, 600, 1000, 1024])
def test_whole_vectors_of_channels_fill_the_chip(ask, cols):
    """Slices are workgroups of the streaming form: some 2 for each of 256 CUs where the rows allow it, whatever the channel count."""
    for rows in (8192, 40000):
        _, written = ask("stream", cols, rows)
        assert written >= min(400, rows // 17, rows * cols // 4 // 4096)

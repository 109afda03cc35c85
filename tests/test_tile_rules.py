"""The tile rules of the single-pass launches (indexing_amd/csrc/wah_tiles.h) over
launches of which work on other streams withholds places: a look-back wait must
end as long as each XCD can hold one block.  tests/tile_model runs the rules that
the kernels compile, on the CPU.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    exe = str(tmp_path_factory.mktemp("tiles") / "tile_model")
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror",
                        "-I" + os.path.join(ROOT, "indexing_amd", "csrc"),
                        os.path.join(ROOT, "tests", "tile_model", "tile_model.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return exe


def test_launches_end_with_places_withheld(model):
    r = subprocess.run([model, "shipped"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[-2000:]


def test_model_sees_the_rule_that_stalls(model):
    """A block's first tile by its index, later ones drawn from past the grid."""
    r = subprocess.run([model, "indexed"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 1 and "0 of" not in r.stdout, r.stdout[-2000:]

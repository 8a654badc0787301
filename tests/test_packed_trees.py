"""The packed trees' packer and step rule (csrc/packed_tree.hpp), on the host:
tests/packed_walk.cpp walks random forests both ways, every row for as many
steps as the deepest tree has, as the kernels do."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def walker(tmp_path_factory):
    out = tmp_path_factory.mktemp("packed") / "packed_walk"
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-fno-fast-math", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'xgboost-metal_amd' / 'csrc'}", "-o", str(out), str(ROOT / "tests" / "packed_walk.cpp")],
                   check=True)
    return lambda *args: subprocess.run([str(out), *args], check=True, capture_output=True, text=True).stdout.split()


@pytest.mark.parametrize("seed", range(8))
def test_walks_end_at_their_leaf(walker, seed):
    """Every leaf holds a walk that has reached it, whatever its value: +0 and
    -0 at every depth, single leaves among deeper trees, infinities, NaN."""
    out = walker("forests", str(seed))
    assert int(out[1]) > 20000 and out[2:] == ["mismatches", "0", "outside", "0"], out


def test_leaf_words_are_not_zero(walker):
    assert walker("leaf") == ["walks", "9", "mismatches", "0", "outside", "0"]

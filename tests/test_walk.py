"""The whole-ray walk against the reference's loop body, on the host (CPU only)."""
import os
import subprocess

import numpy as np
import pytest

import oracle_py as orc
from walk_trees import mixed_tree

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def walk_test(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("walk") / "walk_test")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "sparse-voxel-octrees_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "walk_test.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("tree", ["dragon", "mixed1", "mixed2", "mixed3", "mixed10", "mixed22", "mixed23",
                                  "loose3", "loose10"])
def test_walk_equals_the_reference_loop(walk_test, golden, tmp_path, tree):
    if tree == "dragon":
        _, words = orc.read_oct(os.path.join(golden, "dragon.oct"))
        levels = 8
    else:
        levels = int(tree[5:])
        words = mixed_tree(levels, levels, loose=tree.startswith("loose"))
    path = str(tmp_path / "words.bin")
    np.ascontiguousarray(words, np.uint32).tofile(path)
    r = subprocess.run([walk_test, path, str(levels), "20000"] + (["loose"] if tree.startswith("loose") else []), capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("ok ")


@pytest.mark.parametrize("levels,seed,loose", [(1, 2, False), (2, 2, False), (3, 3, False), (10, 10, False), (23, 23, False),
                                               (3, 3, True), (10, 10, True)])
def test_compared_walks_end_in_leaves_and_cut_offs(walk_test, tmp_path, levels, seed, loose):
    """The comparison above is of rays of every outcome: at least a tenth of its
    walks end in a leaf and a hundredth at a cut-off, misses are the rest."""
    path = str(tmp_path / "words.bin")
    mixed_tree(seed, levels, loose=loose).tofile(path)
    r = subprocess.run([walk_test, path, str(levels), "20000"] + (["loose"] if loose else []), capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    walks, leaves, cuts = (int(r.stdout.split()[k]) for k in (1, 3, 6))
    assert leaves >= walks / 10 and cuts >= walks / 100 and walks - leaves - cuts >= walks / 100, r.stdout

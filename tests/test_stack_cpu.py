"""The traversal stack's bounds (luxcore_amd/csrc/lrh_stack.h, compiled for the
host): the single and the shared pushes and pops of a ray are a plain stack's;
where the ring and the spill array are full a push reports it, and no push or
pop after it touches anything outside the two arrays."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("stack") / "stack_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-D_GLIBCXX_ASSERTIONS", "-o", str(out),
                    os.path.join(ROOT, "tests", "native", "stack_check.cpp")], check=True, timeout=180)
    return out


@pytest.mark.parametrize("width", [4, 8])
@pytest.mark.parametrize("lds,spill", [(4, 1), (4, 3), (4, 40), (8, 1), (8, 25), (16, 7), (64, 1)])
def test_stack_is_a_plain_one_up_to_its_bound(exe, lds, spill, width):
    for seed in range(6):
        p = subprocess.run([str(exe), str(lds), str(spill), str(width), str(seed), "3000"], capture_output=True, text=True,
                           timeout=60)
        assert p.returncode == 0, (seed, p.stdout)
        word, beyond, deepest = p.stdout.split()
        assert word == "ok"
        assert lds + spill > 60 or (int(beyond) > 0 and int(deepest) > lds)

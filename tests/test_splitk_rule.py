"""How many k slices the layer gives FFN2: the rule of include/bytetransformer/common.h, compiled as the host compiles it."""
import os
import subprocess

import pytest

from bytetransformer_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include <cstdio>
#include <cstdlib>
#include "bytetransformer/common.h"
int main(int argc, char **argv) {
  for (int i = 1; i + 2 < argc; i += 3)
    std::printf("%d\\n", bytetransformer::splitk_splits(std::atoll(argv[i]), std::atoll(argv[i + 1]), std::atoi(argv[i + 2])));
}
"""
# capacity, expected rows, k -> slices
CASES = [((32, 32, 3072), 4), ((512, 192, 3072), 4), ((512, 193, 3072), 2), ((513, 192, 3072), 2), ((1024, 640, 3072), 2),
         ((1024, 641, 3072), 1), ((1025, 300, 3072), 1), ((32, 32, 2048), 4), ((32, 32, 1984), 1), ((32, 32, 2176), 2),
         ((32, 32, 2112), 1), ((700, 640, 8192), 2), ((700, 700, 8192), 1)]


@pytest.fixture(scope="module")
def answers(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("rule")
    source, program = str(tmp / "rule.cc"), str(tmp / "rule")
    with open(source, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++"] + build.HOST_FLAGS + ["-I", os.path.join(ROOT, "include"), "-I",
                                                 os.path.join(build.ROCM, "include"), source, "-o", program], check=True)
    env = {k: v for k, v in os.environ.items() if k != "BT_SPLITK"}
    out = subprocess.run([program] + [str(v) for args, _ in CASES for v in args], check=True, stdout=subprocess.PIPE,
                         text=True, env=env).stdout
    return [int(v) for v in out.split()]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_slices(answers, i):
    args, want = CASES[i]
    assert answers[i] == want, args

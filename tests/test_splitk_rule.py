"""How many k slices the layer gives FFN2: the measured rule of the kernels library, and the rule of
include/bytetransformer/common.h for parts that it was not measured on, compiled as the host compiles it."""
import os
import subprocess
import threading
import time

import pytest

from bytetransformer_amd import _lib, build

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


# rows that are all live, hidden, k -> slices, each the fastest of a layer's measured ones or within 1 % of it
@pytest.mark.parametrize("rows,n,k,slices", [
    (32, 768, 3072, 4), (900, 768, 3072, 4), (1500, 768, 3072, 3), (1984, 768, 3072, 2), (2240, 768, 3072, 2), (2400, 768, 3072, 2),
    (2600, 768, 3072, 1), (64, 1024, 4096, 4), (96, 1024, 4096, 4), (1600, 1024, 4096, 2), (2240, 1024, 4096, 1),
    (64, 1280, 5120, 4), (512, 512, 2048, 4), (1088, 512, 2048, 1), (1984, 512, 2048, 1), (1280, 576, 2304, 1)])
def test_measured_slices(rows, n, k, slices):
    assert _lib.kernel_lib().bt_gemm_splitk_slices(rows, 1, n, k, 16) == slices


def test_slices_of_a_padded_batch():
    """60 % of the rows, or less likely all of them; never more slices than there is room for; whole k for short k or no rows."""
    ask = _lib.kernel_lib().bt_gemm_splitk_slices
    assert ask(384, 0, 768, 3072, 16) in (3, 4)
    assert ask(4000, 0, 768, 3072, 16) == 1 and ask(3000, 0, 768, 3072, 16) == 2
    for most in (0, 1, 2, 3, 16):
        assert 1 <= ask(1500, 0, 768, 3072, most) <= max(most, 1)
    assert ask(0, 0, 768, 3072, 16) == ask(100, 0, 768, 32, 16) == ask(100, 0, 768, 3000, 16) == 1
    for n, k in ((768, 3072), (1024, 4096), (512, 2048), (640, 2560)):
        for rows in range(1, 3000, 61):
            assert (k // 64) % ask(rows, 0, n, k, 16) == 0


def test_remembered_answers_are_those_of_their_sizes():
    """Far more sizes than are remembered, in several orders and on several threads at once."""
    ask = _lib.kernel_lib().bt_gemm_splitk_slices
    sizes = [(rows, live, n, 4 * n, most) for n in (512, 768, 1024) for rows in range(1, 3000, 37) for live in (0, 1)
             for most in (2, 16)]
    first = [ask(*s) for s in sizes]
    seen = {}

    def again(step):
        seen[step] = [ask(*sizes[i * step % len(sizes)]) for i in range(len(sizes))]
    threads = [threading.Thread(target=again, args=(step,)) for step in (1, 7, 11, 13)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    for step, got in seen.items():
        assert got == [first[i * step % len(sizes)] for i in range(len(sizes))], step


def test_a_size_is_priced_once():
    """A forward asks the same in every layer: the answer is looked up, for less than a third of what it costs to find."""
    ask = _lib.kernel_lib().bt_gemm_splitk_slices

    def ns(rows):
        best = []
        for _ in range(7):
            t0 = time.perf_counter_ns()
            for r in rows:
                ask(r, 0, 768, 3072, 16)
            best.append(time.perf_counter_ns() - t0)
        return min(best) / len(rows)
    other = ns([0] * 600)                        # (the call itself; no rows are answered at once)
    assert ns([384] * 600) - other < (ns(list(range(300, 900))) - other) / 3

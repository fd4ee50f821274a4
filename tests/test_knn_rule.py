"""Which kernel a neighbour search takes (kernels.h), evaluated on the host."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = """
#include <cstdio>
#include <cstdint>
#include "kernels.h"
int main() {
    int dim, k, line;
    long long nq;
    while (scanf("%d %lld %d %d", &dim, &nq, &k, &line) == 4) printf("%d\\n", (int)pg::knn_by_wave(dim, nq, k, line));
}
"""


@pytest.fixture(scope="module")
def by_wave(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", os.path.join(ROOT, "proteusgpu_amd", "csrc"),
                    str(d / "rule.cpp"), "-o", str(d / "rule")], check=True)

    def ask(*queries):
        r = subprocess.run([str(d / "rule")], input="\n".join(" ".join(map(str, q)) for q in queries), check=True,
                           capture_output=True, text=True)
        return [bool(int(x)) for x in r.stdout.split()]

    return ask


def test_faster_kernel_at_measured_sizes(by_wave):
    """Sizes at which one kernel was measured faster by a tenth or more."""
    wave = [(2, 14000, 1), (2, 50000, 4), (2, 100000, 8), (2, 200000, 12), (2, 1000000, 16), (3, 14000, 1),
            (3, 50000, 1), (3, 100000, 2), (3, 200000, 5), (3, 300000, 8), (3, 400000, 6), (3, 400000, 10), (3, 1000000, 12)]
    heap = [(2, 100000, 1), (2, 200000, 4), (2, 300000, 8), (2, 1000000, 12), (3, 200000, 1), (3, 200000, 2),
            (3, 300000, 1), (3, 300000, 4), (3, 400000, 4), (3, 1000000, 6)]
    assert all(by_wave(*((*q, 20) for q in wave)))
    assert not any(by_wave(*((*q, 20) for q in heap)))


def test_a_set_line_is_kept(by_wave):
    """A program's own row length decides alone, whatever the list's length."""
    q = [(dim, nq, k, line) for dim in (2, 3) for nq in (1000, 300000, 5000000) for k in (1, 8, 16, 24, 32, 100, 256)
         for line in (1, 12, 19, 21, 33, 300)]
    assert by_wave(*q) == [k >= line for _, _, k, line in q]

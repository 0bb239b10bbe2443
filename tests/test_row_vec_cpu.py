"""The causal conv's reads stay inside their row: the rule its kernels read by
(csrc/row_vec.hpp), built for the host and tried at every row length around the
vector's and every vector a thread asks for, the ones ahead of and past the row
among them."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mamba_amd", "csrc")
PROGRAM = """
#include <cstdio>
#include <initializer_list>
#include "row_vec.hpp"
int main() {
    int bad = 0;
    for (int vw : {4, 8})
        for (int64_t n = 1; n <= 4 * vw + 1; ++n)
            for (int64_t i = -vw; i <= n + 2 * vw; i += vw) {
                int64_t first, last;
                if (ss::row_vec_ok(ss::rows_of(n, vw), i, n, vw)) {
                    first = ss::row_vec_at(i, n);
                    last = first + vw - 1;
                    if (ss::row_in(i, n) && first != i) ++bad, std::printf("vector %ld of %ld at %ld\\n", i, n, first);
                } else {
                    first = ss::row_elem(i, n);
                    last = ss::row_elem(i + vw - 1, n);
                    for (int64_t k = i; k < i + vw; ++k)
                        if (ss::row_in(k, n) && ss::row_elem(k, n) != k) ++bad, std::printf("element %ld of %ld\\n", k, n);
                }
                if (first < 0 || last >= n) ++bad, std::printf("vw %d n %ld i %ld reads [%ld, %ld]\\n", vw, n, i, first, last);
            }
    return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_reads_stay_inside_the_row(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout

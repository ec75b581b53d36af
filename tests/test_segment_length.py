"""The common z-segment length of an ensemble's members (csrc/hip/fe_segments.h), in a C++ program of
its own: members of one, two and three levels, alone, mixed and beside a taller member whose segments are
set, have one segment each; the lengths measured best on 256 work-groups; a member without levels to
choose for is no member.
"""
import os
import subprocess

import pytest

SOURCE = r"""
#include "fe_segments.h"
#include <stdio.h>
#include <stdlib.h>

/* slots, then tiles, levels and set length of each member */
int main(int argc, char **argv) {
  std::vector<SegMember> mem;
  for (int i = 2; i + 2 < argc; i += 3) mem.push_back(SegMember{atol(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2])});
  const int len = ens_segment_length(mem, atoi(argv[1]));
  printf("%d\n", len);
  for (auto &m : mem) {
    int zseg = m.zseg, nseg = 0;
    if (zseg <= 0) seg_shape(m.Nz, (m.Nz + len - 1) / len, zseg, nseg);
    printf("%d\n", (m.Nz + zseg - 1) / zseg);
  }
}
"""


@pytest.fixture(scope="module")
def program(repo, tmp_path_factory):
    d = tmp_path_factory.mktemp("segments")
    (d / "main.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wno-unused-function",
                    "-I" + os.path.join(repo, "fasteddy-model_amd", "csrc", "hip"), str(d / "main.cpp"), "-o", str(d / "main")],
                   check=True)
    return str(d / "main")


# members (tiles, levels, set length), segment counts
CASES = [([(1, nz, 0)], [1]) for nz in (1, 2, 3, 4)] + [
    ([(8, 1, 0), (8, 3, 0), (8, 2, 0)], [1, 1, 1]),
    ([(3, 22, 8), (1, 2, 0)], [3, 1]), ([(1, 1, 0), (30, 64, 16)], [1, 4]),
    ([(8, 48, 0)], [12]), ([(8, 48, 0)] * 16, [2] * 16), ([(4, 4, 0)] * 3, [1] * 3),
    ([(2, 22, 8), (9, 33, 34)], [3, 1])]


@pytest.mark.parametrize("mem,nseg", CASES)
def test_segment_length(program, mem, nseg):
    r = subprocess.run([program, "256"] + [str(v) for m in mem for v in m], capture_output=True, text=True, timeout=20)
    assert r.returncode == 0, r.returncode
    out = [int(v) for v in r.stdout.split()]
    assert out[0] >= 4 and out[0] % 2 == 0
    assert out[1:] == nseg

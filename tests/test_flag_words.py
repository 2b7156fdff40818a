"""The arrival test of the local updates' barrier words (flag_arrived), run on the host: a chain's
counter is 32 bits and wraps, words of workgroups that sat out for a while keep an old value."""
import os
import subprocess

import pytest

from dqmc_amd import build

PROGRAM = """
#include "chain.hpp"
#include <cstdio>
int main(int, char** v) {
  unsigned word, target;
  while (scanf("%u %u", &word, &target) == 2) printf("%d\\n", dqmc::flag_arrived(word, target) ? 1 : 0);
}
"""


def test_flag_arrived(tmp_path):
    src, exe = tmp_path / "t.hip", tmp_path / "t"
    src.write_text(PROGRAM)
    try:
        cc = build.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    subprocess.run([cc, "-x", "hip", "--offload-host-only", "-std=c++17", "-I", build.SRC, str(src), "-o", str(exe)],
                   check=True, capture_output=True, cwd=os.path.dirname(exe))
    top = 2**32
    cases = []
    for target in (0, 1, 2, 1000, 2**31 - 1, 2**31, 2**31 + 1, 2**32 - 1):
        for ahead in (0, 1):
            cases.append(((target + ahead) % top, target, 1))
        for behind in (1, 2, 50, 2**31 - 1, 2**31, 2**31 + 1, 2**32 - 50):  # idle for that many barriers
            cases.append(((target - behind) % top, target, 0))
    out = subprocess.run([str(exe)], input="".join("%d %d\n" % c[:2] for c in cases), check=True, capture_output=True,
                         text=True).stdout.split()
    assert [int(x) for x in out] == [c[2] for c in cases]

"""The mapping from workgroups to sets of blocks of the encoders (csrc/sage_grid.h), asked of the host compiler: every member of
every set is taken once, and all members of a set by one XCD (workgroup id modulo 8)."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mojodiffusion_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "sage_grid.h"
int main() {
    int sets, members;
    while (std::scanf("%d %d", &sets, &members) == 2) {
        const long long n = sage::set_grid(sets, members);
        std::vector<int> seen(n), xcd(n / members, -1);
        int bad = n < (long long)sets * members || n >= (long long)(sets + sage::kSetGroup) * members;
        for (long long id = 0; id < n; id++) {
            const sage::SetMember m = sage::set_member((int)id, members);
            if (m.set < 0 || m.set >= n / members || m.member < 0 || m.member >= members) { bad++; continue; }
            seen[(long long)m.set * members + m.member]++;
            if (xcd[m.set] < 0) xcd[m.set] = id & 7;
            bad += xcd[m.set] != (id & 7);
        }
        for (int c : seen) bad += c != 1;
        std::printf("%d\n", bad);
    }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_every_member_once_and_a_set_on_one_xcd(tmp_path):
    src, exe = tmp_path / "m.cpp", tmp_path / "m"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__host__=", "-D__device__=", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    cases = [(s, m) for s in (1, 31, 32, 33, 456, 1020, 2880) for m in (1, 2, 3, 5, 6, 12, 18)]
    out = subprocess.run([str(exe)], input="\n".join("%d %d" % c for c in cases), capture_output=True, text=True, check=True).stdout
    assert out.split() == ["0"] * len(cases)

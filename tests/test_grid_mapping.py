"""The mapping from workgroups to blocks of the backward (csrc/sage_grid.h), asked of the host compiler: every block is
taken once, and the blocks that hold rows that count go to the XCDs (workgroup id modulo 8) in even numbers."""
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
    int heads, sq, rq, sk, rk, kw;
    while (std::scanf("%d %d %d %d %d %d", &heads, &sq, &rq, &sk, &rk, &kw) == 6) {
        const int tq = (sq + 255) / 256, lq = (rq + 255) / 256, tk = (sk + kw - 1) / kw, lk = (rk + kw - 1) / kw;
        std::vector<int> seen(heads * (tq + tk));
        int live[2][8] = {}, bad = 0, last_q = -1, first_k = 1 << 30;
        for (int id = 0; id < heads * (tq + tk); id++) {
            const sage::BwdBlock b = sage::bwd_block(id, heads, tq, lq, tk, lk);
            const int t = b.dkdv ? tk : tq;
            if (b.head < 0 || b.head >= heads || b.tile < 0 || b.tile >= t) { bad++; continue; }
            seen[b.dkdv ? heads * tq + b.head * tk + b.tile : b.head * tq + b.tile]++;
            if (b.tile >= (b.dkdv ? lk : lq)) continue;
            live[b.dkdv][id & 7]++;
            if (b.dkdv) first_k = id < first_k ? id : first_k; else last_q = id;
        }
        for (int n : seen) bad += n != 1;
        int spread = 0;
        for (auto& kind : live) {
            int lo = kind[0], hi = kind[0];
            for (int n : kind) { lo = n < lo ? n : lo; hi = n > hi ? n : hi; }
            spread = hi - lo > spread ? hi - lo : spread;
        }
        std::printf("%d %d %d\n", bad, spread, last_q < first_k);
    }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_every_block_once_and_the_live_ones_evenly(tmp_path):
    src, exe = tmp_path / "m.cpp", tmp_path / "m"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__host__=", "-D__device__=", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    cases = [(12, 4608, 2304, 4608, 2304), (12, 2304, 1612, 2304, 1612), (1, 100, 1, 4000, 4000), (1, 5000, 4999, 64, 1), (60, 1248, 748, 1248, 748)]
    cases += [(h, s, max(1, s * r // 20), s2, max(1, s2 * r // 20)) for h in (1, 3, 7, 8, 9, 16, 24, 30, 40) for s, s2 in ((257, 257), (1248, 1248), (4608, 333))
              for r in (1, 7, 10, 13, 19, 20)]
    cases = [c + (kw,) for c in cases for kw in (128, 256)]
    out = subprocess.run([str(exe)], input="\n".join(" ".join(map(str, c)) for c in cases), capture_output=True, text=True, check=True).stdout
    got = [tuple(map(int, line.split())) for line in out.splitlines()]
    assert len(got) == len(cases)
    # (whole heads per XCD: even as they are.  Otherwise the two ranges of a kind differ by a block at most)
    wrong = [(c, g) for c, g in zip(cases, got) if g[0] != 0 or g[1] > 1 or g[2] != 1]
    assert not wrong, wrong[:5]

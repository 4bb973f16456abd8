"""The decode grid's rule (bmx_amd/csrc/split_plan.h) over batches, head counts, lengths and windows, from a host
program built against the header: heads that are spread over several workgroups never leave the window to the
splits (each block of heads would score all of it), and no plan that spreads them asks for more workgroups than CUs."""

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "bmx_amd" / "csrc"
PROBE = r"""
#include <cstdio>
#include "split_plan.h"
int main() {
  for (int cus : {64, 256, 304})
    for (int batch : {1, 2, 3, 5, 7, 8, 16, 31, 72, 128, 300})
      for (int h = 1; h <= 8; ++h)
        for (int groups : {0, 1, 2, 4, 5, 10, 13, 16, 21, 31, 32, 33, 42, 64, 84, 126, 255, 512})
          for (int tail : {0, 1, 16, 17, 60, 128, 161, 255, 1024})
            for (int split : {0, 64, 512}) {
              const bmx::SplitPlan p = bmx::plan_splits(batch, h, groups, 64 * groups, split, tail, cus);
              printf("%d %d %d %d %d %d %d %d %d %d\n", cus, batch, h, groups, tail, split, p.S, p.blocks, p.hpb,
                     p.win_wgs);
            }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not found")
def test_spread_heads_have_window_workgroups(tmp_path):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PROBE)
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    spread = 0
    for line in out.splitlines():
        cus, batch, h, groups, tail, split, S, blocks, hpb, win = map(int, line.split())
        pairs = (tail + 15) // 16 * h
        assert S >= 1 and blocks >= 1 and blocks * hpb >= h and win >= 0, line
        assert win == 0 or win * blocks * 8 >= pairs, line          # every pair a wave
        if blocks > 1:
            spread += 1
            assert split == 0 and blocks <= h and S <= max(1, groups), line
            assert win > 0 or pairs == 0, line
            assert batch * blocks * (S + win) <= cus, line
    assert spread > 1000

"""The launches that give a lane to every cell of a box of ni planes of pl cells
(dtm_box.h), compiled for the host: every cell of every plane is taken exactly
once, no launch has more blocks than allowed, and few lanes have none: planes of
one cell up to several launches each, units that end with the box or beyond it,
limits of a few blocks in place of the device's 2^24."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dtmaxwell4_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include <vector>
#define __host__
#define __device__
#define __forceinline__ inline
#include "dtm_box.h"
using namespace dtm;
int main() {
  const unsigned nis[] = {1, 2, 7, 8, 9, 100, 2047, 2048, 2049, 5000};
  const unsigned long long pls[] = {1, 2, 3, 16, 255, 256, 257, 680, 1024, 2047, 2048, 2049, 5000};
  const unsigned long long mosts[] = {1, 3, 7, 8, 9, 16, 20, 1000, (1u << 24) - 1};
  for (unsigned ni : nis)
    for (unsigned long long pl : pls)
      for (unsigned long long most : mosts) {
        if (ni * pl > 3000000) continue;
        std::vector<unsigned char> seen(ni * pl, 0);
        unsigned long long lanes = 0, twice = 0, big = 0;
        box_launches(ni, pl, [&](const BoxUnits& B, unsigned blocks) {
          big += blocks > most || blocks == 0;
          lanes += blocks * (unsigned long long)kBoxBlock;
          for (unsigned b = 0; b < blocks; b++)
            for (unsigned t = 0; t < kBoxBlock; t++) {
              unsigned ip;
              unsigned long long loc;
              if (box_lane(B, ni, pl, b, t, ip, loc)) twice += seen[ip * pl + loc]++;
            }
        }, most);
        unsigned long long missed = 0;
        for (unsigned char v : seen) missed += v == 0;
        // a unit leaves less than a block over, and the last unit planes beyond the box
        const bool wasteful = lanes > ni * pl + ni * pl / 8 + 2 * kBoxUnit;
        if (missed || twice || big || wasteful) {
          std::printf("ni %u pl %llu most %llu: missed %llu, twice %llu, launches too large %llu, lanes %llu\n", ni, pl,
                      most, missed, twice, big, lanes);
          return 1;
        }
      }
  // planes of more than 2^32 cells: the first and last cells of the last plane
  const unsigned long long pl = (1ull << 33) + 77;
  unsigned long long first = 0, last = 0;
  box_launches(2, pl, [&](const BoxUnits& B, unsigned blocks) {
    unsigned ip;
    unsigned long long loc;
    if (box_lane(B, 2, pl, 0, 0, ip, loc) && ip == 1 && loc == 0) first++;
    for (unsigned t = 0; t < kBoxBlock; t++)
      if (box_lane(B, 2, pl, blocks - 1, t, ip, loc) && ip == 1 && loc == pl - 1) last++;
  });
  if (first != 1 || last != 1) {
    std::printf("first %llu last %llu\n", first, last);
    return 1;
  }
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_cell_once(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=100)
    assert r.returncode == 0, r.stdout

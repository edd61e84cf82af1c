"""The fp32 kernels' staging addresses (csrc/ssd_stage.h) on the CPU: over every tile width, block size and wave, at
the largest row stride the C ABI takes (65535 heads of 128 columns) and a small one, each piece's resource base plus
its 32-bit byte offset is the address that 64-bit arithmetic gives, and the last byte lies inside the resource
(SSD_BUF_SIZE, 0x7ffffff0). A head's 64-column half (widths above 64 in the forward scan) is the case whose rows lie
furthest apart: 115 of them under one resource would be 3.9 GB there."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "dhammic-ai_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "ssd_stage.h"
int main() {
  long pieces = 0;
  const int64_t strides[] = {65535LL * 128, 36500LL * 128, 33};
  for (int W : {32, 64, 128})
    for (int nthr : {64, 128, 192, 256, 384, 512})
      for (int64_t ld : strides) {
        const int cpr = W / 4, total = 256 * cpr, NB = 8;
        bool seen[256 * 32] = {};
        for (int t = 0; t < nthr; ++t)
          for (int id0 = t; id0 < total; id0 += NB * nthr) {
            const int w0 = id0 - t % 64;  // the wave's first lane
            const int64_t off = stage_off(id0, w0, cpr, ld);
            for (int q = 0; q < NB && id0 + q * nthr < total; ++q) {
              const int id = id0 + q * nthr;
              const int64_t want = (int64_t)stage_row(id, cpr) * ld + stage_col(id, cpr);
              const int64_t base = stage_base(w0, q, nthr, cpr) * ld;
              if (base + off != want || off < 0 || (off + 4) * 4 > 0x7ffffff0LL) {
                std::printf("W %d nthr %d ld %lld id %d: %lld + %lld, want %lld\n", W, nthr, (long long)ld, id,
                            (long long)base, (long long)off, (long long)want);
                return 1;
              }
              seen[id] = true;
              ++pieces;
            }
          }
        for (int id = 0; id < total; ++id)
          if (!seen[id]) return 2;
      }
  std::printf("ok %ld\n", pieces);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_staging_addresses_fit(tmp_path):
    src, exe = tmp_path / "addr.cpp", tmp_path / "addr"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout + out.stderr

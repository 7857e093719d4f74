"""Group parameters of the few-row INT4 kernel on the host: the reads that fill
its LDS (csrc/qg_w4_params.h, compiled by g++) stay inside the arrays and cover
every group of every column."""
from pathlib import Path
import subprocess

CSRC = Path(__file__).resolve().parent.parent / "rdna2-gfx1030-ai-handbook_amd" / "csrc"
PROGRAM = r"""
#include "qg_w4_params.h"
#include <cstdio>
using namespace qg;
int main() {
  for (uint32_t N = 1; N <= 40; ++N)
    for (uint32_t ng = 1; ng <= 24; ++ng)
      for (int f32 = 0; f32 < 2; ++f32) {
        const uint32_t es = f32 ? 4 : 2, end = N * ng * es, zw = (ng + 7) / 8;
        for (uint32_t n = 0; n < N; ++n) {
          const int pitch = w4_scale_pitch(ng, f32);
          for (int w = 0; w < pitch; ++w) {
            const W4Read r = w4_scale_read(n, N, ng, f32, w);
            if (r.offset % 4 != 0 || r.offset + r.bytes > end) {
              std::printf("N %u ng %u f32 %d column %u word %d: bytes %u to %u of %u\n", N, ng, f32, n, w, r.offset,
                          r.offset + r.bytes, end);
              return 1;
            }
          }
          // group g of the column: the kernel reads element odd + g of the column's words
          const uint32_t odd = f32 ? 0 : n * ng & 1;
          for (uint32_t g = 0; g < ng; ++g) {
            const uint32_t at = (odd + g) * es;
            const W4Read r = w4_scale_read(n, N, ng, f32, at / 4);
            if (static_cast<int>(at / 4) >= pitch || r.offset + at % 4 != (n * ng + g) * es || at % 4 + es > r.bytes) {
              std::printf("N %u ng %u f32 %d column %u group %u\n", N, ng, f32, n, g);
              return 1;
            }
          }
          for (int packed = 0; packed < 2; ++packed) {
            const uint32_t per = packed ? zw : ng;
            for (int w = 0; w < w4_zero_pitch(ng, zw, packed); ++w) {
              const W4Read r = w4_zero_read(n, per, w);
              if (r.offset + r.bytes > 4 * N * per) return 1;
              if (static_cast<uint32_t>(w) < per && r.offset != 4 * (n * per + w)) return 1;
            }
          }
        }
      }
  return 0;
}
"""


def test_reads_stay_inside_the_arrays(tmp_path):
    (tmp_path / "reads.cpp").write_text(PROGRAM)
    exe = tmp_path / "reads"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{CSRC}", str(tmp_path / "reads.cpp"), "-o",
                    str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout

"""Row offsets inside a buffer resource (csrc/row_offset.h), on the host: for every pitch that
the launch's own bound lets through, a row of the batch stays where it is and a row past it
never falls back inside the resource."""

import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "llmnputest_amd" / "csrc"

PROGRAM = r"""
#include "row_offset.h"
#include <stdio.h>
using namespace q4nx;
int main() {
  long n = 0;
  const uint32_t row_bytes = 8192 * 4;                       // the widest row, fp32
  for (int rows = 1; rows <= 8; ++rows) {
    const uint64_t top = ((uint64_t(1) << 31) - 1) / rows;   // rows * pitch < 2^31
    for (int step = 0; step < 4096; ++step) {
      const uint32_t pitch = (uint32_t)(row_bytes + (top - row_bytes) * step / 4095) & ~31u;
      const uint64_t records = (uint64_t)rows * pitch;
      for (int r = 0; r < 8; ++r, ++n) {
        const uint64_t first = row_offset(r, rows, pitch);
        const uint32_t last = row_offset(r, rows, pitch) + (row_bytes - 16);
        if (r < rows ? first != (uint64_t)r * pitch || last + 16ull > records
                     : first < records || last < records)
          return printf("rows %d pitch %u row %d: %llu\n", rows, pitch, r, (unsigned long long)first), 1;
      }
    }
  }
  printf("%ld\n", n);
  return 0;
}
"""


def test_rows_past_the_batch_stay_out_of_range(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "t"
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout) == 8 * 4096 * 8


def test_in_kernel_norm_uses_it():
    """The in-kernel RMSNorm takes every row's offset from there (a product of its own would wrap
    for two rows 0.8 GB apart: 6 * 0.8e9 mod 2^32 lies between them)."""
    text = (CSRC / "gemm.hip").read_text()
    body = text[text.index("auto hload"):text.index("auto hnorm")]
    assert "hrow[i]" in body and "x_stride" not in body
    assert "hrow[i] = row_offset(" in text

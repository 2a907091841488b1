"""The synthetic inflow launch's LDS stays within the 64 KB that its form is chosen for, at every row
length that plans accept (host arithmetic, compiled here); rows that were evaluated cooperatively
stay so, and the narrow ones keep two row buffers."""
import os
import subprocess

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "wmles_jax_amd", "csrc")
CODE = r"""
#include <stdio.h>
#include <initializer_list>
#include "inflow.h"
int main() {
  for (int N2 = 9; N2 <= 1024; ++N2)
    for (int nm = 1; nm <= 256; ++nm)
      for (int nt : {1, 64, 4096}) {
        const wmx::InflowForm f = wmx::inflow_form(N2, nm, nt);
        const size_t table = sizeof(double) * ((size_t)(N2 | 1) * nm + 2 * (size_t)N2);
        const size_t fixed = sizeof(double) * ((size_t)f.rows * f.threads + 1);
        if (f.lds > 65536 || f.lds != fixed + (f.coop ? table : 0) + (f.coop == 2 ? 8u * nt : 0) ||
            (f.coop > 0) != (table <= 56 * 1024) || f.rows < 1 || f.rows > 2 || (N2 <= 512 && f.rows != 2) ||
            f.threads < N2 || f.threads > 1024 || f.threads % 64)
          return printf("%d %d %d: coop %d rows %d threads %d lds %zu\n", N2, nm, nt, f.coop, f.rows, f.threads, f.lds), 1;
      }
}
"""


def test_the_launch_fits_64_kb(tmp_path):
    (tmp_path / "form.cpp").write_text(CODE)
    exe = str(tmp_path / "form")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", SRC, str(tmp_path / "form.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout

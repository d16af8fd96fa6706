"""The reverse pass takes a formula's wall terms computed or left out; the mode
that decides per cell would lose their gradient and does not compile."""
import os
import subprocess

import pytest

from pascal_tcs_amd import build

SRC = r"""
#include "rev.h"
using namespace tcs;
__global__ void k(double *o, bool near) {
    double bar = 0.0;
    Rev out{1.0};
    { const Ref x(o[0], &bar);
      const auto y = as<Rev>(with_walls<Rev, MODE>(near, x, [&](const auto &v) { return v * 2.0; }));
      out = y * 3.0; }
    o[1] = bar;
}
"""


@pytest.mark.parametrize("mode,compiles", [(0, True), (1, False), (2, True)])
def test_wall_modes_of_the_reverse_pass(tmp_path, mode, compiles):
    try:
        cc = build.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    src = tmp_path / "t.hip"
    src.write_text(SRC.replace("MODE", str(mode)))
    r = subprocess.run([cc, "-std=c++17", f"--offload-arch={build.ARCH}", "--offload-device-only", "-fsyntax-only",
                        "-DTCS_REV", "-I", build.CSRC, str(src)], capture_output=True, text=True, timeout=120)
    assert (r.returncode == 0) == compiles, r.stderr[-2000:]
    if not compiles:
        assert "wall terms of the reverse pass" in r.stderr

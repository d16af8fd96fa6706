"""Every launch whose dynamic LDS may pass 64 KiB raises its kernel's limit
first: in each source, a launch of a transform or of a solve with run-time
LDS is preceded, in its own function, by lds_limit."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _function(text, name):
    """The body of function `name`, to the next line that starts with '}'."""
    at = re.search(r"^(?:static |template[^\n]*\n)?[^\n;]*\b" + name + r"\([^;]*?\{$", text, re.M | re.S)
    assert at, name
    return text[at.start():text.index("\n}", at.end())]


@pytest.mark.parametrize("source,name", [("pressure.hip", "fft_x_fwd_src_launch"), ("pressure.hip", "fft_x_inv_launch"),
                                         ("pressure.hip", "fft_z_launch"), ("tdma.hip", "ptdma_exact_launch"),
                                         ("tdma_part.hip", "part_launch"), ("tdma_part.h", "part_rows_src_launch")])
def test_limit_raised_before_the_launch(source, name):
    with open(os.path.join(ROOT, "pascal_tcs_amd", "csrc", source)) as f:
        body = _function(f.read(), name)
    assert "lds_limit(" in body and body.index("lds_limit(") < body.rindex("TCS_LAUNCH(")

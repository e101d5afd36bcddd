"""Every kernel that the library times under one name is counted under that name
by the profile summaries: the tridiagonalisation's panels run as one of two kernels,
its resident part as one of two others."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gammcor_amd", "csrc")


@pytest.mark.parametrize("kernel,key", [("sytrd_panel_kernel", "sytrd_panel"), ("sytrd_xpanel_kernel", "sytrd_panel"),
                                        ("sytrd_resident_kernel", "sytrd_resident"),
                                        ("sytrd_resident_rows_kernel", "sytrd_resident")])
def test_tridiagonalisation_kernels(kernel, key):
    from gammcor_amd import profsum
    text = "".join(open(os.path.join(CSRC, f)).read() for f in os.listdir(CSRC))
    assert re.search(rf"__global__[^;{{]*\b{kernel}\(", text)
    for t, suffix in (("float", "f32"), ("double", "f64")):
        assert f'"{key}_{suffix}"' in text
        assert profsum.timing_key(f"void gmc::{kernel}<{t}, true, 8, 1>(gmc::Args<{t}>)") == f"{key}_{suffix}"

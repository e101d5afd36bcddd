"""The exchange between the workgroups of the resident tridiagonalisation takes a
value for there when any of its bits is set, so a value must become visible
whole: it travels in an access of its own size.  The accesses are found in the
compiled kernels by their cache policy (agent scope: sc1); none may be wider than
8 bytes."""
import os
import re
import subprocess

import pytest

SOURCE = """
#include "common.hpp"
#include "wave_ops.hpp"
namespace gmc {
template <int N>
constexpr int ilog2()
{
    int l = 0;
    for (int n = N; n > 1; n /= 2) l++;
    return l;
}
#include "sytrd_resident.hpp"
template __global__ void sytrd_resident_kernel<T, 8, 2>(ResArgs<T>);
template __global__ void sytrd_resident_kernel<T, 16, 4>(ResArgs<T>);
template __global__ void sytrd_resident_rows_kernel<T, 4, 2, 4>(ResArgs<T>);
template __global__ void sytrd_resident_rows_kernel<T, 8, 8, 8>(ResArgs<T>);
}
"""


@pytest.mark.parametrize("dtype", ["double", "float"])
def test_no_exchange_access_beyond_eight_bytes(tmp_path, dtype):
    from gammcor_amd import build
    src, asm = tmp_path / "words.hip", tmp_path / "words.s"
    src.write_text(re.sub(r"\bT\b", dtype, SOURCE))
    cmd = [build.HIPCC, *build.HIPFLAGS, "--cuda-device-only", "-I", build.CSRC, "-S", str(src), "-o", str(asm)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    access = re.findall(r"^\s*(buffer_(?:load|store)_\w+).* sc1", asm.read_text(), re.M)
    assert {"buffer_load_dwordx2", "buffer_store_dwordx2"} <= set(access)
    assert set(access) <= {f"buffer_{a}_dword{w}" for a in ("load", "store") for w in ("", "x2")}

"""Machine code of the staged projections, compiled here without a GPU: their slab
loads take their buffer resource from scalar registers.  One formed in vector
registers puts every load into a loop over the wave's distinct resources (two 64-bit
compares each), 16 % of a pass of LiH in mixed precision."""
import os
import re
import subprocess

import pytest

from sqdft_amd import build as B

SRC = """#include "sq_kernels.hpp"
template __global__ void sqk::k_projs<float, 4, 1, 4, 512, 3>(sqk::PArgs<float>);
template __global__ void sqk::k_projs<float, 4, 0, 4, 512, 3>(sqk::PArgs<float>);
template __global__ void sqk::k_projs<double, 1, 1, 1, 512, 1>(sqk::PArgs<double>);
"""


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="needs hipcc")
def test_slab_loads_use_scalar_resources(tmp_path):
    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(SRC)
    subprocess.run([B.HIPCC, *B.HIP_FLAGS, "--cuda-device-only", "-S", "-c", str(src), "-o", str(out)], check=True,
                   capture_output=True)
    text = out.read_text()
    kernels = re.findall(r"^(_ZN3sqk7k_projs\w+):(.*?)s_endpgm", text, re.S | re.M)
    assert len(kernels) == 3
    for name, body in kernels:
        assert body.count("buffer_load") >= 20, name
        assert "v_cmp_eq_u64" not in body, name

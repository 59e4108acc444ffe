"""What the kernels rely on and the compiler might change, read off the
assembly that it makes of them."""
import re
import subprocess

import pytest

from prismkv_amd import build


def test_four_word_stores_have_no_scalar_offset(tmp_path):
    # such a store lost its last word to the next vector instruction (update.hip, encode_kernel)
    hipcc = build._hipcc("/opt/rocm")
    try:
        subprocess.run([hipcc, "--version"], capture_output=True, check=True)
    except OSError:
        pytest.skip("no hipcc")
    out = tmp_path / "update.s"
    subprocess.run([hipcc, *build.HIP_FLAGS, f"-I{build.CSRC}", f"-I{build.INCLUDE}", "--cuda-device-only", "-S",
                    str(build.CSRC / "update.hip"), "-o", str(out)], check=True, capture_output=True)
    stores = re.findall(r"buffer_store_dwordx4 [^;\n]*", out.read_text())
    # four columns of a step, in two loops of two key types, where activations are stored
    assert len(stores) >= 16
    for store in stores:
        assert re.fullmatch(r"buffer_store_dwordx4 v\[\d+:\d+\], v\d+, s\[\d+:\d+\], 0 offen( offset:\d+)?\s*", store), store

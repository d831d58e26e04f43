"""Properties of the compiled kernels that their results on a GPU do not show, read from the assembly
hipcc writes for them (no GPU needed)."""
import os
import re
import shutil
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ml-framework_amd")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def kernels(source, *flags):
    """{kernel symbol: its assembly} of a source, built with the Makefile's device flags and `flags`."""
    cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", f"-I{PKG}/../include", f"-I{PKG}/csrc", *flags, "--cuda-device-only", "-S", "-o", "-",
           os.path.join(PKG, "csrc", source)]
    text = subprocess.run(cmd, check=True, stdout=subprocess.PIPE, stderr=subprocess.DEVNULL, text=True).stdout
    return {m[1]: m[2] for m in re.finditer(r"^(_Z\w+):(.*?)^\.Lfunc_end", text, flags=re.M | re.S)}


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_short_row_decode_uses_no_null_tile():
    """The short-row decode stages no V tile for the appended token: nothing is written through the null
    pointer that stands for one. Built with the option that keeps accesses through null, which the optimiser
    drops otherwise; they have no known address space, hence the flat form, and the kernel has no other."""
    rows = {k: v for k, v in kernels("decode_mfma_d64.hip", "-fno-delete-null-pointer-checks").items()
            if "paged_decode_mfma_row_kernel" in k}
    assert len(rows) == 6
    for name, text in rows.items():
        assert "s_endpgm" in text
        assert re.findall(r"^\s*flat_\w+.*$", text, flags=re.M) == [], name

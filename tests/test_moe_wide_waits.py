"""The wide expert kernel's products stand in inline assembly, for which the compiler sets no waits: in the assembly of every instance the sums' registers
are neither written between the opening wait and the first product nor touched between the last product and the closing wait."""

import re
import subprocess

from paged_llm_amd.csrc import build


def test_waits_stand_between_the_products_and_every_other_access(tmp_path):
    out = tmp_path / "moe_wide.s"
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([build._hipcc(), *flags, "--cuda-device-only", "-S", f"{build.CSRC}/moe_wide.hip", "-o", str(out)], check=True, capture_output=True, cwd=tmp_path)
    kernels = re.findall(r"^_Z\w*moe_wide_kernel(\w+):(.*?)^\.Lfunc_end", out.read_text(), re.S | re.M)
    assert len(kernels) == 30
    for name, body in kernels:
        lines = [line.split(";")[0].strip() for line in body.split("\n")]
        products = [i for i, line in enumerate(lines) if line.startswith("v_mfma")]
        waits = [i for i, line in enumerate(lines) if line == "s_nop 15"]
        opening = max(i for i in waits if i < products[0])
        closing = [i for i in waits if i > products[-1]][1]                       # (two in a row)
        sums = re.compile(r"\ba(\d+|\[\d+:\d+\])")
        early = [line for line in lines[products[-1] + 1:closing] if sums.search(line)]
        late = [line for line in lines[opening:products[0]] if sums.search(line)]
        assert not early and not late, (name, early[:2], late[:2])

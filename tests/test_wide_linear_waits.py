"""The wide kernel's products stand in inline assembly, for which the compiler sets no waits: in the assembly of every instance the sums' registers
are neither written between the opening wait and the first product nor touched between the last product and the closing wait."""

import re
import subprocess

from paged_llm_amd.csrc import build


def test_waits_stand_between_the_products_and_every_other_access(tmp_path):
    out = tmp_path / "wide_linear.s"
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([build._hipcc(), *flags, "--cuda-device-only", "-S", f"{build.CSRC}/wide_linear.hip", "-o", str(out)], check=True, capture_output=True, cwd=tmp_path)
    kernels = re.findall(r"^_Z\w*wide_linear_kernel(\w+):(.*?)s_endpgm", out.read_text(), re.S | re.M)
    assert len(kernels) >= 25
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


def test_sums_of_the_large_tiles_are_the_products_alone(tmp_path):
    """The kernel with eight wavefronts: both of its loops' products, from the opening wait to the closing one, are all that names a register of a sum."""
    out = tmp_path / "wide_linear.s"
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([build._hipcc(), *flags, "--cuda-device-only", "-S", f"{build.CSRC}/wide_linear.hip", "-o", str(out)], check=True, capture_output=True, cwd=tmp_path)
    kernels = re.findall(r"^_Z\w*big_linear_kernel(\w+):(.*?)s_endpgm", out.read_text(), re.S | re.M)
    assert len(kernels) >= 16
    register = re.compile(r"\b([av])(?:(\d+)|\[(\d+):(\d+)\])")

    def registers(text):
        return {(kind, i) for kind, one, low, high in register.findall(text) for i in range(int(one or low), int(one or high) + 1)}
    for name, body in kernels:
        lines = [line.split(";")[0].strip() for line in body.split("\n")]
        waits = [i for i, line in enumerate(lines) if line == "s_nop 15"]
        products = [i for i, line in enumerate(lines) if line.startswith("v_mfma")]
        assert len(products) % 4 == 0
        loops = [products[:len(products) // 2], products[len(products) // 2:]]
        for loop in loops:
            assert not any(loop[0] < i < loop[-1] for i in waits), name
            sums = set().union(*(registers(lines[i].split(",")[0]) for i in loop))
            opening = max(i for i in waits if i < loop[0])
            end = next(i for i in range(loop[-1] + 1, len(lines)) if lines[i].startswith(("s_branch", "s_nop 15")))
            between = [lines[i] for i in range(opening, end) if i not in loop and registers(lines[i]) & sums]
            assert not between, (name, between[:3])
        assert waits[-2] > products[-1] and waits[-1] == waits[-2] + 1, name       # (two in a row, behind both loops)

"""Kernels that must not spill registers, by the resources that the compiler states for them (built here; no GPU)."""
import os
import re
import subprocess

from evoformer_triton_amd import build


def test_short_rows_at_head_dim_64_in_fp32_do_not_spill(tmp_path):
    """The kernels of up to 64 keys on the fp32 instruction: dK/dV with a bias spilled 29 registers where the bias was asked for a tile ahead."""
    out = str(tmp_path / "kernel.s")
    flags = next(u[2] for u in build._units() if u[0] == "f32")
    subprocess.check_call([build._hipcc(), *build.HIPCC_FLAGS, *flags, "-S", "--cuda-device-only", os.path.join(build.CSRC, "f32.hip"), "-o", out],
                          stderr=subprocess.DEVNULL)
    with open(out) as f:
        text = f.read()
    spills = dict(re.findall(r"\.symbol: +(\S+)\.kd.*?\.vgpr_spill_count: +(\d+)", text, re.S))
    short = {n: int(c) for n, c in spills.items() if re.search(r"f32_(fwd|dq|dkdv)ILi64ELi2E", n)}
    assert len(short) == 6 and not any(short.values()), short

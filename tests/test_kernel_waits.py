"""Waits that no result shows to be missing, read from the compiled kernels' own assembly (built here; no GPU)."""
import os
import re
import subprocess

import pytest

from evoformer_triton_amd import build


def _assembly(source, defines, tmp_path):
    out = str(tmp_path / "kernel.s")
    subprocess.check_call([build._hipcc(), *build.HIPCC_FLAGS, *defines, *build.VGPR_FORM, "-S", "--cuda-device-only",
                           os.path.join(build.CSRC, source), "-o", out], stderr=subprocess.DEVNULL)
    with open(out) as f:
        return f.read()


def _functions(text, name):
    """The body of every function whose mangled name contains `name`."""
    for m in re.finditer(r"^(_Z\w*%s\w*):[^\n]*\n(.*?)^\.Lfunc_end" % name, text, re.M | re.S):
        yield m.group(1), m.group(2).split("\n")


@pytest.mark.parametrize("head_dim", [32, 64, 128])
def test_a_split_forwards_fetch_follows_the_reads_of_its_buffer(head_dim, tmp_path):
    """A wave alternates between two buffers for V: the load path may write one again only when the wave's reads of it have
    returned.  Between the head of the loop and its first load into LDS there is a wait for all reads of LDS, wherever the
    compiler has put the products that use them."""
    text = _assembly("mfma_stream.hip", [f"-DEVO_D={head_dim}"], tmp_path)
    seen = 0
    for name, lines in _functions(text, "split_fwd"):
        head, waited, inside = None, False, False
        for line in lines:
            if re.match(r"\.LBB\w+:.*Inner Loop Header", line):
                head, waited, inside = line.split(":")[0], False, True
            elif re.match(r"\.LBB\w+:", line):
                inside = head is not None and "Header=" + head[2:] in line
            elif inside and re.search(r"s_waitcnt.*lgkmcnt\(0\)", line):
                waited = True
            elif inside and re.search(r"\bds_read", line):
                waited = False
            elif inside and re.search(r"buffer_load_dword\w* .*\blds\b", line):
                assert waited, (name, line)
                seen += 1
    assert seen >= 6      # two dtypes, three kinds of bias

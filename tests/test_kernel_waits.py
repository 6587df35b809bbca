"""Waits that no result shows to be missing, read from the compiled kernels' own assembly (built here; no GPU)."""
import os
import re
import shutil
import subprocess

import pytest

from evoformer_triton_amd import build


def _assembly(source, defines, tmp_path, csrc=build.CSRC):
    out = str(tmp_path / "kernel.s")
    flags = [x for x in build.HIPCC_FLAGS if x != "-I" + build.CSRC] + ["-I" + str(csrc)]
    subprocess.check_call([build._hipcc(), *flags, *defines, *build.VGPR_FORM, "-S", "--cuda-device-only",
                           os.path.join(csrc, source), "-o", out], stderr=subprocess.DEVNULL)
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


@pytest.mark.parametrize("head_dim", [8, 16, 32])
def test_a_mask_is_read_by_its_own_entries(head_dim, tmp_path):
    """The forward that reads a mask as given: by loads of an entry's size, of a resource that ends with the row, and none of the four bytes around an entry."""
    text = _assembly("mfma_fwd_ring.hip", [f"-DEVO_D={head_dim}"], tmp_path)
    seen = 0
    for name, lines in _functions(text, "mfma_fwd_ring"):
        size = int(re.search(r"ELi(\d)EEEv", name).group(1))
        loads = re.findall(r"^\s+((?:global|buffer)_load_(?:ubyte|ushort|dword))\b", "\n".join(lines), re.M)
        assert "global_load_dword" not in loads, name
        assert {x for x in loads if x.startswith("buffer")} == {0: set(), 1: {"buffer_load_ubyte"}, 2: {"buffer_load_ushort"}, 4: {"buffer_load_dword"}}[size], name
        seen += size != 0
    assert seen == 24      # two dtypes, bias or none, gate or none, three sizes of entry


def test_a_load_into_lds_declares_what_it_changes():
    """Written as an instruction that the compiler does not know, it sets m0 and writes LDS."""
    seen = 0
    for name in sorted(os.listdir(build.CSRC)):
        with open(os.path.join(build.CSRC, name)) as f:
            for statement in re.findall(r"asm volatile\((.*?)\);", f.read(), re.S):
                if "m0" in statement.split(":")[0]:
                    seen += 1
                    assert statement.rstrip().endswith(': "m0", "memory"'), (name, statement)
    assert seen >= 2


def test_no_wide_buffer_store_has_a_uniform_offset():
    """The compiler puts no wait state between such a store and the next write of its data, which the store may still be reading."""
    seen = 0
    for name in sorted(os.listdir(build.CSRC)):
        with open(os.path.join(build.CSRC, name)) as f:
            for line in f:
                if re.search(r"raw(_ptr)?_buffer_store_b(96|128)\(", line):
                    seen += 1
                    assert re.search(r", 0, 0\);\s*$", line), (name, line)
    assert seen >= 2


VMEM = re.compile(r"(buffer|global|flat|scratch)_(load|store|atomic)")


def _blocks(lines):
    """Basic blocks as (instructions, successors): by label, with whether an instruction was written by hand."""
    blocks, name, hand = {"entry": []}, "entry", False
    order = ["entry"]
    for line in lines:
        label = re.match(r"(\.LBB\w+):", line)
        s = line.strip()
        if label:
            name = label.group(1)
            blocks[name] = []
            order.append(name)
        elif s.startswith(";"):
            hand = "#ASMSTART" in s or (hand and "#ASMEND" not in s)
        elif s and not s.startswith("."):
            blocks[name].append((s.split(";")[0].strip(), hand))
            if s.startswith(("s_cbranch", "s_branch", "s_endpgm")):   # (what follows a branch is a block of its own)
                name = f"{order[-1]}+"
                blocks[name] = []
                order.append(name)
    following = {}
    for i, b in enumerate(order):
        end = blocks[b][-1][0] if blocks[b] else ""
        following[b] = []
        if end.startswith(("s_cbranch", "s_branch")):
            following[b].append(end.split()[1])
        if not end.startswith(("s_branch", "s_endpgm")) and i + 1 < len(order):
            following[b].append(order[i + 1])
    return blocks, following


def _after(instructions, younger, check=None):
    """`younger`: the fewest memory instructions that may have been issued since the last load into LDS that may be under way; None where none is."""
    for s, hand in instructions:
        wait = re.match(r"s_waitcnt\b.*vmcnt\((\d+)\)", s)
        if wait:
            if younger is not None and int(wait.group(1)) <= younger:
                younger = None
            if hand and check is not None:
                check(s, younger)
        elif VMEM.match(s):
            younger = 0 if s.endswith(" lds") else younger if younger is None else min(younger + 1, 64)
    return younger


@pytest.mark.parametrize("source", ["mfma_bwd_fused.hip", "mfma_bwd_fused8.hip"])
def test_a_stage_is_there_when_it_is_prepared(source, tmp_path):
    """The kernels that form dQ, dK and dV at once wait for all but so many of the youngest loads before they read what they had loaded into LDS: on every way
    through the kernel at least as many have been issued since."""
    text = _assembly(source, [], tmp_path)
    assert not re.search(r"buffer_store_dwordx[34] .*, s\d+ offen", text)   # (see the test above)
    # two dtypes, three kinds of bias, three widths or more, the first stage and the others
    assert _waits_behind_loads(text, "bwd_fused") >= 36


def _waits_behind_loads(text, kernels):
    """How many waits written by hand the kernels have; each finds every load into LDS done, on every way to it."""
    seen = 0
    for name, lines in _functions(text, kernels):
        blocks, following = _blocks(lines)
        into = {"entry": None}
        todo = ["entry"]
        while todo:
            b = todo.pop()
            out = _after(blocks[b], into[b])
            for f in following[b]:
                new = out if f not in into else into[f] if out is None else out if into[f] is None else min(out, into[f])
                if f not in into or new != into[f]:
                    into[f] = new
                    todo.append(f)

        def check(s, younger):
            nonlocal seen
            seen += 1
            assert younger is None, (name, s, younger)

        for b in blocks:
            if b in into:
                _after(blocks[b], into[b], check)
    return seen


# What holds in every stage but a row's last, for a wave with 32 queries: the stage has a second tile, whose rows of the bias are whole, and all of dBias is stored
WHOLE_STAGES = {
    "mfma_stream.hip": [("const bool active = q0 < p.N;", "const bool active = true;", 4), ("const bool active = key0 < p.N;", "const bool active = true;", 1),
                        ("            if (2 * s + 1 < NT) {\n                init = bias.take(ct[AHEAD - 1]);", "            if (true) {\n                init = bias.take(ct[AHEAD - 1]);", 1),
                        ("if (2 * s + 1 < NT) tile(", "if (true) tile(", 2),
                        ("                if (2 * s + 1 < NT) {\n                    const f32x16 b1 = bias.take(ct);", "                if (true) {\n                    const f32x16 b1 = bias.take(ct);", 1),
                        ("if (qt + 1 < NT) tile(", "if (true) tile(", 2),
                        ("if (q0 + r >= p.N) continue;", "", 1), ("if (col + 4 <= p.N) {", "if (true) {", 1), ("if (q0 + li >= p.N) return;\n#pragma unroll\n        for (int rr", "#pragma unroll\n        for (int rr", 1),
                        ("if ((ds_vec || ds_f32) && kg + 4 <= p.N) {", "if (ds_vec || ds_f32) {", 1), ("if (kg + i < p.N) {", "{", 1)],
    "stream_common.h": [("if (BT == 5 && !COLS && t * 32 + 32 > N) {", "if (false) {", 1)],
}


def test_a_stage_is_there_when_it_is_computed_on(tmp_path):
    """The kernels at head dim 64 that wait for all but the eight youngest loads and stores between stages: on every way from one stage to the next, at least eight are
    younger than what the stage's rows were loaded into LDS by.  (On the kernel as it is for stages before the last: the ways to a last stage's end lead to no wait.)"""
    csrc = tmp_path / "csrc"
    shutil.copytree(build.CSRC, csrc)
    for source, changes in WHOLE_STAGES.items():
        text = (csrc / source).read_text()
        for old, new, times in changes:
            assert text.count(old) == times, (source, old)
            text = text.replace(old, new)
        (csrc / source).write_text(text)
    text = _assembly("mfma_stream.hip", ["-DEVO_D=64"], tmp_path, csrc)
    seen = sum(_waits_behind_loads(text, k) for k in ("stream_fwd", "stream_dq", "stream_dkdv", "stream_bwd_one"))
    assert seen >= 100 and text.count("s_waitcnt vmcnt(8)") >= 10, seen

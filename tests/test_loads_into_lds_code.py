"""What the loads into LDS that are written in assembly (csrc/common.h, ia_load_to_lds) ask of the kernels that use them, read from the
assembly that the compiler makes of these kernels: it knows nothing of such a load, so nobody but the kernel waits for it."""
import os
import re
import subprocess

import pytest

from infernum_amd.csrc import build

LIBRARIES = {"gemm_mfma.hip": "core", "attention_mfma.hip, 128": "attn_d128", "attention_mfma.hip, 256": "attn_d256"}


@pytest.fixture(scope="module", params=list(LIBRARIES))
def kernels(request, tmp_path_factory):
    """Name -> text of the kernels of a source that hold such a load."""
    hipcc = build.find_hipcc()
    if hipcc is None:
        pytest.skip("no hipcc here")
    source, name = request.param.split(",")[0], LIBRARIES[request.param]
    out = str(tmp_path_factory.mktemp("asm") / "out.s")
    flags = [f for f in build.HIPCC_FLAGS + build.library_plan(name)["defines"] if f != "-fPIC"]
    subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", "-o", out, os.path.join(build.CSRC_DIR, source)], check=True, timeout=600,
                   capture_output=True)
    with open(out) as f:
        bodies = re.findall(r"^(_Z\w+):(.*?)\.end_amdhsa_kernel", f.read(), re.S | re.M)
    found = {kernel: body for kernel, body in bodies if "global_load_lds" in body}
    assert len(found) >= 4
    return found


def _blocks(body):
    """label -> (instructions, labels that it can go on to), in the order of the text; the first is the kernel's start."""
    parts = re.split(r"^(\.LBB\d+_\d+):.*$", body, flags=re.M)
    labels, texts = ["start", *parts[1::2]], parts[0::2]
    blocks = {}
    for i, (label, text) in enumerate(zip(labels, texts)):
        code, after, open_end = [], [], True
        for line in text.split("\n"):
            line = line.split(";")[0].strip()
            if not re.match(r"[a-z]\w+", line):
                continue
            code.append(line)
            op, _, arg = line.partition(" ")
            if op == "s_branch" or op.startswith("s_cbranch"):
                after.append((len(code), arg.strip()))
            if op in ("s_branch", "s_endpgm"):
                open_end = False
                break
        if open_end and i + 1 < len(labels):
            after.append((len(code), labels[i + 1]))
        blocks[label] = (code, after)
    return blocks


def test_no_load_is_under_way_where_a_kernel_ends(kernels):
    for name, body in kernels.items():
        blocks = _blocks(body)
        under_way = {"start": False}
        work, ends = ["start"], 0
        while work:
            label = work.pop()
            state = under_way[label]
            code, after = blocks[label]
            for i, line in enumerate(code):
                for at, to in after:
                    if at == i and (to not in under_way or state and not under_way[to]):
                        under_way[to] = state
                        work.append(to)
                if line.startswith("global_load_lds"):
                    state = True
                elif line.startswith("s_waitcnt") and re.search(r"vmcnt\(0\)", line):
                    state = False
                elif line.startswith("s_endpgm"):
                    ends += 1
                    assert not state, (name, label)
            for at, to in after:
                if at == len(code) and (to not in under_way or state and not under_way[to]):
                    under_way[to] = state
                    work.append(to)
        assert ends, name

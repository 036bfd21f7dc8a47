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


def test_nothing_else_of_such_a_kernel_uses_m0(kernels):
    for name, body in kernels.items():
        written_out = False
        for line in body.split("\n"):
            if "#ASMSTART" in line or "#ASMEND" in line:
                written_out = "#ASMSTART" in line
            code = line.split(";")[0]
            assert written_out or not re.search(r"\bm0\b|_lds_dword|movrel|gpr_idx|sendmsg|ds_gws", code), (name, line)


def _scalars(text):
    """s7 or s[8:9] -> the registers' numbers."""
    one, span = re.fullmatch(r"s(\d+)", text), re.fullmatch(r"s\[(\d+):(\d+)\]", text)
    return {int(one.group(1))} if one else set(range(int(span.group(1)), int(span.group(2)) + 1)) if span else set()


def test_a_scalar_address_does_not_come_from_a_vector_instruction_just_before(kernels):
    """Five wait states between a vector instruction's write of a scalar register and a load that takes its address from it."""
    for name, body in kernels.items():
        blocks = _blocks(body)
        before = {label: [] for label in blocks}
        for label, (_, after) in blocks.items():
            for at, to in after:
                before[to].append((label, at))

        def look(label, at, distance, wanted, seen):
            code = blocks[label][0]
            for line in reversed(code[:at]):
                if distance >= 5:
                    return
                op, _, args = line.partition(" ")
                if op.startswith("v_") and _scalars(args.split(",")[0].strip()) & wanted:
                    raise AssertionError((name, label, line, wanted, distance))
                nop = re.fullmatch(r"s_nop (\d+)", line)
                distance += int(nop.group(1)) + 1 if nop else 1
            for other, end in before[label]:
                if distance < 5 and (other, distance) not in seen:
                    seen.add((other, distance))
                    look(other, end, distance, wanted, seen)

        for label, (code, _) in blocks.items():
            for at, line in enumerate(code):
                if line.startswith("global_load_lds"):
                    base = line.split(",")[1].split()[0]
                    if base != "off":
                        look(label, at, 0, _scalars(base), set())

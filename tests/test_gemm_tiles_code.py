"""What csrc/gemm_tiles.hip promises its matrix instructions, which are written in assembly, read from the assembly that the compiler
makes of it: inside the loops their operands come from LDS and from nothing else, no accumulator is moved (the compiler keeps no distance
between such an instruction and one that it does not know), and nothing is spilled there."""
import os
import re
import subprocess

import pytest

from infernum_amd.csrc import build


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    hipcc = build.find_hipcc()
    if hipcc is None:
        pytest.skip("no hipcc here")
    out = str(tmp_path_factory.mktemp("asm") / "gemm_tiles.s")
    flags = [f for f in build.HIPCC_FLAGS if f != "-fPIC"]
    subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", "-o", out, os.path.join(build.CSRC_DIR, "gemm_tiles.hip")], check=True,
                   capture_output=True, timeout=600)
    with open(out) as f:
        return f.read()


def _registers(text):
    """v7 or v[8:11] -> the registers' numbers."""
    one = re.fullmatch(r"v(\d+)", text)
    if one:
        return {int(one.group(1))}
    span = re.fullmatch(r"v\[(\d+):(\d+)\]", text)
    return set(range(int(span.group(1)), int(span.group(2)) + 1)) if span else set()


def _instructions(text):
    return [(op, [x.strip() for x in args.split(",")]) for op, args in re.findall(r"^\s+([a-z]\w+) ?(.*?)$", text, re.M)]


def test_operands_of_the_loops_come_from_lds_alone(assembly):
    kernels = re.findall(r"^(_Z\w*gemm_tiles_kernel\w+):(.*?)\.end_amdhsa_kernel", assembly, re.S | re.M)
    assert len(kernels) >= 15
    for name, body in kernels:
        blocks = re.split(r"^(\.LBB\d+_\d+):", body, flags=re.M)
        loops = 0
        for label, part in zip(blocks[1::2], blocks[2::2]):
            if "v_mfma_f32_16x16x32_bf16" not in part:
                continue
            found = _instructions(part)
            matrix = [i for i, (op, _) in enumerate(found) if op == "v_mfma_f32_16x16x32_bf16"]
            again = any(op.startswith("s_cbranch") and args[0] == label for op, args in found)
            # a loop's body from its label to its branch, and once more from there: what its end leaves meets its beginning; the odd last
            # step, and what stands in front of it in its block, up to its last product
            found = found + found if again else found[:matrix[-1] + 1]
            loops += again
            wrote = {}                                  # register -> the instruction that wrote it last
            for op, args in found:
                if op == "v_mfma_f32_16x16x32_bf16":
                    assert args[0] == args[3] and args[0].startswith("a["), (name, args)
                    for r in _registers(args[1]) | _registers(args[2]):
                        assert wrote.get(r, "ds_read_b128") == "ds_read_b128", (name, label, r, wrote[r])
                elif op.startswith(("v_", "ds_read")):
                    assert "accvgpr" not in op, (name, label, op)
                    for r in _registers(args[0]):
                        wrote[r] = op
                else:
                    assert op.startswith(("s_", "buffer_load")) and "scratch" not in op, (name, label, op)
        assert loops >= 1 and sum("v_mfma" in p for p in blocks[2::2]) >= 2, name       # two steps a turn, and the odd last one


TILES = [(256, 256), (256, 224), (256, 192), (256, 160), (256, 128), (224, 256), (192, 256), (192, 192), (192, 128), (160, 256),
         (160, 192), (160, 128), (128, 256), (128, 192), (128, 128)]


def test_the_tiles_of_the_kernel_are_those_of_its_callers():
    from infernum_amd.kernels import api
    with open(os.path.join(build.CSRC_DIR, "gemm_tiles.hip")) as f:
        text = f.read()
    listed = re.findall(r"F\((\d+), (\d+), (\d), (\d), (\d), (\d)\)", text)
    assert [(int(a), int(b)) for a, b, *_ in listed] == TILES == list(api.GEMM_TILES)
    for bm, bn, *t in listed:
        x0, x1, w0, w1 = map(int, t)
        assert int(bm) == 32 * (x0 + x1) and int(bn) == 32 * (w0 + w1) and x0 >= x1 and w0 >= w1


def test_accumulators_are_read_behind_the_wait_for_the_last_products(assembly):
    for name, body in re.findall(r"^(_Z\w*gemm_tiles_kernel\w+):(.*?)\.end_amdhsa_kernel", assembly, re.S | re.M):
        lines = body.split("\n")
        last = 0
        for i, line in enumerate(lines):
            if "v_mfma" in line:
                last = i
            elif "v_accvgpr_read" in line:
                assert any("s_nop 15" in other for other in lines[last:i]), (name, line)

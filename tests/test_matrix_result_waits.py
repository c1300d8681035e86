"""The listing of the kernels with rings of slabs, as built: no result of a matrix instruction is read or overwritten by another kind of instruction before it is through, whichever way leads
there.  (The compiler puts the waits in, but with a way out between the two sets of sums of the loop it once left one out on the short path, and one number in six was wrong.)"""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from torchlet_amd.kernels import build

# wait states between a matrix instruction and another kind of instruction on its result: four passes, and eight in 32 bits
WAITS = {"v_mfma_f32_16x16x32_bf16": 7, "v_mfma_f32_16x16x4_f32": 10}


def _registers(operands):
    out = set()
    for m in re.finditer(r"\b([va])\[(\d+):(\d+)\]|\b([va])(\d+)\b", operands):
        out |= {(m[1], i) for i in range(int(m[2]), int(m[3]) + 1)} if m[1] else {(m[4], int(m[5]))}
    return out


def _functions(listing, wanted):
    name, body = None, []
    for line in listing.splitlines():
        head = re.match(r"^[0-9a-f]+ <(\S+)>:$", line)
        if head:
            if body:
                yield name, body
            name, body = (head[1] if wanted in head[1] else None), []
        elif name and "//" in line:
            text, _, code = line.partition("//")
            target = re.search(r"<\S+\+0x([0-9a-f]+)>", code)
            body.append((int(code.split(":")[0], 16), text.strip(), int(target[1], 16) if target else 0))
    if body:
        yield name, body


def early_uses(body):
    """Pairs (matrix instruction, instruction too close behind it) of a function's [(address, text, branch target behind its start)]."""
    first, at = body[0][0], {a: i for i, (a, _, _) in enumerate(body)}
    found = []
    for i, (_, text, _) in enumerate(body):
        if not text.startswith("v_mfma"):
            continue
        wait = WAITS[text.split(None, 1)[0]]
        result = _registers(text.split(None, 1)[1].split(",")[0])
        ways, best = [(i + 1, 0)], {}
        while ways:
            p, waited = ways.pop()
            if p >= len(body) or waited >= wait or best.get(p, wait) <= waited:
                continue
            best[p] = waited
            _, other, target = body[p]
            op, _, operands = other.partition(" ")
            if op.startswith("v_mfma"):
                if _registers(operands.split(",")[0]) & result:
                    continue                                    # (sums on: the hardware waits)
            elif op[:2] in ("v_", "ds", "gl", "bu", "fl", "sc") and _registers(operands) & result:
                found.append((text, other))
                continue
            if op == "s_endpgm":
                continue
            if op == "s_branch" or op.startswith("s_cbranch"):
                ways.append((at[first + target], waited + 1))
                if op == "s_branch":
                    continue
            ways.append((p + 1, waited + (int(operands, 0) + 1 if op == "s_nop" else 1)))
    return found


def test_the_check_sees_the_short_path():
    loop = [(0, "v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]", 0), (8, "s_cbranch_scc1 2", 28), (12, "s_nop 7", 0), (16, "v_accvgpr_read_b32 v8, a3", 0), (24, "s_endpgm", 0),
            (28, "s_nop 1", 0), (32, "v_accvgpr_read_b32 v9, a3", 0)]
    assert early_uses(loop) == [(loop[0][1], loop[6][1])]
    loop[5] = (28, "s_nop 5", 0)
    assert early_uses(loop) == []


def test_the_check_waits_longer_for_32_bit_products():
    line = [(0, "v_mfma_f32_16x16x4_f32 v[0:3], v8, v9, 0", 0), (8, "s_nop 6", 0), (12, "v_add_f32_e32 v4, v3, v4", 0), (16, "s_endpgm", 0)]
    assert early_uses(line) == [(line[0][1], line[2][1])]
    line[1] = (8, "s_nop 8", 0)
    assert early_uses(line) == [(line[0][1], line[2][1])]
    line[1] = (8, "s_nop 9", 0)
    assert early_uses(line) == []


# instances in bfloat16 and in 32 bits: of the latter up to 8 and up to 16 rows, six shapes of the plain product, five of the gate and five of the rotation
@pytest.mark.parametrize("library,kernel,instances", [("gemm", "gemm_ring_kernel", {"v_mfma_f32_16x16x32_bf16": 132, "v_mfma_f32_16x16x4_f32": 32}),
                                                      ("experts", "experts_ring_kernel", {"v_mfma_f32_16x16x32_bf16": 2})])
def test_results_are_through_before_they_are_read(library, kernel, instances, tmp_path):
    objdump = Path(build.hipcc()).resolve().parent.parent / "llvm/bin/llvm-objdump"
    if not objdump.exists():
        objdump = Path("/opt/rocm/llvm/bin/llvm-objdump")
    if not objdump.exists():
        pytest.skip("no llvm-objdump beside the compiler")
    shutil.copy(build.build(library, quiet=True), tmp_path / "lib.so")
    subprocess.run([objdump, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    code, = tmp_path.glob(f"*{build.ARCH}*")
    listing = subprocess.run([objdump, "-d", "--no-show-raw-insn", code], check=True, capture_output=True, text=True).stdout
    found, bad = dict.fromkeys(instances, 0), []
    for name, body in _functions(listing, kernel):
        for instruction in {text.split(None, 1)[0] for _, text, _ in body if text.startswith("v_mfma")}:
            found[instruction] += 1
        bad += [(name, *pair) for pair in early_uses(body)]
    assert not bad, bad[:4]
    assert all(found[instruction] >= least for instruction, least in instances.items()), found

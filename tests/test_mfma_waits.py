"""Wait states behind matrix instructions in the built gfx950 code (CPU only).

Nothing in the hardware holds up a vector instruction that touches an MFMA's
result too early: the compiler leaves instructions or s_nop between them.  It has
left too few before copies in a loop's header (settle in proj_gemm.hip), where
the sums came out wrong.  This walks every path from every MFMA and counts, one
wait state an instruction (a taken branch two, as the compiler does), up to the
first instruction other than an MFMA that touches a result register.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "glacier.tune_amd", "libglacier_attn.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

# what the compiler leaves in straight code: by passes (4, 8, 8, 16)
WAITS = {"v_mfma_f32_16x16x32_bf16": 8, "v_mfma_f32_16x16x4_f32": 10,
         "v_mfma_f32_32x32x16_bf16": 12, "v_mfma_f32_32x32x2_f32": 18}
VECTOR = ("v_", "ds_", "buffer_", "global_", "flat_", "scratch_")


def registers(text):
    out = set()
    for kind, lo, hi, one in re.findall(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)", text):
        out |= {(kind, i) for i in range(int(lo or one), int(hi or one) + 1)}
    return out


def functions(listing):
    """(name, [(address, mnemonic, operands, branch offset or None)]) of each function."""
    name, code = None, []
    for line in listing.splitlines():
        head = re.match(r"^[0-9a-f]+ <(.+)>:", line)
        if head:
            if code:
                yield name, code
            name, code = head[1], []
        ins = re.match(r"^\s+(\S+)\s*(.*?)\s*//\s*([0-9A-F]+):", line)
        if ins:
            target = re.search(r"<\S+\+0x([0-9a-f]+)>", line)
            code.append((int(ins[3], 16), ins[1], ins[2], int(target[1], 16) if target else None))
    if code:
        yield name, code


def short_waits(code):
    """[(MFMA, wait states, instruction)] closer than WAITS."""
    at = {address: i for i, (address, *_) in enumerate(code)}
    base, found = code[0][0], []
    for i, (_, op, args, _) in enumerate(code):
        if op not in WAITS:
            assert not op.startswith("v_mfma"), f"no wait states known for {op}"
            continue
        result = registers(args.split(", ")[0])
        seen, todo = {}, [(i + 1, 0)]
        while todo:
            j, waits = todo.pop()
            if j >= len(code) or waits >= WAITS[op] or seen.get(j, 99) <= waits:
                continue
            seen[j] = waits
            _, other, operands, target = code[j]
            if other.startswith("v_mfma"):
                if not registers(operands.split(", ")[0]) & result:  # else its own wait begins
                    todo.append((j + 1, waits + 1))
                continue
            if other.startswith(VECTOR) and registers(operands) & result:
                found.append((f"{op} {args}", waits, f"{other} {operands}"))
                continue
            if other in ("s_endpgm", "s_setpc_b64"):
                continue
            if target is not None:
                todo.append((at[base + target], waits + 2))
            if other != "s_branch":
                todo.append((j + 1, waits + (int(operands.split()[0], 0) + 1 if other == "s_nop" else 1)))
    return found


def test_a_short_wait_is_found():
    listing = """
0000000000001000 <kernel>:
\tv_mov_b32_e32 v9, v0                                       // 000000001000: 00000000
\tv_mfma_f32_32x32x16_bf16 v[0:15], v[20:23], v[24:27], v[0:15]// 000000001004: 00000000 00000000
\ts_nop 2                                                    // 00000000100C: 00000000
\ts_cbranch_scc1 65531                                       // 000000001010: 00000000 <kernel+0x0>
\ts_nop 15                                                   // 000000001014: 00000000
\tv_add_f32_e32 v30, v0, v1                                  // 000000001018: 00000000
\ts_endpgm                                                   // 00000000101C: 00000000
"""
    ((name, code),) = functions(listing)
    assert name == "kernel" and len(code) == 7
    ((_, waits, reader),) = short_waits(code)
    assert (waits, reader) == (5, "v_mov_b32_e32 v9, v0")


@pytest.mark.skipif(not (os.path.exists(LIB) and os.access(OBJDUMP, os.X_OK)),
                    reason="needs the built library and ROCm's llvm-objdump")
def test_built_kernels_wait_for_their_matrix_instructions(tmp_path):
    lib = tmp_path / "lib.so"
    shutil.copy(LIB, lib)  # the extractor writes next to its input
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp_path, check=True, capture_output=True,
                   timeout=120)
    kernels = 0
    for obj in sorted(tmp_path.glob("lib.so.*gfx950")):
        listing = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", str(obj)], check=True,
                                 capture_output=True, text=True, timeout=120).stdout
        for name, code in functions(listing):
            kernels += any(op in WAITS for _, op, _, _ in code)
            short = short_waits(code)
            assert not short, f"{name}: {short[:3]}"
    assert kernels > 50

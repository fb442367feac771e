"""Wait states around the matrix instructions of the built library.

Kernels that tie their accumulators to one register block write their matrix instructions as inline assembly, which the
compiler's hazard pass does not look into.  What it guarantees for the builtin forms on gfx950 has to hold there by the
kernels' own schedule, and is checked here on the code that was built: two wait states between a vector instruction that
writes a register and a matrix instruction that reads it, and the passes of a matrix instruction plus four (its result is
not interlocked) before a vector or memory instruction touches what it wrote."""
import concurrent.futures
import os
import re
import shutil
import subprocess

import pytest

LLVM_OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
LLVM_READELF = "/opt/rocm/llvm/bin/llvm-readelf"
WRITE_TO_MATRIX = 2
# wait states the compiler puts between the builtin and an ordinary reader of its result: 4, 8 and 16 passes
RESULT = {"16x16x32": 8, "16x16x128": 12, "32x32x16": 12, "32x32x64": 20}
REG = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])")
BRANCH = re.compile(r"<([^>+]+)(?:\+0x([0-9a-f]+))?>")
WRITES_TWO = ("v_swap_", "v_permlane32_swap", "v_permlane16_swap")


def _regs(operand):
    m = REG.search(operand)
    if not m:
        return ()
    if m.group(2):
        return ((m.group(1), int(m.group(2))),)
    return tuple((m.group(1), r) for r in range(int(m.group(3)), int(m.group(4)) + 1))


def hazards(lines):
    """(kernel, address, instruction, what is wrong) for each hazard in a disassembly."""
    found, kernel, start = [], "", 0
    code = []

    def finish():
        if not any(op.startswith("v_mfma") for _, op, _, _ in code):
            return
        # (address, registers -> wait states still to pass) along every fall-through, and once more over each branch
        at = {address: i for i, (address, _, _, _) in enumerate(code)}

        def walk(i, written, results, budget):
            """One straight line from instruction i on; at most `budget` wait states of it (None: to the end)."""
            while i < len(code):
                address, op, args, target = code[i]
                operands = args.split(", ")
                if op.startswith("v_mfma"):
                    reads = [r for o in operands[1:4] for r in _regs(o)]
                    if any(r in written for r in reads):
                        found.append((kernel, address, op + " " + args, "operand written too recently"))
                elif op.startswith(("v_", "ds_", "buffer_", "global_", "scratch_", "flat_")):
                    if results and any(r in results for o in operands for r in _regs(o)):
                        found.append((kernel, address, op + " " + args, "matrix result touched too early"))
                states = 1
                if op == "s_nop":
                    states = int(args.split()[0], 0) + 1
                for table in (written, results):
                    for r in [r for r, left in table.items() if left <= states]:
                        del table[r]
                    for r in table:
                        table[r] -= states
                if op.startswith("v_mfma"):
                    need = next(v for k, v in RESULT.items() if k + "_" in op)
                    results.update(dict.fromkeys(_regs(operands[0]), need))
                elif op.startswith("v_"):
                    for o in operands[:2 if op.startswith(WRITES_TWO) else 1]:
                        written.update(dict.fromkeys(_regs(o), WRITE_TO_MATRIX))
                if budget is not None:
                    budget -= states
                    if budget <= 0 or not (written or results):
                        return
                elif target is not None and target in at and (written or results):
                    walk(at[target], dict(written), dict(results), max(RESULT.values()))
                if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
                    if budget is not None:
                        return
                    written.clear(), results.clear()
                i += 1

        walk(0, {}, {}, None)

    for line in lines:
        if line.endswith(">:\n"):
            finish()
            address, name = line[:-3].split(" <")
            kernel, start, code = name, int(address, 16), []
            continue
        if not line.startswith("\t"):
            continue
        text, _, comment = line.partition("//")
        op, _, args = text.strip().partition(" ")
        target = None
        if op.startswith(("s_cbranch", "s_branch")):
            m = BRANCH.search(comment)
            target = start + int(m.group(2) or "0", 16) if m else None
        code.append((int(comment.split(":")[0], 16) if comment else -1, op, args.strip(), target))
    finish()
    return found


@pytest.mark.parametrize("body,count", [
    ("v_perm_b32 v7, v0, v1, s2;v_mfma_f32_32x32x64_f8f6f4 v[16:31], v[0:7], v[8:15], v[16:31]", 1),
    ("v_perm_b32 v7, v0, v1, s2;s_waitcnt lgkmcnt(0);v_mfma_f32_32x32x64_f8f6f4 v[16:31], v[0:7], v[8:15], v[16:31]", 1),
    ("v_perm_b32 v7, v0, v1, s2;s_nop 1;v_mfma_f32_32x32x64_f8f6f4 v[16:31], v[0:7], v[8:15], v[16:31]", 0),
    ("v_mov_b32_e32 v16, 0;v_mfma_f32_16x16x32_bf16 a[16:19], v[0:3], v[8:11], a[16:19]", 0),
    ("v_accvgpr_write_b32 a17, 0;v_mfma_f32_16x16x32_bf16 a[16:19], v[0:3], v[8:11], a[16:19]", 1),
    ("v_mfma_f32_16x16x32_f16 a[16:19], v[0:3], v[8:11], 0;s_nop 6;v_accvgpr_read_b32 v0, a19", 1),
    ("v_mfma_f32_16x16x32_f16 a[16:19], v[0:3], v[8:11], 0;s_nop 7;v_accvgpr_read_b32 v0, a19", 0),
    ("v_mfma_f32_32x32x64_f8f6f4 v[16:31], v[0:7], v[8:15], 0;s_nop 15;s_nop 2;ds_write_b32 v0, v20", 1),
    ("v_permlane32_swap_b32_e32 v40, v3;s_nop 0;v_mfma_f32_16x16x32_f16 a[16:19], v[0:3], v[8:11], 0", 1),
])
def test_the_scan_sees_a_hazard(body, count):
    lines = ["0000000000000000 <k>:\n"] + ["\t%s // %012X: 0\n" % (s, 4 * i) for i, s in enumerate(body.split(";"))]
    assert len(hazards(lines)) == count


def test_the_scan_follows_a_branch():
    lines = ["0000000000000100 <k>:\n", "\tv_mfma_f32_16x16x32_f16 a[0:3], v[0:3], v[8:11], 0 // 000000000100: 0\n",
             "\ts_nop 7 // 000000000108: 0\n", "\tv_mov_b32_e32 v3, 0 // 00000000010C: 0\n",
             "\ts_cbranch_scc1 65531 // 000000000110: 0 <k>\n", "\ts_endpgm // 000000000114: 0\n"]
    assert [h[1] for h in hazards(lines)] == [0x100]


def _hazards_of(part):
    with subprocess.Popen([LLVM_OBJDUMP, "-d", str(part)], stdout=subprocess.PIPE, text=True) as dump:
        found = hazards(dump.stdout)
    assert dump.returncode == 0
    return found


@pytest.fixture(scope="module")
def device_code(pkg, tmp_path_factory):
    if not os.path.exists(LLVM_OBJDUMP):
        pytest.skip("no disassembler")
    folder = tmp_path_factory.mktemp("code")
    shutil.copy(pkg.lib_path(), folder / "lib.so")
    subprocess.run([LLVM_OBJDUMP, "--offloading", "lib.so"], cwd=folder, check=True, stdout=subprocess.DEVNULL)
    parts = sorted(folder.glob("*gfx950*"))
    assert parts, "no device code in %s" % pkg.lib_path()
    return parts


def test_w4a8_persistent_loops_keep_their_registers(device_code):
    """No scratch memory in the persistent W4A8 forms: a reload in the loop waits for every request in flight."""
    seen = {}
    for part in device_code:
        notes = subprocess.run([LLVM_READELF, "--notes", str(part)], check=True, stdout=subprocess.PIPE, text=True).stdout
        for name, scratch in re.findall(r"\.name:\s+(\S+).*?\.private_segment_fixed_size:\s+(\d+)", notes, re.S):
            if re.match(r"_ZN3woq16gemm_w4a8_kernelILi1ELb[01]ELi16ELb0ELi[12]E", name):
                seen[name] = int(scratch)
    assert len(seen) == 4 and not any(seen.values()), seen


def test_built_kernels_keep_the_wait_states(pkg, device_code):
    parts = device_code
    with concurrent.futures.ProcessPoolExecutor(4) as pool:
        found = sum(pool.map(_hazards_of, parts), [])
    assert not found, "%d hazards, the first: %s" % (len(found), found[:8])

"""The recurrent passes (csrc/seq_stack.hip) multiply with a lane-broadcast operand in asm statements, whose wait states the compiler does not look after: an operand that
goes through lane controls (DPP, permlane swaps) must have been written two wait states before it is read. Read off the device assembly of the source, built here.

The passes of wide MLPs (csrc/sac_wide.hip) exchange registers between lanes in such statements, next to matrix instructions. For every instruction with a lane control in the built library, whoever wrote it:
two wait states behind what writes its controlled operand, two before a matrix instruction that reads its result, and two more than a matrix instruction has passes behind one that writes a register which
it reads or writes."""
import collections
import os
import re
import struct
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOOLS = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


def _registers(operand):
    span = re.match(r"v\[(\d+):(\d+)\]$", operand)
    if span:
        return set(range(int(span[1]), int(span[2]) + 1))
    one = re.match(r"v(\d+)$", operand)
    return {int(one[1])} if one else set()


def _operands(line):
    parts = line.split(None, 1)
    return [_registers(o.strip().split()[0]) for o in parts[1].split(",")] if len(parts) == 2 else []


def violations(assembly):
    """[(distance, writer, reader)]; labels are passed over as if control fell through (a loop's first instructions are waits)"""
    code = [line.split(";")[0].strip() for line in assembly.splitlines()]
    code = [line for line in code if re.match(r"(v|s|ds|global|flat|buffer|scratch)_", line)]
    found, readers = [], 0
    for i, line in enumerate(code):
        name = line.split()[0]
        swap = "permlane" in name and "swap" in name
        if not swap and not ("row_newbcast" in line):
            continue
        readers += 1
        ops = _operands(line)
        read = ops[0] | ops[1] if swap else ops[1]
        states, j = 0, i - 1
        while states < 2 and j >= 0:
            before = code[j]
            if before.startswith("s_nop"):
                states += int(before.split()[1], 0)
            elif before.startswith("v_"):
                written = _operands(before)
                if read & (written[0] | (written[1] if "permlane" in before and "swap" in before else set())):
                    found.append((states, before, line))
                    break
            states += 1
            j -= 1
    return found, readers


def test_the_check_sees_a_missing_wait():
    mul = "v_mul_f32_dpp v1, v2, v3 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
    assert violations("v_add_f32_e32 v2, v4, v5\n" + mul)[0] and violations("v_add_f32_e32 v2, v4, v5\nv_mov_b32_e32 v9, v8\n" + mul)[0]
    assert violations("v_permlane16_swap_b32_e32 v7, v2\ns_nop 0\n" + mul)[0] and violations(mul + "v_permlane32_swap_b32_e32 v1, v8\n")[0]
    assert not violations("v_add_f32_e32 v2, v4, v5\ns_nop 1\n" + mul)[0] and not violations("v_add_f32_e32 v4, v2, v5\n" + mul)[0]


def test_recurrent_passes_wait_before_lane_controls(tmp_path):
    out = tmp_path / "seq_stack.s"
    source = os.path.join(ROOT, "rl-tools_amd", "csrc", "seq_stack.hip")
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--cuda-device-only", "-S", source, "-o", str(out)], check=True, capture_output=True)
    found, readers = violations(out.read_text())
    assert readers > 1000 and not found, found[:5]


MATRIX = re.compile(r"v_mfma_\w+?_(4x4|16x16|32x32)x")
PASSES = {"4x4": 2, "16x16": 8, "32x32": 16}      # of the fp32 forms, the longest of each shape


def lane_control_violations(lines):
    """([(rule, states between, earlier, later)], instructions with a lane control): over any number of lines of device code, labels passed over as in violations()"""
    found = []
    before = collections.deque()      # (state at which it was issued, instruction, its name, its operands) of the vector instructions of the last eighteen wait states
    now = controlled = 0
    for line in lines:
        code = line.split("//")[0].split(";")[0].strip()
        name = code.split(" ", 1)[0]
        if name == "s_nop":
            now += int(code.split()[1], 0) + 1
            continue
        if not re.match(r"(v|s|ds|global|flat|buffer|scratch)_", name):
            continue
        if name.startswith("v_"):
            while before and now - before[0][0] > 18:
                before.popleft()
            dpp, matrix = name.endswith("_dpp"), MATRIX.match(name)
            if dpp or matrix:
                ops = _operands(code)
                controlled += dpp
                for issued, earlier, earlier_name, earlier_ops in before:
                    states = now - issued - 1
                    if dpp and MATRIX.match(earlier_name):
                        if states < PASSES[MATRIX.match(earlier_name)[1]] + 2 and earlier_ops[0] & set().union(*ops[:3]):
                            found.append(("matrix, lane control", states, earlier, code))
                    elif dpp and states < 2 and ops[1] & earlier_ops[0]:
                        found.append(("write, lane control", states, earlier, code))
                    elif matrix and earlier_name.endswith("_dpp") and states < 2 and earlier_ops[0] & set().union(*ops[1:4]):
                        found.append(("lane control, matrix", states, earlier, code))
            else:
                ops = _operands(code)
            if ops:
                before.append((now, code, name, ops if len(ops) > 3 else ops + [set()] * (4 - len(ops))))
        now += 1
    return found, controlled


def code_objects(library, scratch):
    """The gfx950 code objects of a built library, one after the other in a file: each translation unit's offload bundle is its magic, the number of entries, then offset, size and name of each."""
    bundles = scratch / "bundles"
    subprocess.run([os.path.join(TOOLS, "llvm-objcopy"), "--dump-section", f".hip_fatbin={bundles}", library, "/dev/null"], check=True)
    data = bundles.read_bytes()
    for bundle in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at = bundle.end() + 8
        for _ in range(struct.unpack_from("<Q", data, bundle.end())[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            target, at = data[at + 24:at + 24 + length], at + 24 + length
            if b"gfx950" in target:
                (scratch / "code").write_bytes(data[bundle.start() + offset:bundle.start() + offset + size])
                yield scratch / "code"


def disassembly(library, scratch):
    for code in code_objects(library, scratch):
        with subprocess.Popen([os.path.join(TOOLS, "llvm-objdump"), "-d", "--no-show-raw-insn", code], stdout=subprocess.PIPE, text=True) as dump:
            yield from dump.stdout
        assert dump.returncode == 0


def built_library():
    library = os.path.join(ROOT, "rl-tools_amd", "librlt_rocm.so")
    if not os.path.exists(library):
        subprocess.run([sys.executable, os.path.join(ROOT, "rl-tools_amd", "build.py")], check=True, capture_output=True)
    return library


def test_the_check_sees_what_the_rules_forbid():
    select = "v_cndmask_b32_dpp v1, v2, v3, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf bound_ctrl:1"
    product, narrow = "v_mfma_f32_16x16x4_f32 v[0:3], v8, v9, v[0:3]", "v_mfma_f32_4x4x1_16b_f32 v[0:3], v8, v9, v[0:3] cbsz:2 abid:1"
    rules = lambda *lines: [v[0] for v in lane_control_violations(lines)[0]]      # noqa: E731
    assert rules("v_add_f32_e32 v2, v4, v5", select) == rules("v_add_f32_e32 v2, v4, v5", "s_nop 0", select) == ["write, lane control"]
    assert rules("v_add_f32_e32 v2, v4, v5", "s_nop 1", select) == rules("v_add_f32_e32 v3, v4, v5", select) == []
    assert rules(product, "s_nop 8", select) == rules(narrow, "s_nop 2", select) == ["matrix, lane control"]
    assert rules(product, "s_nop 9", select) == rules(narrow, "s_nop 3", select) == rules("v_mfma_f32_16x16x4_f32 v[12:15], v1, v2, v[0:3]", select) == []
    for reader in ("v_mfma_f32_16x16x4_f32 v[4:7], v1, v9, v[4:7]", "v_mfma_f32_16x16x4_f32 v[4:7], v9, v1, 0", product):
        assert rules(select, "s_nop 0", reader) == ["lane control, matrix"] and rules(select, "s_nop 1", reader) == []


def test_lane_controls_of_the_built_library_keep_their_distances(tmp_path):
    found, controlled = lane_control_violations(disassembly(built_library(), tmp_path))
    assert controlled > 10000 and not found, (len(found), found[:5])

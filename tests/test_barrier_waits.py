"""Workgroup barriers that order LDS traffic (csrc/common.h, rlt_lds_barrier): no path may reach one with LDS operations of the wavefront outstanding. The compiler has been
seen to drop the fence's wait where a barrier opens a loop, so this reads the device assembly of kernels with such loops, built here, along its control flow."""
import concurrent.futures
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def unwaited_barriers(assembly):
    """([function that holds a barrier reachable with LDS operations outstanding], number of barriers)"""
    blocks, name, function = {}, None, None
    order = []
    for line in assembly.splitlines():
        code = line.split(";")[0].strip()
        label = re.match(r"(\S+):$", code)
        if label:
            if label[1].startswith("_Z"):
                function = label[1]
            name = label[1]
            blocks[name] = (function, [])
            order.append(name)
        elif name and re.match(r"[a-z]\w*(\s|$)", code) and function:
            blocks[name][1].append(code)
    following = dict(zip(order, order[1:]))
    pending = {k: False for k in blocks}      # LDS operations outstanding at a block's entry, on any path
    bad, todo = set(), list(order)
    while todo:
        block = todo.pop()
        state, falls, out = pending[block], True, []
        for code in blocks[block][1]:
            if code.startswith("ds_"):
                state = True
            elif code.startswith("s_waitcnt") and "lgkmcnt(0)" in code:
                state = False
            elif code == "s_barrier" and state:
                bad.add(blocks[block][0])
            elif code.startswith(("s_cbranch", "s_branch")):
                out.append((code.split()[1], state))
                falls = not code.startswith("s_branch")
            elif code.startswith(("s_endpgm", "s_setpc")):
                falls = False
            if not falls:
                break
        if falls and block in following:
            out.append((following[block], state))
        for to, value in out:
            if value and to in pending and not pending[to]:
                pending[to] = True
                todo.append(to)
    return sorted(bad), sum(code == "s_barrier" for _, lines in blocks.values() for code in lines)


def test_the_check_sees_a_wait_that_the_way_round_a_loop_lacks():
    loop = "_Zk:\n\tds_write_b32 v0, v1\n\ts_waitcnt lgkmcnt(0)\n.L1:\n%s\ts_barrier\n\tds_read_b32 v2, v3\n\ts_waitcnt lgkmcnt(0)\n\tds_write_b32 v0, v2\n\ts_cbranch_scc1 .L1\n\ts_endpgm\n"
    assert unwaited_barriers(loop % "") == (["_Zk"], 1) and unwaited_barriers(loop % "\ts_waitcnt lgkmcnt(0)\n") == ([], 1)


CSRC = os.path.join(ROOT, "rl-tools_amd", "csrc")
SOURCES = sorted(f for f in os.listdir(CSRC) if f.endswith(".hip") and "rlt_lds_barrier" in open(os.path.join(CSRC, f)).read())


@pytest.fixture(scope="module")
def assemblies(tmp_path_factory):
    """the device assembly of every source with such a barrier, compiled side by side"""
    folder = tmp_path_factory.mktemp("assembly")

    def assemble(source):
        out = folder / (source + ".s")
        subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "--cuda-device-only", "-S", os.path.join(CSRC, source), "-o", str(out)], check=True, capture_output=True)
        return out.read_text()

    with concurrent.futures.ThreadPoolExecutor(max_workers=6) as pool:
        return dict(zip(SOURCES, pool.map(assemble, SOURCES)))


def test_every_kernel_with_such_a_barrier_is_looked_at():
    assert {"gru.hip", "seq_stack.hip", "sac_wide.hip", "mlp_fused.hip", "mlp_small.hip", "mlp_row.hip", "gemm.hip"} <= set(SOURCES)


@pytest.mark.parametrize("source", SOURCES)
def test_barriers_wait_for_lds(assemblies, source):
    bad, barriers = unwaited_barriers(assemblies[source])
    assert barriers and not bad

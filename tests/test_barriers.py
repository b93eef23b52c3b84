"""Every path from a store to LDS to a workgroup barrier waits for the store.

__syncthreads() asks for that wait, and the compiler (ROCm 7.2) has left it out where the store is the last thing of a
loop whose header holds the barrier: the other wavefronts then read the old value now and then (a form of grid pass A
whose next work item was taken at the loop's end gridded images wrong by 4e-4; all 33 of its instances had the
barrier without the wait). So the assembly of the kernels is looked through, whatever form the loops have."""
import os
import re
import shlex
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "ddfacet_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"
READS = re.compile(r"ds_(read|bpermute|permute|swizzle|nop)")


def kernels(text):
    """(name, instructions, successors) of every function of an assembly file."""
    for m in re.finditer(r"\n(_Z\S+):\s*; @", text):
        labels, ins = {}, []
        for line in text[m.end():text.find(".Lfunc_end", m.end())].split("\n"):
            line = line.split(";")[0].strip()
            lab = re.match(r"^(\.\w+):", line)
            if lab:
                labels[lab.group(1)] = len(ins)
            elif line and not line.startswith(".") and not line.startswith("_"):
                ins.append(line)
        succ = []
        for k, line in enumerate(ins):
            op = line.split()[0]
            to = {"s_branch": lambda: [labels[line.split()[1]]], "s_endpgm": list, "s_setpc_b64": list}.get(op)
            to = to() if to else [k + 1] + ([labels[line.split()[1]]] if op.startswith("s_cbranch") else [])
            succ.append([x for x in to if x < len(ins)])
        yield m.group(1), ins, succ


def unwaited(ins, succ):
    """Barriers that an LDS store can reach without s_waitcnt lgkmcnt(0), with the number of barriers."""
    barriers = [k for k, x in enumerate(ins) if x.startswith("s_barrier")]
    if not barriers:
        return [], 0
    pending, work = {0: False}, [0]
    while work:
        k = work.pop()
        p = pending[k]
        if ins[k].startswith("ds_") and not READS.match(ins[k]):
            p = True
        elif ins[k].startswith("s_waitcnt") and "lgkmcnt(0)" in ins[k]:
            p = False
        for x in succ[k]:
            if x not in pending or (p and not pending[x]):
                pending[x] = p
                work.append(x)
    return [k for k in barriers if pending.get(k)], len(barriers)


def test_the_check_itself():
    text = """
_Zk:                ; @_Zk
	ds_write_b32 v0, v1
.LBB0_1:
	s_barrier
	ds_read_b32 v2, v0
	s_waitcnt lgkmcnt(0)
	s_cbranch_scc1 .LBB0_2
	ds_write_b32 v0, v1
	s_branch .LBB0_1
.LBB0_2:
	s_barrier
	s_endpgm
.Lfunc_end0:
"""
    (name, ins, succ), = kernels(text)
    assert unwaited(ins, succ) == ([1], 2)
    (name, ins, succ), = kernels(text.replace("	s_barrier\n	ds_read", "	s_waitcnt lgkmcnt(0)\n	s_barrier\n	ds_read"))
    assert unwaited(ins, succ) == ([], 2)


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_stores_to_lds_are_waited_for_at_barriers():
    # the build's own lines, to assembly
    plan = subprocess.run(["make", "-n", "-B", "-C", CSRC], check=True, capture_output=True, text=True).stdout
    lines = [shlex.split(x) for x in plan.split("\n") if "hipcc" in x and " -c " in x]
    assert len(lines) >= 7
    with tempfile.TemporaryDirectory() as d:
        def assemble(args):
            out = os.path.join(d, os.path.basename(args[-1]) + ".s")
            i = args.index("-c")
            assert args[i + 1] == "-o"
            subprocess.run(args[:i] + ["-S", "--offload-device-only", "-o", out, args[-1]], check=True, cwd=CSRC,
                           capture_output=True, timeout=900)
            with open(out) as f:
                return f.read()
        with ThreadPoolExecutor(4) as pool:
            texts = list(pool.map(assemble, lines))
    total, bad = 0, []
    for text in texts:
        for name, ins, succ in kernels(text):
            where, n = unwaited(ins, succ)
            total += n
            bad += [(name, k) for k in where]
    assert total > 500
    assert not bad

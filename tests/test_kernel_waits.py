"""The built kernels' waits around workgroup barriers, read from this build's own machine code.

A kernel that streams tiles into LDS by direct-to-LDS loads refills a stage after the barrier that
ends its reading. A wave's LDS reads must have returned by then, not only been issued: the refill of
another wave can otherwise land first. The compiler places the wait in front of a read's first use,
which may move below a barrier written in inline assembly, so the source alone does not show it."""
import glob
import os
import re
import shutil
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"
BUILD = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "worldattention_amd", "csrc", "_build")
OBJECTS = sorted(glob.glob(os.path.join(BUILD, "*.o")))


def _kernels(obj, tmp):
    """{kernel: [(address, instruction)]} of an object's gfx950 code."""
    fat, code = os.path.join(tmp, "fat"), os.path.join(tmp, "code")
    sections = subprocess.run([f"{LLVM}/llvm-objdump", "-h", obj], capture_output=True, text=True, check=True).stdout
    if ".hip_fatbin" not in sections:
        return {}
    subprocess.run([f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", obj, "/dev/null"], check=True)
    subprocess.run([f"{LLVM}/clang-offload-bundler", "--type=o", "--unbundle", f"--input={fat}", f"--output={code}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    if os.path.getsize(code) == 0:
        return {}
    text = subprocess.run([f"{LLVM}/llvm-objdump", "-d", code], capture_output=True, text=True, check=True).stdout
    out, cur = {}, None
    for line in text.splitlines():
        m = re.match(r"^[0-9a-f]+ <(.*)>:", line)
        if m:
            cur = out.setdefault(m.group(1), [])
        elif cur is not None and line.startswith("\t") and "//" in line:
            ins, rest = line.strip().split("//", 1)
            cur.append((int(rest.split(":")[0], 16), ins.strip()))
    return out


def _successors(ins, index, i):
    address, text = ins[i]
    op = text.split()[0]
    following = [i + 1] if i + 1 < len(ins) else []
    if op in ("s_endpgm", "s_setpc_b64"):
        return []
    if op == "s_branch" or op.startswith("s_cbranch"):
        words = int(text.split()[1])
        target = index.get(address + 4 + 4 * (words - 65536 if words >= 32768 else words))
        return ([] if op == "s_branch" else following) + ([] if target is None else [target])
    return following


def reads_in_flight_at_barriers(ins):
    """Barriers that some path reaches with an LDS read that was not waited for since it was issued."""
    index = {a: i for i, (a, _) in enumerate(ins)}
    state, work = {0: frozenset()}, [0]
    while work:
        i = work.pop()
        text, flying = ins[i][1], state[i]
        if text.startswith("s_waitcnt") and "lgkmcnt(0)" in text:
            flying = frozenset()
        elif text.startswith("ds_read"):
            flying = frozenset([i])
        for j in _successors(ins, index, i):
            if j not in state or not flying <= state[j]:
                state[j] = state.get(j, frozenset()) | flying
                work.append(j)
    return [(i, sorted(ins[r][1] for r in state[i])) for i, (_, t) in enumerate(ins) if t == "s_barrier" and state.get(i)]


def test_the_scan_sees_a_read_past_a_barrier_and_around_a_loop():
    read, use = (0, "ds_read_b128 v[0:3], v4"), (8, "s_waitcnt lgkmcnt(0)")
    assert not reads_in_flight_at_barriers([read, use, (12, "s_barrier"), (16, "s_endpgm")])
    assert reads_in_flight_at_barriers([read, (8, "s_waitcnt vmcnt(0)"), (12, "s_barrier"), (16, "s_endpgm")])
    loop = [(0, "s_barrier"), (4, "ds_read_b128 v[0:3], v4"), (12, "s_cbranch_scc1 65532"), (16, "s_endpgm")]
    assert [i for i, _ in reads_in_flight_at_barriers(loop)] == [0]


@pytest.mark.skipif(not OBJECTS or not shutil.which(f"{LLVM}/llvm-objdump"), reason="no build objects or no llvm-objdump here")
@pytest.mark.parametrize("obj", OBJECTS, ids=[os.path.basename(o) for o in OBJECTS])
def test_lds_reads_return_before_a_stage_is_refilled(obj, tmp_path):
    for name, ins in _kernels(obj, str(tmp_path)).items():
        if any(t.startswith("buffer_load") and " lds" in t for _, t in ins):
            assert not reads_in_flight_at_barriers(ins), name

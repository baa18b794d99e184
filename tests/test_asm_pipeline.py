"""The prefill GEMMs' load pipeline is inline asm: the compiler does not know that an asm
load's destination registers fill in later, so a copy or other use of them that it places
before the kernel's explicit `s_waitcnt vmcnt` reads stale values (no error, wrong output).
This compiles prefill.hip to gfx950 assembly (CPU only) and checks every grouped-GEMM kernel
along every path, taken branches and loops included: after a vector load, no instruction
touches its destination registers until an `s_waitcnt vmcnt(N)` with at least N vector memory
operations issued since the load on that path (vector memory completes in issue order, so that
wait covers it; of the paths to one place the one with the fewest operations decides).

Some paths of the assembly never run: a tile switch sooner than a tile's fewest stages, a store
loop with another number of passes.  The source marks those places with comments ("; path + NAME"
counts a pass, "; path NAME >= N" or "== N" states the count there and restarts it), and a path
that contradicts a stated count is not followed."""
import os
import re
import shutil
import subprocess
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
from tarfa_amd import build as B  # noqa: E402

LOAD = re.compile(r"^(global|buffer)_load_(dword\w*|ushort|ubyte|short|sbyte)\s+(v\[\d+:\d+\]|v\d+)")
REG = re.compile(r"v\[(\d+):(\d+)\]|\b(v\d+)\b")


def _regs(text):
    out = set()
    for a, b, c in REG.findall(text):
        if c:
            out.add(int(c[1:]))
        else:
            out |= set(range(int(a), int(b) + 1))
    return out


PATH = re.compile(r"; path (?:(\+) (\w+)|(\w+) (>=|==) (\d+))")


def _mask(regs):
    m = 0
    for r in regs:
        m |= 1 << r
    return m


def parse(lines, facts=True):
    """The body's instructions as (text, wait count, is a vector memory operation, VGPR mask, path
    marker) and every instruction's successors."""
    code, labels = [], {}
    for line in lines:
        mark = PATH.search(line) if facts else None
        if mark:
            code.append((line.strip(), None, False, 0, mark.groups()))
            continue
        l = line.split(";")[0].strip()
        if l.endswith(":"):
            labels[l[:-1]] = len(code)
        elif l and not l.startswith("."):
            op, _, ops = l.partition(" ")
            w = re.search(r"vmcnt\((\d+)\)", ops) if op == "s_waitcnt" else None
            vm = op.startswith(("global_", "buffer_", "flat_", "scratch_"))
            regs = 0 if op.startswith("s_") else _mask(_regs(ops))
            code.append((l, int(w.group(1)) if w else None, vm, regs, None))
    succ = []
    for i, (l, *_) in enumerate(code):
        op, _, ops = l.partition(" ")
        if op == "s_branch":
            succ.append([labels.get(ops.strip())])
        elif op.startswith("s_cbranch"):
            succ.append([i + 1, labels.get(ops.strip())])
        elif op.startswith(("s_endpgm", "s_setpc")):
            succ.append([])
        else:
            succ.append([i + 1])
    return code, [[j for j in s if j is not None and j < len(code)] for s in succ]


def early_uses(lines, facts=True):
    """(load, first instruction touching its destination before a covering wait) pairs, over every path
    that agrees with the stated path facts (all paths without them)."""
    code, succ = parse(lines, facts)
    names = sorted({m[1] or m[2] for *_, m in code if m})
    cap = {n: max([int(m[4]) for *_, m in code if m and m[2] == n], default=0) + 1 for n in names}

    def passed(j, counts):
        """The counts after instruction j, None where they contradict it."""
        m = code[j][4]
        if not m:
            return counts
        k = names.index(m[1] or m[2])
        c = counts[k]
        if m[0]:
            c = min(c + 1, cap[names[k]])
        elif c < int(m[4]) or (m[3] == "==" and c > int(m[4])):
            return None
        else:
            c = 0
        return counts[:k] + (c,) + counts[k + 1:]

    # Every (instruction, counts) that some path from the entry reaches.
    reach, work = set(), [(0, (0,) * len(names))]
    while work:
        state = work.pop()
        if state in reach:
            continue
        reach.add(state)
        after = passed(*state)
        if after is not None:
            work += [(j, after) for j in succ[state[0]]]
    starts = {}
    for j, counts in reach:
        if LOAD.match(code[j][0]) and "_lds" not in code[j][0]:
            starts.setdefault(j, []).append(counts)

    bad = {}
    for i, entries in sorted(starts.items()):
        dst = _mask(_regs(LOAD.match(code[i][0]).group(3)))
        fewest = {}                      # (instruction, counts) -> fewest operations issued since the load
        work = [(j, counts, 0) for counts in entries for j in succ[i]]
        while work:
            j, counts, issued = work.pop()
            while issued < fewest.get((j, counts), 1 << 30):
                fewest[j, counts] = issued
                text, wait, vm, regs, _ = code[j]
                if wait is not None and issued >= wait:
                    break
                if regs & dst:
                    bad.setdefault((i, j), (code[i][0], text))
                    break
                counts = passed(j, counts)
                if counts is None or not succ[j]:
                    break
                issued = min(issued + vm, 64)
                work += [(k, counts, issued) for k in succ[j][1:]]
                j = succ[j][0]
    return list(bad.values())


def test_checker_flags_a_copy_before_the_wait():
    load = "global_load_dwordx2 v[194:195], v154, s[76:77]"
    covered = [load, "global_load_dword v7, v1, s[0:1]", "s_waitcnt vmcnt(1)", "v_mov_b32_e32 v3, v194"]
    early = [load, "global_load_lds_dwordx4 v206, s[2:3]", "v_mov_b32_e32 v3, v194", "s_waitcnt vmcnt(0)"]
    short = [load, "global_load_dword v7, v1, s[0:1]", "s_waitcnt vmcnt(2)", "v_mov_b32_e32 v3, v195"]
    waw = ["global_load_dword v10, v1, s[0:1]", "v_mov_b32_e32 v10, 0", "s_waitcnt vmcnt(0)"]
    other = [load, "v_mov_b32_e32 v3, v196", "s_branch .LBB0_1", "v_mov_b32_e32 v3, v194",
             ".LBB0_1:", "s_endpgm"]
    assert early_uses(covered) == []
    assert early_uses(early) == [(load, early[2])]
    assert early_uses(short) == [(load, short[3])]     # the wait leaves this load outstanding
    assert early_uses(waw) == [(waw[0], waw[1])]
    assert early_uses(other) == []                     # past an unconditional branch: no path leads there


def test_walk_follows_branches_and_back_edges():
    load = "global_load_dwordx4 v[8:11], v1, s[0:1]"
    # A loop whose load is read one trip later; the wait at its head covers it, or does not.
    loop = [".LBB0_1:", "s_waitcnt vmcnt({})", "v_mov_b32_e32 v3, v8", load, "global_store_dword v1, v2, s[0:1]",
            "s_cbranch_scc1 .LBB0_1", "s_endpgm"]
    assert early_uses([l.format(1) for l in loop]) == []
    assert early_uses([l.format(2) for l in loop]) == [(load, loop[2])]
    # A copy that only a taken branch reaches, and one past an unconditional branch.
    taken = [load, "s_cbranch_vccnz .LBB0_2", "s_waitcnt vmcnt(0)", "s_endpgm", ".LBB0_2:", "s_branch .LBB0_3",
             ".LBB0_3:", "v_mov_b32_e32 v20, v9", "s_endpgm"]
    assert early_uses(taken) == [(load, taken[7])]
    # A load overwritten by its own next trip before it has landed.
    again = [".LBB0_1:", load, "s_cbranch_scc1 .LBB0_1", "s_waitcnt vmcnt(0)", "s_endpgm"]
    assert early_uses(again) == [(load, load)]


def test_walk_heeds_path_facts():
    load = "global_load_dword v8, v1, s[0:1]"
    # Two stores between the load and its wait: a fact about the loop's trips rules the one-trip path out.
    body = [load, ".LBB0_1:", "; path + store", "global_store_dword v1, v2, s[0:1]", "s_cbranch_scc1 .LBB0_1",
            "; path store == 2", "s_waitcnt vmcnt(2)", "v_mov_b32_e32 v3, v8", "s_endpgm"]
    assert early_uses(body) == []
    assert early_uses(body, facts=False) == [(load, body[7])]
    assert early_uses([l.replace("vmcnt(2)", "vmcnt(3)") for l in body]) == [(load, body[7])]
    # At least two trips: more of them only issue more.
    least = [l.replace("== 2", ">= 2") for l in body]
    assert early_uses(least) == []
    assert early_uses([l.replace("vmcnt(2)", "vmcnt(3)") for l in least]) == [(load, body[7])]


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    if not shutil.which(B.HIPCC) and not os.path.exists(B.HIPCC):
        pytest.skip("hipcc not installed")
    out = tmp_path_factory.mktemp("asm") / "prefill.s"
    r = subprocess.run([B.HIPCC, *B.CFLAGS, "--cuda-device-only", "-S", os.path.join(B.CSRC, "prefill.hip"),
                        "-o", str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return out.read_text()


def test_grouped_gemms_use_no_scratch(asm):
    """A spilled register is reloaded behind a vmcnt(0), which drains the stages in flight."""
    sizes = dict(re.findall(r"\.set (_ZN4tmoe\d+k_grouped_gemm\w*)\.private_seg_size, (\d+)", asm))
    assert any("gemm_w" in n for n in sizes), sizes
    assert not {n: s for n, s in sizes.items() if int(s)}


def test_grouped_gemm_pipeline_loads_untouched_before_a_wait(asm):
    names = re.findall(r"^(_ZN4tmoe\d+k_grouped_gemm\w*):", asm, re.M)
    for kernel in ("gemm_pI", "gemm_wI", "gemm_qI"):
        assert any(kernel in n for n in names), (kernel, names)
    problems = {}
    for n in names:
        i = asm.index(n + ":")
        body = asm[i:asm.index(".Lfunc_end", i)].splitlines()
        bad = early_uses(body)
        if bad:
            problems[n] = bad[:3]
        if "gemm_pI" in n:
            # A down tile of one cycle contradicts "cycle >= 2".  It does not gather: its row-index words
            # (dwords, fetched for the launches that do) may be read early, and are then not selected.
            for load, use in early_uses(body, facts=False):
                dst, written = _regs(LOAD.match(load).group(3)), use.partition(" ")[2].split(",")[0]
                if not load.startswith("global_load_dword ") or _regs(written) & dst:
                    problems.setdefault(n, []).append((load, use))
    assert not problems, problems

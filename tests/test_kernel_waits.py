"""The kernels that refill an LDS buffer behind a barrier, as compiled: at each of their barriers no LDS access of the
wave is in flight. Such a read is ordered before another wave's store to the same buffer by nothing else."""
import os
import re
import shlex
import shutil
import subprocess

import pytest

from conftest import ROOT

PKG = os.path.join(ROOT, "historic-htr-ocr_amd")


def _assembly(name, tmp_path):
    """the gfx950 assembly of csrc/<name>.hip, with the flags that the library is built with"""
    if not shutil.which("make"):
        pytest.skip("no make")
    plan = subprocess.run(["make", "-n", "-B", "-C", PKG], capture_output=True, text=True, check=True).stdout
    line = next(s for s in plan.splitlines() if f"csrc/{name}.hip " in s + " " and " -c " in s)
    cmd = shlex.split(line)
    if not shutil.which(cmd[0]):
        pytest.skip("no hipcc")
    out = tmp_path / f"{name}.s"
    cmd[cmd.index("-c")] = "-S"
    cmd[cmd.index("-o") + 1] = str(out)
    subprocess.run(cmd + ["--cuda-device-only"], check=True, capture_output=True)
    return out.read_text()


def _functions(text):
    """kernel name → its instructions and labels, in order"""
    body = None
    for s in text.splitlines():
        s = s.split(";")[0].strip()
        if m := re.match(r"(\w+):$", s):
            if m[1].startswith("_Z"):
                name, body = m[1], []
                continue
        if s.startswith(".Lfunc_end") and body is not None:
            yield name, body
            body = None
        elif body is not None and s and (s.endswith(":") or not s.startswith(".")):
            body.append(s)


def _pending_at_barriers(body, cap=64):
    """the largest number of LDS accesses that may be in flight at each barrier of the function: over all paths, an
    access adds one, a wait for lgkmcnt(n) leaves n at most (LDS accesses complete in order, and scalar loads, which
    share the counter, only make the wait stronger)"""
    at = {s[:-1]: i for i, s in enumerate(body) if s.endswith(":")}
    best, todo, barriers = {}, [(0, 0)], {}
    while todo:
        i, n = todo.pop()
        while i < len(body):
            if best.get(i, -1) >= n:
                break
            best[i] = n
            s = body[i]
            op = s.split()[0]
            if op == "s_waitcnt":
                if m := re.search(r"lgkmcnt\((\d+)\)", s):
                    n = min(n, int(m[1]))
                elif re.fullmatch(r"s_waitcnt (0|0x0)", s):
                    n = 0
            elif op == "s_barrier":
                barriers[i] = max(barriers.get(i, 0), n)
            elif op.startswith("ds_"):
                n = min(n + 1, cap)
            elif op == "s_branch":
                i = at[s.split()[1]]
                continue
            elif op.startswith("s_cbranch"):
                todo.append((at[s.split()[1]], n))
            elif op == "s_endpgm":
                break
            else:
                assert not op.startswith(("s_setpc", "s_swappc")), s  # no calls: every path is seen
            i += 1
    return barriers


def test_pending_accesses_are_counted_over_all_paths():
    body = """ds_read_b64 v0, v1
.L1:
ds_read_b64 v2, v1
s_waitcnt vmcnt(0) lgkmcnt(1)
s_cbranch_scc1 .L2
s_barrier
s_waitcnt lgkmcnt(0)
s_barrier
s_branch .L1
.L2:
ds_write_b64 v0, v1
s_barrier
s_endpgm""".splitlines()
    assert _pending_at_barriers(body) == {5: 1, 7: 0, 11: 2}


@pytest.mark.parametrize("source,kernels", [("attention", "k_attn_causal"), ("vision", "k_attn_vision"),
                                            ("gemm", "k_gemm_q8_0"), ("mfma_gemm", r"k_gemm_f16\w+Li64ELi2EE")])
def test_no_lds_access_in_flight_at_a_barrier(tmp_path, source, kernels):
    """(k_gemm_f16's tiles in a ring of four stages refill the buffer before the one that is read, and are not among these)"""
    seen = 0
    for name, body in _functions(_assembly(source, tmp_path)):
        if not re.search(kernels, name):
            continue
        at = _pending_at_barriers(body)
        seen += len(at)
        assert not any(at.values()), (name, sorted(at.items()))
    assert seen


def test_inline_assembly_names_the_m0_it_writes():
    """an asm statement that writes m0 lists it as clobbered: the compiler may hold a value of its own there"""
    seen = 0
    for path in sorted(os.listdir(os.path.join(PKG, "csrc"))):
        with open(os.path.join(PKG, "csrc", path)) as f:
            text = f.read()
        for stmt in re.findall(r"\basm(?:__)?\s*(?:volatile)?\s*\((.*?)\);", text, re.S):
            code, *operands = re.split(r'"\s*:', stmt, maxsplit=1)
            if re.search(r"\bm0\s*,", code):
                seen += 1
                assert operands and '"m0"' in operands[0].split(":")[-1], (path, stmt)
    assert seen

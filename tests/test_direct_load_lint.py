"""The waits of every unit whose loads are inline assembly, in the gfx950 code that
the build left (test_tile_kernel_wait_lint.py compiles the tile kernels for it):
between a load and the ``s_waitcnt vmcnt(n)`` that covers it, no instruction reads
or writes the load's destination registers.  Beside that the wait states that the
compiler does not keep for inline assembly, in every unit with direct-to-LDS loads,
and that no spilled register moves inside the loops over K.

``vmcnt`` completes in order, so "covered" is positional: a wait for ``n``
leaves the youngest ``n`` vector-memory operations outstanding.  The scan is
linear in file order, which is execution order for the straight-line loop
bodies these kernels are made of.  CPU only: hipcc cross-compiles.
"""
import os
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

import pytest

from mlx_amd import _build

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "mlx_amd" / "csrc"
UNITS = ("qmm_mfma.hip", "qmm_mfma_pairs.hip", "qmm_mfma_fp.hip", "qmm_mfma_experts.hip",
         "qq_mfma.hip", "qmm_own_bf16.hip", "qmm_own_f16.hip", "qmm_own_fp_bf16.hip",
         "qmm_own_fp_f16.hip", "qmm_own_experts_bf16.hip", "qmm_own_experts_f16.hip")
# direct-to-LDS loads as well, the other loads the compiler's
DMA_UNITS = ("qmm_slab.hip", "qmm_mid_bf16.hip", "qmm_mid_f16.hip")

_SREG = re.compile(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b")
_REG = re.compile(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b")


def _regs(text, kind=_REG):
    out = set()
    for m in kind.finditer(text):
        if m.group(1):
            out.update(range(int(m.group(1)), int(m.group(2)) + 1))
        else:
            out.add(int(m.group(3)))
    return out


def _sregs(text):
    return _regs(text, _SREG)


def lint(asm_text):
    """Returns (functions seen, loads tracked, list of violations)."""
    fn = None
    outstanding = []  # (destination registers, a reload) of the vector-memory ops in flight, oldest first
    functions = loads = 0
    problems = []
    for ln, line in enumerate(asm_text.splitlines(), 1):
        t = line.strip()
        if not t or t.startswith(";") or t.startswith("."):
            continue
        if re.match(r"^_Z\w+:", t):
            fn, outstanding = t.split(":")[0], []
            functions += 1
            continue
        t = t.split(";")[0].strip()
        if not t:
            continue
        op = t.split()[0]
        args = t[len(op):]
        if op == "s_waitcnt":
            m = re.search(r"vmcnt\((\d+)\)", t)
            if m:
                n = int(m.group(1))
                outstanding = outstanding[-n:] if n else []
            continue
        if op == "s_endpgm":
            outstanding = []
            continue
        # reloads of spilled registers are the compiler's own: it lets a later one fill registers
        # of an earlier one (they arrive in order) and puts the waits itself
        reload = op.startswith("scratch_load")
        live = set().union(*(r for r, own in outstanding if not (own and reload)))
        is_vmem = op.startswith(("global_", "buffer_", "flat_", "scratch_"))
        touched = _regs(args)
        if touched & live:
            problems.append(f"{fn} line {ln}: `{t}` touches in-flight v{sorted(touched & live)}")
        if is_vmem:
            if "load" in op and "lds" not in op:
                outstanding.append((_regs(args.split(",")[0]), reload))
                loads += 1
            else:
                outstanding.append((set(), False))  # stores and direct-to-LDS loads: counted, no registers
    return functions, loads, problems


def lint_hazards(asm_text):
    """Wait states that the compiler keeps by itself and does not keep for inline assembly:
    one between a write of M0 and a direct-to-LDS load, five between a vector instruction that
    writes a scalar register and a vector-memory instruction that reads it.  Every instruction
    is one wait state, ``s_nop n`` is n + 1.  Returns (direct-to-LDS loads, violations)."""
    fn, now, m0, written = None, 0, None, {}
    loads, problems = 0, []
    for line in asm_text.splitlines():
        t = line.split(";")[0].strip()
        if re.match(r"^_Z\w+:", t):
            fn, m0, written = t.split(":")[0], None, {}
            continue
        if not t or t.startswith(".") or t.endswith(":"):
            continue
        op = t.split()[0]
        args = t[len(op):]
        if op == "s_nop":
            now += int(args, 0) + 1
            continue
        if op.startswith(("global_", "buffer_", "flat_", "scratch_")):
            if "lds" in t:
                loads += 1
                if m0 is not None and now - m0 < 1:
                    problems.append(f"{fn}: `{t}` right behind the write of m0")
            for r in _sregs(args):
                if now - written.get(r, -5) < 5:
                    problems.append(f"{fn}: `{t}` reads s{r}, just written by a vector instruction")
        now += 1
        first = args.split(",")[0]
        if re.search(r"\bm0\b", first):
            m0 = now
        if op.startswith("v_"):
            for r in _sregs(first):
                written[r] = now
    return loads, problems


def spills_in_loops(listing):
    """``listing``: (address, instruction, branch target or None) of one function.  Instructions
    that move spilled registers inside an innermost loop with matrix instructions."""
    at = {address: i for i, (address, _, _) in enumerate(listing)}
    loops = [(at[target], i) for i, (_, _, target) in enumerate(listing)
             if target is not None and at.get(target, i + 1) <= i]
    with_mfma = [(a, b) for a, b in loops
                 if any(op.startswith("v_mfma") for _, op, _ in listing[a:b])]
    inner = [x for x in with_mfma
             if not any(y != x and x[0] <= y[0] and y[1] <= x[1] for y in with_mfma)]
    return inner, [op for a, b in inner for _, op, _ in listing[a:b] if op.startswith("scratch_")]


_LLVM = Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "llvm" / "bin"
_TARGET = "hipv4-amdgcn-amd-amdhsa--gfx950"


def _object(unit, into):
    """The unit's object as the build left it, or compiled here where that is older than a source."""
    built = Path(_build.OBJ_DIR) / (unit[:-4] + ".o")
    newest = max(f.stat().st_mtime for d in (CSRC, ROOT / "include") for f in d.iterdir())
    if built.exists() and built.stat().st_mtime > newest:
        return built
    fresh = into / built.name
    subprocess.run([_build.HIPCC, *_build.FLAGS, "-c", str(CSRC / unit), "-o", str(fresh)],
                   check=True, capture_output=True)
    return fresh


def _assembly(unit, into):
    """(text for the lints, {function: listing for spills_in_loops})"""
    bundle, device = into / (unit + ".fb"), into / (unit + ".dev")
    for cmd in (
            ["llvm-objcopy", "--dump-section", f".hip_fatbin={bundle}", _object(unit, into), "/dev/null"],
            ["clang-offload-bundler", "--unbundle", "--type=o", f"--targets={_TARGET}",
             f"--input={bundle}", f"--output={device}"]):
        subprocess.run([_LLVM / cmd[0], *map(str, cmd[1:])], check=True, capture_output=True)
    raw = subprocess.run([_LLVM / "llvm-objdump", "-d", "--no-show-raw-insn", str(device)],
                         check=True, capture_output=True, text=True).stdout
    text, functions, base = [], {}, 0
    for line in raw.splitlines():
        head = re.match(r"^([0-9a-f]+) <(_Z\w+)>:", line)
        if head:
            base = int(head.group(1), 16)
            text.append(head.group(2) + ":")
            listing = functions.setdefault(head.group(2), [])
            continue
        m = re.match(r"^\s+(\S.*?)\s*// ([0-9A-F]+): [0-9A-F ]+(?:<\w+\+0x([0-9a-f]+)>)?", line)
        if m:
            text.append(m.group(1))
            target = base + int(m.group(3), 16) if m.group(3) else None
            listing.append((int(m.group(2), 16), m.group(1), target))
    return "\n".join(text), functions


needs_tools = pytest.mark.skipif(
    shutil.which(_build.HIPCC) is None or not (_LLVM / "llvm-objdump").exists(),
    reason="hipcc or the LLVM tools not present")


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    into = tmp_path_factory.mktemp("asm")
    with ThreadPoolExecutor(max_workers=8) as pool:
        units = UNITS + DMA_UNITS
        return dict(zip(units, pool.map(lambda u: _assembly(u, into), units)))


def test_lint_catches_a_use_before_the_wait():
    bad = """
_Zkernel:
  global_load_dwordx4 v[4:7], v1, s[2:3]
  v_add_u32 v9, v5, v8
  s_waitcnt vmcnt(0)
  s_endpgm
"""
    good = bad.replace("v_add_u32 v9, v5, v8\n  s_waitcnt vmcnt(0)", "s_waitcnt vmcnt(0)\n  v_add_u32 v9, v5, v8")
    assert len(lint(bad)[2]) == 1
    assert lint(good)[2] == []
    # in-order completion: vmcnt(1) covers the older of two loads only
    two = """
_Zkernel:
  global_load_dword v4, v1, s[2:3]
  global_load_dword v5, v1, s[2:3] offset:4
  s_waitcnt vmcnt(1)
  v_mov_b32 v6, v4
  v_mov_b32 v7, v5
  s_endpgm
"""
    assert len(lint(two)[2]) == 1 and "v[5]" in lint(two)[2][0]
    reloads = """
_Zkernel:
  scratch_load_dwordx2 v[4:5], off, off
  scratch_load_dword v5, off, off offset:8
  s_waitcnt vmcnt(0)
  s_endpgm
"""
    assert lint(reloads)[2] == []
    assert len(lint(reloads.replace("scratch_load_dwordx2 v[4:5], off, off", "global_load_dwordx2 v[4:5], v1, s[2:3]"))[2]) == 1


@needs_tools
def test_no_load_destination_is_touched_before_its_wait(assembly):
    for unit in UNITS:
        functions, loads, problems = lint(assembly[unit][0])
        assert functions > 0, unit
        if unit != "qq_mfma.hip":  # that kernel loads by DMA only: nothing lands in registers
            assert loads > 100, (unit, loads)
        assert not problems, f"{unit}:\n" + "\n".join(problems[:20])


def test_lint_catches_missing_wait_states():
    bad = """
_Zkernel:
  s_mov_b32 m0, s4
  global_load_lds_dwordx4 v1, s[2:3]
  v_readfirstlane_b32 s7, v3
  s_nop 3
  global_load_dword v4, v1, s[6:7]
"""
    good = bad.replace("m0, s4", "m0, s4\n  s_nop 0").replace("s_nop 3", "s_nop 4")
    assert [p.split("`")[2].split()[0] for p in lint_hazards(bad)[1]] == ["right", "reads"]
    assert lint_hazards(good) == (1, [])


@needs_tools
def test_wait_states_ahead_of_loads_in_inline_assembly(assembly):
    for unit, (text, _) in assembly.items():
        loads, problems = lint_hazards(text)
        assert loads > 100, (unit, loads)
        assert not problems, f"{unit}:\n" + "\n".join(problems[:20])


def test_lint_catches_a_spill_in_a_loop():
    body = [(0, "s_nop 0", None), (4, "v_mfma_f32_16x16x32_bf16 a", None),
            (8, "scratch_load_dword v1, off, off", None), (12, "s_cbranch_scc1 65532", 4),
            (16, "scratch_load_dword v1, off, off", None), (20, "s_endpgm", None)]
    assert spills_in_loops(body) == ([(1, 3)], ["scratch_load_dword v1, off, off"])
    body[2] = (8, "s_nop 0", None)
    assert spills_in_loops(body)[1] == []


@needs_tools
def test_no_spilled_register_moves_inside_a_loop_of_matrix_instructions(assembly):
    for unit in UNITS:
        loops = 0
        for name, listing in assembly[unit][1].items():
            inner, moves = spills_in_loops(listing)
            loops += len(inner)
            assert not moves, (unit, name, moves[:3])
        assert loops > 0, unit

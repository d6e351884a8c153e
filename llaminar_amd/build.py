"""Compile the gfx950 quantized-linear library in-tree with hipcc.

Every ``*.hip`` / ``*.cpp`` source under ``llaminar_amd/csrc`` is compiled into
one shared object, ``llaminar_amd/lib/libllaminar_ql.so``.  hipcc cross-compiles
for gfx950 without a GPU, so this runs anywhere the ROCm toolchain is present.

The host-side operator (``csrc/host``) is linked into a second library,
``libllaminar_ql_host.so``, on top of the first.

Sequence models (``csrc/seq``: kernels, operators and step driver over plain bf16 weights)
are a library of their own, ``libllaminar_seq.so``, which needs neither of the others: with
the sampler and the error plumbing it shares with them it builds in well under a minute.

Usage: ``python -m llaminar_amd.build [--incremental] [--seq-only]``
"""
from __future__ import annotations

import fcntl
import os
import re
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
LIBDIR = PKG / "lib"
LIB = LIBDIR / "libllaminar_ql.so"
HOST_LIB = LIBDIR / "libllaminar_ql_host.so"
SEQ_LIB = LIBDIR / "libllaminar_seq.so"
OBJDIR = PKG / "build"

ARCH = "gfx950"
# -packed-fp32-ops is switched OFF: scalar fp32 code must not be fused into
# v_pk_*_f32 forms.  The host pass warns that it does not know the feature.
HIP_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    f"-I{ROOT / 'include'}",
    f"-I{CSRC}",
]
# Register allocation of every kernel is reported by the compiler and checked below.
RESOURCE_FLAG = "-Rpass-analysis=kernel-resource-usage"


class SpillError(RuntimeError):
    """A kernel needs per-lane scratch memory (register spills)."""


def check_kernel_resources(remarks: str, src_name: str) -> dict[str, dict[str, int]]:
    """Parse hipcc's kernel-resource-usage remarks and refuse any kernel that spills.

    Several kernels issue their global loads as inline assembly and wait for them by
    hand many instructions later.  The compiler takes the destination registers of such
    a load as written at the point of issue.  If it has to spill, it may store such a
    register to scratch straight after the load instruction (before the data has
    arrived: the spill slot gets stale contents) and hand the register to another
    value, for instance an address; the load then lands in that value and the kernel
    reads a wild address.  The kernels are only correct with zero spills, so a spill
    fails the build instead of the GPU.
    """
    usage: dict[str, dict[str, int]] = {}
    name = None
    for line in remarks.splitlines():
        # the remark's position is printed before "remark:" or, under -save-temps, after it
        m = re.search(r"remark:(?: \S+:\d+:\d+:)? Function Name: (\S+)", line)
        if m:
            name = m.group(1)
            usage[name] = {}
            continue
        m = re.search(r"remark:(?: \S+:\d+:\d+:)?\s+(ScratchSize \[bytes/lane\]|VGPRs Spill|SGPRs Spill|VGPRs|Dynamic Stack): (\S+)", line)
        if m and name is not None:
            v = m.group(2)
            usage[name][m.group(1)] = int(v) if v.isdigit() else int(v == "True")
    bad = [
        f"{k}: scratch {u.get('ScratchSize [bytes/lane]', 0)} B/lane, {u.get('VGPRs Spill', 0)} VGPRs spilled"
        for k, u in usage.items()
        if u.get("ScratchSize [bytes/lane]", 0) or u.get("VGPRs Spill", 0) or u.get("Dynamic Stack", 0)
    ]
    if bad:
        raise SpillError(
            f"{src_name}: kernels with register spills are refused (hand-scheduled loads are unsafe "
            "once the compiler spills):\n  " + "\n  ".join(bad)
        )
    return usage


class InFlightRegisterError(RuntimeError):
    """Compiler-generated code touches the destination register of a hand-issued load before its wait."""


_VREG = re.compile(r"\bv(\d+)\b|\bv\[(\d+):(\d+)\]")
# (a load into LDS has no destination register: what it names first is its address)
_ASM_LOAD = re.compile(r"^\s*(global_load_(?!lds_)\w+|buffer_load_\w+)\s+(v\d+|v\[\d+:\d+\])\s*,")
_VMEM = re.compile(r"^\s*(global_|buffer_|flat_|scratch_)(load|store|atomic)")
_VMCNT = re.compile(r"vmcnt\((\d+)\)")


def _vregs(text: str) -> set[int]:
    regs: set[int] = set()
    for m in _VREG.finditer(text):
        if m.group(1) is not None:
            regs.add(int(m.group(1)))
        else:
            regs.update(range(int(m.group(2)), int(m.group(3)) + 1))
    return regs


def _device_functions(asm: str):
    """(name, blocks) of every function in the device assembly; a block is a label (None: the function's first) and its
    instructions, in order, each with whether it lies inside inline assembly."""
    name, blocks, in_asm = "?", [(None, [])], False
    for raw_line in asm.splitlines():
        text = raw_line.strip()
        if text.startswith(";;#ASMSTART") or text.startswith(";;#ASMEND"):
            in_asm = text.startswith(";;#ASMSTART")
            continue
        text = text.split(";")[0].strip()
        m = re.match(r"^([A-Za-z_.][\w$.]*):", text)
        if m and not m.group(1).startswith(".L"):
            yield name, blocks
            name, blocks = m.group(1), [(None, [])]
            continue
        if m and m.group(1).startswith(".LBB"):
            blocks.append((m.group(1), []))
            continue
        if text and not text.startswith(".") and not text.endswith(":"):
            blocks[-1][1].append((text, in_asm))
    yield name, blocks


def _control(text: str):
    """("jump" or "branch", label) or ("end", None) of an instruction that control may leave its block at, else None."""
    if m := re.match(r"^s_c?branch\w*\s+(\S+)", text):
        return "jump" if text.startswith("s_branch") else "branch", m.group(1)
    return ("end", None) if re.match(r"^(s_endpgm|s_setpc_b64)\b", text) else None


def _queue_operations(instructions):
    """What of a block's instructions matters to the in-flight check: (kind, registers or label or count, text)."""
    ops = []
    for text, in_asm in instructions:
        if text.startswith("s_waitcnt"):
            w = _VMCNT.search(text)
            if w:
                ops.append(("wait", int(w.group(1)), text))
        elif control := _control(text):
            ops.append((*control, text))
        else:
            load = _ASM_LOAD.match(text) if in_asm else None
            touched = frozenset(_vregs(text))
            if load:
                ops.append(("load", (frozenset(_vregs(load.group(2))), touched), text))
            elif _VMEM.match(text):
                ops.append(("memory", touched, text))
            elif touched:
                ops.append(("use", touched, text))
    return ops


# states of the queue a block may be entered with before the check gives up (the kernels here need up to about a hundred)
MAX_QUEUES = 4000


def check_inflight_registers(asm: str, src_name: str) -> int:
    """Scan the device assembly for the second way the hand-scheduled loads can break.

    The kernels issue global loads inside inline assembly and wait for them (s_waitcnt
    vmcnt, also inline assembly) many instructions later.  To the compiler the destination
    registers hold their values from the point of issue, so besides spilling them it may
    COPY them (a phi move at a loop entry, a move into another allocation) or reuse them
    while the data is still on its way: the copy reads stale contents, or the load lands in
    whatever lives in the register by then.  This pass keeps the queue of vector memory
    operations that vmcnt counts (hand-issued loads with their destination registers, everything
    else as a placeholder), retires entries at each s_waitcnt vmcnt(N), and reports any
    instruction that names a register of a hand-issued load still in the queue.  It follows every
    jump both ways, a block once for each queue it can be entered with; a path that no run
    takes (the same condition tested twice with different outcomes) counts as well.  Returns the number of
    hand-issued loads it found.
    """
    findings: dict[str, None] = {}
    followed = 0
    for func, blocks in _device_functions(asm):
        blocks = [(label, _queue_operations(instructions)) for label, instructions in blocks]
        loads = sum(op[0] == "load" for _, ops in blocks for op in ops)
        followed += loads
        if not loads:
            continue
        at = {label: i for i, (label, _) in enumerate(blocks)}
        seen: list[set] = [set() for _ in blocks]
        work: list[tuple[int, tuple]] = []

        def enter(i, queue):
            while queue and queue[0] is None:   # finished with the wait for anything newer, and no registers
                queue = queue[1:]
            if i is not None and i < len(blocks) and queue not in seen[i]:
                seen[i].add(queue)
                if len(seen[i]) > MAX_QUEUES:
                    raise InFlightRegisterError(f"{src_name}: {func}: too many ways to reach {blocks[i][0]}")
                work.append((i, queue))

        enter(0, ())
        while work:
            i, queue = work.pop()   # oldest first; None: an operation whose registers the compiler tracks
            pending = frozenset().union(*(q for q in queue if q))
            for kind, what, text in blocks[i][1]:
                if kind == "wait":
                    queue = queue[len(queue) - what:] if 0 < what < len(queue) else (() if what == 0 else queue)
                    pending = frozenset().union(*(q for q in queue if q))
                elif kind in ("jump", "branch"):
                    enter(at.get(what), queue)
                    if kind == "jump":
                        break
                elif kind == "end":
                    break
                elif kind == "load":
                    dst, touched = what
                    if hit := touched & pending:
                        findings[f"{func}: '{text}' uses v{min(hit)} while a hand-issued load into it is in flight"] = None
                    queue, pending = (*queue, dst)[-64:], pending | dst   # (vmcnt counts to 63)
                else:
                    if hit := what & pending:
                        findings[f"{func}: '{text}' touches v{min(hit)} before the wait for the hand-issued load into it"] = None
                    if kind == "memory" and queue:
                        queue = (*queue, None)[-64:]
            else:
                enter(i + 1, queue)
    if findings:
        shown = list(findings)[:12]
        raise InFlightRegisterError(
            f"{src_name}: registers of hand-issued loads are touched before their s_waitcnt "
            "(the data has not arrived; see check_inflight_registers):\n  " + "\n  ".join(shown)
            + ("" if len(findings) <= 12 else f"\n  ... and {len(findings) - 12} more"))
    return followed


class ScalarHazardError(RuntimeError):
    """A hand-issued load reads a scalar register too soon after it has been written."""


_SREG = re.compile(r"\bs(\d+)\b|\bs\[(\d+):(\d+)\]")
_VALU_TO_SREG = re.compile(r"^v_\w+\s+(s\d+|s\[\d+:\d+\])\s*,")
SCALAR_WAIT_STATES = 5
# m0: the address of a load into LDS
_M0_WRITE = re.compile(r"^[sv]_\w+\s+m0\s*,")
_LDS_LOAD = re.compile(r"^(global_load_lds_\w+|(buffer|global)_load_\w+\s.*\blds\b)")
M0_WAIT_STATES = 1
M0 = -1


def _sregs(text: str) -> set[int]:
    regs: set[int] = set()
    for m in _SREG.finditer(text):
        regs.update([int(m.group(1))] if m.group(1) is not None else range(int(m.group(2)), int(m.group(3)) + 1))
    return regs


def check_scalar_hazards(asm: str, src_name: str) -> int:
    """Scan the device assembly for vector memory instructions inside inline assembly that read a scalar register
    less than five wait states after a vector instruction (v_readfirstlane, v_cmp) wrote it.

    The hardware does not wait by itself, and the compiler inserts the wait states for its own instructions only: such
    a load takes a stale value, half of another pointer, for its base.  An instruction counts as one wait state,
    s_nop N as N + 1.  Likewise a load into LDS whose address was written into m0 less than one wait state before: it may
    land at the address before.  Every jump is followed both ways; where ways meet, a register counts as written as lately as on any of
    them.  Returns the number of loads and stores looked at.
    """
    findings: dict[str, None] = {}
    looked = 0
    for func, blocks in _device_functions(asm):
        own = sum(in_asm and _VMEM.match(text) is not None for _, instructions in blocks for text, in_asm in instructions)
        looked += own
        if not own:
            continue
        at = {label: i for i, (label, _) in enumerate(blocks)}
        # scalar register -> fewest wait states since a vector instruction (m0: any) wrote it, where a block begins (None: not reached)
        begin: list[dict[int, int] | None] = [None] * len(blocks)
        work: list[int] = []

        def enter(i, written):
            if i is None or i >= len(blocks):
                return
            if begin[i] is None:
                begin[i] = dict(written)
            else:
                less = {r: n for r, n in written.items() if n < begin[i].get(r, SCALAR_WAIT_STATES)}
                if not less:
                    return
                begin[i].update(less)
            work.append(i)

        enter(0, {})
        while work:
            i = work.pop()
            written = dict(begin[i])
            for text, in_asm in blocks[i][1]:
                if in_asm and written and _VMEM.match(text):
                    hit = sorted(r for r in _sregs(text) if r in written)
                    if hit:
                        findings[f"{func}: '{text}' reads s{hit[0]} {written[hit[0]]} wait states after a vector instruction wrote it"] = None
                    if _LDS_LOAD.match(text) and written.get(M0, M0_WAIT_STATES) < M0_WAIT_STATES:
                        findings[f"{func}: '{text}' reads m0 {written[M0]} wait states after it was written"] = None
                if written:
                    passed = int(text.split()[1], 0) + 1 if text.startswith("s_nop") else 1
                    written = {r: n + passed for r, n in written.items() if n + passed < SCALAR_WAIT_STATES}
                if m := _VALU_TO_SREG.match(text):
                    written.update(dict.fromkeys(_sregs(m.group(1)), 0))
                if _M0_WRITE.match(text):
                    written[M0] = 0
                if control := _control(text):
                    enter(at.get(control[1]), written)
                    if control[0] != "branch":
                        break
            else:
                enter(i + 1, written)
    if findings:
        shown = "\n  ".join(list(findings)[:12]) + ("" if len(findings) <= 12 else f"\n  ... and {len(findings) - 12} more")
        raise ScalarHazardError(f"{src_name}: hand-issued loads take a stale scalar register (see check_scalar_hazards):\n  {shown}")
    return looked


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(exe).exists():
        raise RuntimeError("hipcc not found: the ROCm toolchain is required to build llaminar_amd")
    return exe


def sources() -> list[Path]:
    return sorted(list(CSRC.glob("*.hip")) + list(CSRC.glob("*.cpp")))


def seq_sources() -> list[Path]:
    seq = CSRC / "seq"
    return sorted(list(seq.glob("*.hip")) + list(seq.glob("*.cpp"))) + [CSRC / "ql_common.hip", CSRC / "sampling.hip"]


def _deps_mtime() -> float:
    files = [f for f in CSRC.rglob("*") if f.is_file()] + list((ROOT / "include" / "llaminar_amd").glob("*.h*"))
    return max(f.stat().st_mtime for f in files)


def build_host(verbose: bool = True) -> Path:
    """Link the C++ operator layer against the kernel library (no device code)."""
    srcs = sorted((CSRC / "host").glob("*.cpp"))
    cmd = [hipcc(), "-std=c++17", "-O2", "-fPIC", "-shared", f"-I{ROOT / 'include'}", *map(str, srcs),
           f"-L{LIBDIR}", "-lllaminar_ql", "-Wl,-rpath,$ORIGIN", "-o", str(HOST_LIB)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"host library build failed:\n{proc.stderr}")
    if verbose:
        print(f"[llaminar_amd.build] wrote {HOST_LIB} ({HOST_LIB.stat().st_size} bytes)", flush=True)
    return HOST_LIB


def _drop_resource_remarks(lines: list[str]) -> list[str]:
    """Compiler output without the kernel-resource-usage remarks and their source excerpts."""
    out, skip = [], 0
    for l in lines:
        if "[-Rpass-analysis=kernel-resource-usage]" in l:
            skip = 2 if "Function Name" in l else 0  # the excerpt: source line and caret line
            continue
        if skip and (re.match(r"\s*\d+ \|", l) or re.match(r"\s*\|\s*\^", l)):
            skip -= 1
            continue
        skip = 0
        if re.match(r"In file included from ", l) or re.search(r"\d+ (warning|remark)s? generated", l):
            continue
        out.append(l)
    return out


def _headers_mtime() -> float:
    files = list(CSRC.glob("*.h")) + list((CSRC / "seq").glob("*.h")) + list((ROOT / "include" / "llaminar_amd").glob("*.h*"))
    return max(f.stat().st_mtime for f in files)


def _compile(src: Path, force: bool = True) -> Path:
    obj = OBJDIR / (src.stem + ".o")
    # without force an object newer than its source and every header is kept (it passed the checks below
    # when it was made)
    if not force and obj.exists() and obj.stat().st_mtime >= max(src.stat().st_mtime, _headers_mtime()):
        return obj
    # -save-temps leaves the device assembly beside the object file for check_inflight_registers
    cmd = [hipcc(), *HIP_FLAGS, RESOURCE_FLAG, "-save-temps=obj", "-c", str(src), "-o", str(obj)]
    if src.suffix == ".cpp":
        cmd.insert(1, "-x")
        cmd.insert(2, "hip")
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    lines = [l for l in proc.stderr.splitlines() if noise not in l]
    if proc.returncode == 0:
        try:
            check_kernel_resources(proc.stderr, src.name)
            for asm_file in OBJDIR.glob(f"{src.stem}-hip-amdgcn-*.s"):
                asm = asm_file.read_text()
                check_inflight_registers(asm, src.name)
                check_scalar_hazards(asm, src.name)
        except Exception:
            obj.unlink(missing_ok=True)   # (a later build without force would keep it)
            raise
    err = "\n".join(_drop_resource_remarks(lines))
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _link(objs: list[Path], lib: Path, verbose: bool) -> None:
    # into a name of its own first: a process that loads the library meanwhile sees the old one or the new one
    part = lib.with_suffix(f".{os.getpid()}.part")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), f"-Wl,-soname,{lib.name}", "-o", str(part)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        part.unlink(missing_ok=True)
        raise RuntimeError(f"link failed:\n{proc.stderr}")
    part.replace(lib)
    if verbose:
        print(f"[llaminar_amd.build] wrote {lib} ({lib.stat().st_size} bytes)", flush=True)


def build_seq(force: bool = True, verbose: bool = True) -> Path:
    """Compile and link the sequence-model library alone.  With force=False an up-to-date one is kept."""
    OBJDIR.mkdir(exist_ok=True)
    LIBDIR.mkdir(exist_ok=True)
    srcs = seq_sources()
    with open(OBJDIR / ".seq.lock", "w") as lock:
        fcntl.flock(lock, fcntl.LOCK_EX)  # one builder at a time in a checkout
        newest = max([f.stat().st_mtime for f in srcs] + [_headers_mtime()])
        if not force and SEQ_LIB.exists() and SEQ_LIB.stat().st_mtime >= newest:
            return SEQ_LIB
        if verbose:
            print(f"[llaminar_amd.build] hipcc {ARCH}: {len(srcs)} sources of the sequence models", flush=True)
        with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as pool:
            objs = list(pool.map(lambda src: _compile(src, force), srcs))
        _link(objs, SEQ_LIB, verbose)
    return SEQ_LIB


def build(force: bool = True, verbose: bool = True) -> Path:
    """Compile and link the libraries.  With force=False up-to-date ones are kept."""
    build_seq(force, verbose)
    if not force and LIB.exists() and HOST_LIB.exists() and LIB.stat().st_mtime >= _deps_mtime():
        return LIB
    OBJDIR.mkdir(exist_ok=True)
    LIBDIR.mkdir(exist_ok=True)
    srcs = sources()
    if verbose:
        print(f"[llaminar_amd.build] hipcc {ARCH}: {len(srcs)} sources", flush=True)
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as pool:
        objs = list(pool.map(lambda src: _compile(src, force), srcs))
    _link(objs, LIB, verbose)
    build_host(verbose)
    return LIB


if __name__ == "__main__":
    (build_seq if "--seq-only" in sys.argv else build)(force="--incremental" not in sys.argv)

"""Build libccfuser_moe.so (the product) and libccfuser_probe.so (measurement probes) from the
HIP sources with hipcc for gfx950.

    python -m ccfuser_amd.build          # compile every source, check, link both libraries

hipcc cross-compiles without a GPU.  Objects go to ``ccfuser_amd/csrc/_obj`` and the
libraries next to this file, so they travel with the source tree.
"""
from __future__ import annotations

import os
import re
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
LIB = HERE / "libccfuser_moe.so"
PROBE_LIB = HERE / "libccfuser_probe.so"
SOURCES = ["api.hip", "gate.hip", "route.hip", "rows.hip", "bwd.hip", "few.hip", "thin.hip", "ffn.hip"]
PROBE_SOURCES = ["probe.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
COMMON = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    # packed fp32 VALU forms are kept off on this hardware pool
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]
PER_FILE = {
    # the gate's fp32 accumulation order must survive the optimiser
    "gate.hip": ["-ffp-contract=off"],
    # the 16x16x32 main loop names its accumulation registers itself: nothing of the compiler's may live there
    "ffn.hip": ["-mllvm", "-amdgpu-spill-vgpr-to-agpr=0"],
    "probe.hip": ["-mllvm", "-amdgpu-spill-vgpr-to-agpr=0"],
}
# Sources whose kernels name accumulation registers (AGPRs) literally in inline asm, and the
# kernels (regex on the mangled name) that do.  If the compiler parks a value of its own in
# such a register, or spills, the asm overwrites it; both times that happened the value was an
# address and the kernel faulted the GPU.  So these are compiled to assembly and scanned, and a
# library that fails the scan is never linked.
ACC_CHECKED = {
    "ffn.hip": r"_ZN3ccf\S*grouped_gemm\S*",
    "probe.hip": r"_ZN3ccf\S*mfma_probe_kernel\S*",
}
# Sources whose kernels leave LDS reads written in inline asm in flight behind the statement that issues them, and the
# kernels that do.  The compiler takes such a register as written at once: a copy of it, or another value put into it,
# ahead of the wait would be silently wrong.  They are scanned for that, along all branches, and for spills.
READS_CHECKED = {
    "few.hip": r"_ZN3ccf\S*few_rows_kernel\S*",
}
# Kernels with such reads whose branches depend on each other in ways that the scan cannot see, so that it finds uses on
# ways that no wavefront takes: scanned for copies of pending registers, which the compiler makes where loops meet.
COPIES_CHECKED = {
    "ffn.hip": r"_ZN3ccf\S*grouped_gemm\S*",
}
_NOISE = "is not a recognized feature for this target"


def _run(cmd):
    res = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in res.stderr.splitlines() if _NOISE not in l)
    return res.returncode, err


def _compile(src: str) -> Path:
    obj_dir = CSRC / "_obj"
    obj_dir.mkdir(exist_ok=True)
    obj = obj_dir / (src + ".o")
    rc, err = _run([HIPCC, *COMMON, *PER_FILE.get(src, []), "-c", str(CSRC / src), "-o", str(obj)])
    if rc != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def kernel_bodies(asm_text: str, name_regex: str):
    """(name, assembly text) of every kernel whose mangled name matches: from its label to the
    end-of-function label, so code behind an early s_endpgm is part of the body."""
    out = []
    for m in re.finditer(r"^(" + name_regex + r"):[^\n]*\n", asm_text, flags=re.M):
        end = asm_text.find(".Lfunc_end", m.end())
        out.append((m.group(1), asm_text[m.end(): end if end >= 0 else len(asm_text)]))
    return out


def acc_register_violations(asm_text: str, name_regex: str):
    """Accumulation-register moves of the compiler's own, and scratch accesses, in the kernels
    that name those registers themselves.  The hand-written asm uses the bracket form a[N]; the
    compiler prints aN."""
    bad = []
    for name, body in kernel_bodies(asm_text, name_regex):
        stray = re.findall(r"^\s*(v_accvgpr_(?:write_b32 a\d+, v\d+|read_b32 v\d+, a\d+|mov_b32 .*))$", body, flags=re.M)
        if stray:
            bad.append((name, stray[:5]))
        if "scratch_" in body:
            bad.append((name, ["scratch access"]))
    return bad


_REGISTER = re.compile(r"(?<![\w.])([va])(?:(\d+)|\[(\w+)(?::(\w+))?\])")


def _registers(operands: str) -> int:
    """The vector and accumulation registers that an operand list names, as a bit mask."""
    mask = 0
    for kind, one, lo, hi in _REGISTER.findall(operands):
        first = int(one or lo, 0)
        last = int(hi, 0) if hi else first
        mask |= ((1 << (last - first + 1)) - 1) << (first + (512 if kind == "a" else 0))
    return mask


def _instructions(body: str):
    """(operation, operands) of every instruction of a kernel, and the index that each label stands for."""
    code, labels = [], {}
    for line in body.splitlines():
        text = line.split(";")[0].split("//")[0].strip()
        label = re.match(r"([.\w$]+):$", text)
        if label:
            labels[label.group(1)] = len(code)
        elif text and not text.startswith("."):
            op, _, operands = text.replace("\t", " ").partition(" ")
            code.append((op, operands.strip()))
    return code, labels


def pending_read_violations(body: str, copies_only: bool = False):
    """Instructions of a kernel that name the destination of an LDS or memory load ahead of the wait that covers it;
    copies_only: register moves that name an LDS read's.

    Loads of either kind return in order, so a wait for at most n of them leaves the n newest.  Per block of code the
    state is, for either kind, the destinations by age, newest last; where branches meet, a destination has every age
    that it may have, which can only find too much.  A load may overwrite the destination of an earlier one of its kind."""
    code, labels = _instructions(body)
    steps = []
    for op, operands in code:
        first, _, rest = operands.partition(",")
        if op.startswith("ds_"):
            loads = re.search(r"read|permute|swizzle|rtn", op) is not None
            steps.append(("lds", _registers(rest if loads else operands), _registers(first) if loads else 0))
        elif re.match(r"(global|buffer|scratch)_", op):
            loads = "load" in op and "_lds_" not in op or "atomic" in op and "sc0" in operands
            steps.append(("mem", _registers(rest if loads else operands), _registers(first) if loads else 0))
        elif op == "s_waitcnt":
            left = {kind: re.search(name + r"\((\d+)\)", operands) for kind, name in (("lds", "lgkmcnt"), ("mem", "vmcnt"))}
            if "cnt(" not in operands:
                raise ValueError(f"{op} {operands}")
            steps.append(("wait", {kind: int(m.group(1)) for kind, m in left.items() if m}, 0))
        elif op == "s_branch" or op.startswith("s_cbranch"):
            steps.append(("jump" if op == "s_branch" else "branch", labels[operands], 0))
        elif op == "s_endpgm":
            steps.append(("end", 0, 0))
        elif re.match(r"flat_|s_(setpc|swappc|call)", op):
            raise ValueError(f"{op} {operands}")
        else:
            steps.append(("other", _registers(operands), 0))
    heads = sorted({0, *labels.values(), *(i + 1 for i, s in enumerate(steps) if s[0] in ("jump", "branch", "end"))})
    block_end = dict(zip(heads, heads[1:] + [len(steps)]))
    entry, todo, bad = {0: {"lds": [], "mem": []}}, [0], set()

    def meet(at, state):
        known = entry.setdefault(at, {"lds": None, "mem": None})
        grown = False
        for kind, ages in state.items():
            ages = ages[-64:]
            old = known[kind]
            if old is None:
                known[kind], grown = list(ages), True
                continue
            old[:0] = [0] * (len(ages) - len(old))
            for q in range(1, len(ages) + 1):
                grown = grown or bool(ages[-q] & ~old[-q])
                old[-q] |= ages[-q]
        if grown:
            todo.append(at)

    while todo:
        at = todo.pop()
        state = {kind: list(ages) for kind, ages in entry[at].items()}
        end = block_end.get(at, len(steps))
        while at < end:
            kind, named, dest = steps[at]
            at += 1
            if kind == "wait":
                for which, left in named.items():
                    del state[which][:max(len(state[which]) - left, 0)]
            elif kind in ("jump", "branch"):
                meet(named, state)
                if kind == "jump":
                    break
            elif kind == "end":
                break
            else:
                for which, ages in state.items():
                    if copies_only and not (which == "lds" and re.match(r"v_(mov|accvgpr)", code[at - 1][0])):
                        continue
                    if any(p & (named if which == kind else named | dest) for p in ages):
                        bad.add((at - 1, " ".join(code[at - 1])))
                if kind != "other":
                    state[kind].append(dest)
        else:
            if at < len(steps):
                meet(at, state)
    return [text for _, text in sorted(bad)]


def spilled_bytes(asm_text: str, name_regex: str):
    """{kernel: bytes of scratch memory a thread needs} from the kernels' metadata."""
    records = re.findall(r"\.name:\s+(\S+)((?:(?!\.name:).)*?)\.private_segment_fixed_size:\s+(\d+)", asm_text, flags=re.S)
    return {name: int(size) for name, _, size in records if re.fullmatch(name_regex, name)}


def device_assembly(src: str, out: Path) -> str:
    rc, err = _run([HIPCC, *COMMON, *PER_FILE.get(src, []), "-S", "--cuda-device-only", str(CSRC / src), "-o", str(out)])
    if rc != 0:
        raise RuntimeError(f"hipcc -S failed on {src}:\n{err}")
    return out.read_text()


def _check(src: str) -> None:
    obj_dir = CSRC / "_obj"
    obj_dir.mkdir(exist_ok=True)
    text = device_assembly(src, obj_dir / (src + ".s"))
    if src in ACC_CHECKED:
        bad = acc_register_violations(text, ACC_CHECKED[src])
        if bad:
            raise RuntimeError(f"{src}: the compiler uses accumulation registers that the kernels name themselves, "
                               f"or spills; such a binary faults the GPU and is not linked: {bad[:3]}")
    if src in READS_CHECKED:
        for name, body in kernel_bodies(text, READS_CHECKED[src]):
            bad = pending_read_violations(body)
            if bad:
                raise RuntimeError(f"{src}: {name} touches the destination of a read in flight; not linked: {bad[:3]}")
    for name, body in kernel_bodies(text, COPIES_CHECKED[src]) if src in COPIES_CHECKED else []:
        bad = pending_read_violations(body, copies_only=True)
        if bad:
            raise RuntimeError(f"{src}: {name} copies the destination of a read in flight; not linked: {bad[:3]}")
    if src in READS_CHECKED:
        bad = {k: n for k, n in spilled_bytes(text, READS_CHECKED[src]).items() if n}
        if bad:
            raise RuntimeError(f"{src}: spills next to reads in flight; not linked: {bad}")


def _link(objs, lib: Path) -> None:
    rc, err = _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc",
                    "-Wno-unused-command-line-argument", *map(str, objs), "-o", str(lib)])
    if rc != 0:
        raise RuntimeError(f"link failed:\n{err}")


def build(verbose: bool = True) -> Path:
    """Compile every HIP source, scan the kernels that own their accumulation registers or leave reads in flight, and
    link both shared libraries.  Always recompiles."""
    srcs = SOURCES + PROBE_SOURCES
    with ThreadPoolExecutor(max_workers=8) as pool:
        checks = [pool.submit(_check, s) for s in {**ACC_CHECKED, **READS_CHECKED, **COPIES_CHECKED}]
        objs = dict(zip(srcs, pool.map(_compile, srcs)))
        for c in checks:
            c.result()
    _link([objs[s] for s in SOURCES], LIB)
    _link([objs[s] for s in PROBE_SOURCES], PROBE_LIB)
    if verbose:
        print(f"built {LIB} ({LIB.stat().st_size} bytes), {PROBE_LIB} ({PROBE_LIB.stat().st_size} bytes)")
    return LIB


if __name__ == "__main__":
    build()

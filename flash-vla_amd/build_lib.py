"""Build libpi0hip.so (gfx950) from csrc/*.hip with hipcc, in-tree.

Usage: python flash-vla_amd/build_lib.py   (or __graft_entry__.build())
Objects go to flash-vla_amd/_build/, the library to flash_vla_amd/lib/.
"""
from __future__ import annotations

import concurrent.futures as cf
import glob
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(ROOT, "include")
BUILD = os.path.join(HERE, "_build")
LIBDIR = os.path.join(HERE, "flash_vla_amd", "lib")
LIB = os.path.join(LIBDIR, "libpi0hip.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", f"-I{INCLUDE}",
    # packed fp32 VALU ops are kept out of generated code on this hardware
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, os.path.basename(src).replace(".hip", ".o"))
    cmd = [HIPCC, *FLAGS, "-c", src, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{res.stderr}")
    return obj


# packed fp32 VALU forms must not appear in the device code (see FLAGS)
_PACKED_FP32 = re.compile(r"\bv_pk_(add|mul|fma)_f32\b")


def check_kblock_waits(asm: str) -> list[str]:
    """Names of skinny GEMM kernels whose k-block waits do not cover their LDS copies.

    skinny_gemm_kernel issues, per k-block, buffer loads that write x straight into
    LDS and that k-block's weight loads (x first, or the weights some k-blocks ahead:
    one k-block's copies are contiguous, the k-blocks' copies go out in order, and the
    loop waits once per k-block); before the MFMAs of k-block j it waits with vmcnt(N). Vector-memory operations complete in issue order, so the wait is
    sufficient only if N is at most the number of operations issued after k-block j's
    last LDS copy. This re-checks that order in the generated code (the scheduling
    barriers in the source are what keep it).
    """
    bad = []
    for m in re.finditer(r"^(_ZN3pi018skinny_gemm_kernelI\w+):", asm, re.M):
        body = asm[m.end():asm.index("s_endpgm", m.end())]
        lines = [ln.strip() for ln in body.split("\n")]
        first_ds = next(i for i, ln in enumerate(lines) if ln.startswith("ds_read"))
        issue = [i for i, ln in enumerate(lines[:first_ds])
                 if ln.startswith(("global_load", "buffer_load"))]
        kinds = ["lds" if lines[i].endswith(" lds") else "reg" for i in issue]
        waits = [int(w) for w in re.findall(r"s_waitcnt vmcnt\((\d+)\)",
                                            "\n".join(lines[issue[-1] + 1:]))]
        tail = lines[issue[-1] + 1:]
        loop = "\n".join(tail[:next((i for i, ln in enumerate(tail) if ln.startswith("s_barrier")),
                                     len(tail))])
        nkb = len(re.findall(r"s_waitcnt vmcnt\(\d+\)", loop))
        copies = [j for j, k in enumerate(kinds) if k == "lds"]
        per = len(copies) // nkb if nkb and len(copies) % nkb == 0 else 0
        last_copy = copies[per - 1::per] if per else []
        ok = bool(last_copy) and len(waits) >= len(last_copy) and all(
            waits[j] <= len(kinds) - 1 - c for j, c in enumerate(last_copy))
        if not ok:
            bad.append(m.group(1))
    return bad


def _kernels(asm: str, pattern: str):
    """(name, events) of the kernels matching `pattern`. Events, in text order: "C" a buffer load
    into LDS, "L" any other load, "R" an LDS read, "B" a barrier, ("V", n) / ("K", n) a wait that
    leaves n vector-memory / LDS operations outstanding, "E" the end of the text."""
    for m in re.finditer(rf"^(_ZN3pi0\d+(?:{pattern})I?\w*):", asm, re.M):
        events = []
        for ln in asm[m.end():asm.index("s_endpgm", m.end())].split("\n"):
            ln = ln.split(";")[0].strip()
            if ln.startswith(("global_load", "buffer_load")):
                events.append("C" if ln.endswith(" lds") else "L")
            elif ln.startswith("ds_read"):
                events.append("R")
            elif ln.startswith("s_barrier"):
                events.append("B")
            elif ln.startswith("s_waitcnt"):
                for op, kind in (("vmcnt", "V"), ("lgkmcnt", "K")):
                    w = re.search(rf"\b{op}\((\d+)\)", ln)
                    if w:
                        events.append((kind, int(w.group(1))))
        yield m.group(1), events + ["E"]


# kernels whose waves read only what they copied themselves, in chunks of four copies that four
# LDS reads consume, through four slots a wave
_PRIVATE_CHUNKS = "rows32_res_kernel|qkv_rows32_kernel|gate_stream_kernel"


def check_chunk_waits(asm: str) -> tuple[list[str], list[str]]:
    """The kernels of _PRIVATE_CHUNKS (names with a wait that is too loose, names with a wait for
    everything in flight before the last chunk).

    Vector-memory operations complete in issue order, so at a wait vmcnt(N) all but the N newest
    have landed: the last copy of a chunk must be among those when the chunk is read, and a copy
    into a slot must follow the completed reads of the chunk that the slot held."""
    loose, full = [], []
    for name, events in _kernels(asm, _PRIVATE_CHUNKS):
        issued = landed = reads = read_done = 0
        copies, ok, drained = [], True, False
        for e in events[:events.index("B")]:
            if e in ("C", "L"):
                if e == "C":
                    ok &= len(copies) // 4 < 4 or read_done >= (len(copies) // 4 - 3) * 4
                    copies.append(issued)
                issued += 1
            elif e == "R":
                last = reads // 4 * 4 + 3
                ok &= last < len(copies) and copies[last] < landed
                reads += 1
            elif e[0] == "V":
                drained |= e[1] == 0 and reads // 4 + 1 < len(copies) // 4
                landed = max(landed, issued - e[1])
            elif e[0] == "K":
                read_done = max(read_done, reads - e[1])
        if not ok or reads != len(copies) or not copies:
            loose.append(name)
        if drained:
            full.append(name)
    return loose, full


# kernels whose k loop shares its copies between waves, a wait and a barrier per step, and the
# steps that may still be in flight at a wait of a loop unrolled over n steps
_SHARED_STEPS = {"tile_gemm_kernel": lambda n: n - 2,    # step s read next, up to s + n - 2 issued
                 "block_gemm_kernel": lambda n: n - 2,   # s + 1 read next, s + n - 1 issued
                 "enc_attn_wide_kernel": lambda n: 1}    # b + 1 read next, b + 2 issued


def check_step_waits(asm: str) -> list[str]:
    """Names of the kernels of _SHARED_STEPS whose k loop waits for less than the copies of the
    step behind the barrier and the reads of the slot that is filled next, or for more."""
    bad = []
    for kernel, in_flight in _SHARED_STEPS.items():
        strip = kernel == "tile_gemm_kernel"             # weights to registers, not to LDS
        for name, events in _kernels(asm, kernel):
            waits = {}                                   # barrier -> its wait's vmcnt
            for i, e in enumerate(events):
                if e == "B":
                    waits.update({i: v[1] for v in events[i - 2:i] if v[0] == "V"})
            steps = sorted(waits)
            end = events.index(("V", 0), steps[0])       # everything lands before the epilogue
            steps = [i for i in steps if i < end]
            loop = events[steps[0]:end]
            lead = None if strip else steps.pop(0)       # the wait in front of the loop
            n, copies, loads = len(steps), loop.count("C"), loop.count("L")
            if n == 0 or copies == 0 or copies % n or loads % n:
                bad.append(name)
                continue
            copies, loads = copies // n, loads // n
            # a strip's weight loads of the step itself are waited for where they are used
            bound = in_flight(n) * (copies + loads) + (loads if strip else 0)
            ok = all(waits[i] == bound for i in steps)
            for i, j in zip(steps, steps[1:]):
                ok &= events[i:j].count("C") == copies and events[i:j].count("L") == loads
            if strip:                                    # a step's copies before its weights
                ok &= all("L" not in events[i:events.index("C", i)] for i in steps)
            else:
                ok &= all(events[i - 1] == ("K", 0) for i in steps)
                ok &= waits[lead] <= events[:lead].count("C") - copies
            if not ok:
                bad.append(name)
    return bad


# kernels whose every copy lies inside its resource, whatever the call's sizes
_COPIES_IN_RANGE = ("enc_attn_wide_kernel",)      # clamped blocks of the packed K and V^T


def unchecked_copies(asm: str) -> list[str]:
    """Names of kernels with a buffer load into LDS whose scalar offset is not zero.

    Rows past M, and the columns past a row's end that a padded K asks for, rely on the range
    check of the activation's buffer resource. The check is documented for the lane and the
    immediate offset only, so nothing may sit in the scalar one."""
    bad = []
    for m in re.finditer(r"^(_ZN3pi0\w+):", asm, re.M):
        body = asm[m.end():asm.index("s_endpgm", m.end())]
        copies = [ln.split(";")[0].rstrip() for ln in body.split("\n")
                  if re.match(r"\s*buffer_load\w*\s.*\blds\b", ln)]
        soffs = {ln.split(",")[-1].split()[0] for ln in copies}
        if soffs - {"0"} and not any(k in m.group(1) for k in _COPIES_IN_RANGE):
            bad.append(m.group(1))
    return bad


def scratch_kernels(asm: str) -> list[str]:
    """Kernels whose private (scratch) segment is not empty: a spill, or a kernel argument
    indexed at run time and so copied to the stack -- both silent slowdowns."""
    bad = []
    for m in re.finditer(r"^\s*\.amdhsa_kernel\s+(\S+)(.*?)^\s*\.end_amdhsa_kernel", asm, re.M | re.S):
        size = re.search(r"\.amdhsa_private_segment_fixed_size\s+(\d+)", m.group(2))
        if size and int(size.group(1)) > 0:
            bad.append(m.group(1))
    return bad


def check_device_code(src: str) -> None:
    """Compile `src` to device assembly and fail if any packed fp32 VALU op was
    generated, if any kernel uses scratch memory, if a copy into LDS could leave its
    resource's range check, or if a counted wait does not cover the copies it stands for."""
    cmd = [HIPCC, *FLAGS, "--cuda-device-only", "-S", src, "-o", "-"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc -S failed for {src}:\n{res.stderr}")
    if _PACKED_FP32.search(res.stdout):
        raise RuntimeError(f"{src}: packed fp32 VALU instructions in the device code")
    scratch = scratch_kernels(res.stdout)
    if scratch:
        raise RuntimeError(f"{src}: kernels with a scratch segment: {scratch}")
    loose = unchecked_copies(res.stdout)
    if loose:
        raise RuntimeError(f"{src}: LDS copies outside the range check in {loose}")
    waits = check_chunk_waits(res.stdout)[0] + check_step_waits(res.stdout)
    if waits:
        raise RuntimeError(f"{src}: counted waits do not match the LDS copies in {waits}")
    if os.path.basename(src) == "pi0_gemm.hip":
        bad = check_kblock_waits(res.stdout)
        if bad:
            raise RuntimeError(f"{src}: k-block vmcnt waits do not cover the LDS copies in {bad}")


def build(verbose: bool = False, check_isa: bool = True) -> str:
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    with cf.ThreadPoolExecutor(max_workers=min(8, len(sources))) as ex:
        objs = list(ex.map(_compile, sources))
        if check_isa:
            list(ex.map(check_device_code, sources))
    tmp = LIB + ".tmp"
    # --no-undefined: a kernel whose host stub was not emitted fails here, not at load time
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-Wl,--no-undefined", *objs,
           "-o", tmp]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)

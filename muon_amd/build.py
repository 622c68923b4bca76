"""Builds muon_amd/libmuon_amd.so from muon_amd/csrc/*.hip with hipcc for gfx950.

    python -m muon_amd.build

After the library is built, the GEMM kernels are compiled once more to assembly and checked
(`check_fragment_waits`): their main loop requests its LDS fragments through inline assembly and
waits for them by hand, which is only correct while the compiler does not touch a requested
register before the wait that covers it.  The same listing is checked for vector instructions that
overwrite the data of a wide store right behind it (`check_store_data`).
"""
from __future__ import annotations

import os
import re
import shutil
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libmuon_amd.so")
SOURCES = ["capi.hip", "elementwise.hip", "aol.hip", "ns_gemm.hip", "small.hip", "step.hip"]
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    # hipcc -O3 must not form packed-fp32 instructions on this target
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
# The GEMM kernels' arguments arrive in scalar registers with the dispatch instead of through a load of each wave's own: 0.2 us
# for each of the 15 dependent launches of a small matrix (768 x 3072: 174.8 -> 171.2 us, runs of one build differ by 0.1 %).  In a
# step of one launch that does not show in the call (64 x 64 x 3 x 3: the kernel 37.0 -> 36.7 us, the call 47.6-48.3 -> 46.9-48.1 us
# with runs of one build 0.3-3 % apart; Adam over 50257 x 768 171.9 -> 171.9 us), so the other sources are built without it.
SOURCE_FLAGS = {"ns_gemm.hip": ["-mllvm", "-amdgpu-kernarg-preload-count=16"]}


_VREG = re.compile(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b")


def _vregs(text: str) -> frozenset:
    out = set()
    for m in _VREG.finditer(text):
        if m.group(1):
            out |= set(range(int(m.group(1)), int(m.group(2)) + 1))
        else:
            out.add(int(m.group(3)))
    return frozenset(out)


def check_fragment_waits(asm_text: str) -> int:
    """Walks the control-flow graph of every ns_gemm_kernel in a hipcc -S listing.  A register that an
    inline-assembly LDS read (ds_read_b128, ds_read_b64_tr_b16) has requested is pending until a `s_waitcnt lgkmcnt(n)` leaves at
    most n younger requests outstanding (LDS reads return in order).  Raises if any instruction --
    a copy the register allocator put at a loop edge, an address computation, an MFMA -- names a
    pending register: it would see the register before its data.  Returns the number of such reads
    it followed."""
    lines = asm_text.split("\n")
    starts = [i for i, l in enumerate(lines) if re.match(r"^_ZN8muon_amd14ns_gemm_kernel\S*:", l)]
    if not starts:
        raise RuntimeError("check_fragment_waits: no ns_gemm_kernel in the listing")
    nreads = 0
    for k0 in starts:
        instrs, labels, inasm = [], {}, False
        for i in range(k0 + 1, len(lines)):
            t = lines[i].strip()
            if t.startswith(".Lfunc_end"):
                break
            if ";;#ASMSTART" in t:
                inasm = True
            elif ";;#ASMEND" in t:
                inasm = False
            elif re.match(r"^\.LBB\d+_\d+:", t):
                labels[t.split(":")[0]] = len(instrs)
            elif t and not t.startswith(";") and not t.startswith("."):
                instrs.append((t, inasm, i + 1))
        seen, stack = set(), [(0, ())]
        while stack:
            pc, pend = stack.pop()
            while pc < len(instrs) and (pc, pend) not in seen:
                seen.add((pc, pend))
                t, from_asm, line_no = instrs[pc]
                op = t.split()[0]
                if op == "s_waitcnt":
                    m = re.search(r"lgkmcnt\((\d+)\)", t)
                    if m:
                        n = int(m.group(1))
                        pend = pend[len(pend) - n:] if n else ()
                elif op in ("ds_read_b128", "ds_read_b64_tr_b16") and from_asm:
                    dst, addr = t.split(None, 1)[1].split(",")[:2]
                    if any(p & _vregs(addr) for p in pend):
                        raise RuntimeError(f"ns_gemm.hip: line {line_no} of the listing reads LDS through a pending register: {t}")
                    pend = pend + (_vregs(dst),)
                    nreads += 1
                elif op == "s_endpgm":
                    break
                elif op == "s_branch":
                    pc = labels[t.split()[1]]
                    continue
                else:
                    if op.startswith("s_cbranch"):
                        stack.append((labels[t.split()[1]], pend))
                    elif pend and any(p & _vregs(t) for p in pend):
                        raise RuntimeError(
                            f"ns_gemm.hip: line {line_no} of the listing touches a fragment register whose LDS read "
                            f"is still in flight: {t}")
                pc += 1
    if nreads == 0:
        raise RuntimeError("check_fragment_waits: the listing holds no inline-assembly fragment reads")
    return nreads


def check_store_data(asm_text: str) -> int:
    """No vector instruction may overwrite a data register of a buffer, global or flat store of more than 8 bytes
    within two wait states of it: the store still reads that register for its last lanes.  The compiler
    leaves out those wait states after a buffer store with a scalar offset.  A vector instruction writes its first
    operand, a swap both.  Raises if the listing holds such a pair; returns the number of stores looked at."""
    code = [t for t in (l.split(";")[0].strip() for l in asm_text.split("\n")) if t and not t.startswith(".") and not t.endswith(":")]
    nstores = 0
    for i, t in enumerate(code):
        m = re.match(r"(buffer|global|flat)_store_dwordx[34]\s+(.*)", t)
        if not m:
            continue
        nstores += 1
        data = _vregs(m.group(2).split(",")[0 if m.group(1) == "buffer" else 1])
        states = 0
        for u in code[i + 1:i + 3]:
            if states >= 2 or u.startswith("s_endpgm"):
                break
            op, _, args = u.partition(" ")
            written = args if re.match(r"v_(permlane\d+_)?swap", op) else args.split(",")[0]
            if op.startswith("v_") and _vregs(written) & data:
                raise RuntimeError(f"ns_gemm.hip: '{u}' overwrites the data of '{t}' while it is read")
            states += int(args) + 1 if op == "s_nop" else 1
    return nstores


def build(verbose: bool = True, check: bool = True) -> str:
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    tmp = OUT + ".tmp"
    with tempfile.TemporaryDirectory() as d:
        objects = [os.path.join(d, src + ".o") for src in SOURCES]
        compile_flags = [f for f in FLAGS if f != "-shared"]
        cmds = [[hipcc, *compile_flags, *SOURCE_FLAGS.get(src, []), "-c", os.path.join(CSRC, src), "-o", obj]
                for src, obj in zip(SOURCES, objects)]
        if verbose:
            print("\n".join(" ".join(c) for c in cmds), flush=True)
        procs = [subprocess.Popen(c, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True) for c in cmds]
        outputs = [p.communicate()[0] for p in procs]
        if not any(p.returncode for p in procs):
            link = subprocess.run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objects, "-o", tmp], capture_output=True, text=True)
            procs, outputs = [link], [link.stdout + link.stderr]
        if any(p.returncode for p in procs):
            sys.stderr.write("".join(outputs))
            raise RuntimeError("hipcc failed building libmuon_amd.so")
    if check:
        with tempfile.TemporaryDirectory() as d:
            listing = os.path.join(d, "ns_gemm.s")
            flags = [f for f in FLAGS if f not in ("-shared", "-fPIC")]
            cmd = [hipcc, *flags, *SOURCE_FLAGS["ns_gemm.hip"], "-S", "--cuda-device-only", os.path.join(CSRC, "ns_gemm.hip"), "-o", listing]
            proc = subprocess.run(cmd, capture_output=True, text=True)
            if proc.returncode != 0:
                sys.stderr.write(proc.stdout + proc.stderr)
                raise RuntimeError("hipcc failed writing the assembly listing of ns_gemm.hip")
            text = open(listing).read()
            n = check_fragment_waits(text)
            check_store_data(text)
            if verbose:
                print(f"ns_gemm.hip: {n} hand-waited fragment reads followed through the listing, none touched early", flush=True)
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    print(build())

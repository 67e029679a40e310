"""Builds libdflash_hip.so (hand-written HIP for gfx950) in-tree with hipcc."""
from __future__ import annotations

import glob
import importlib.util
import os
import re
import subprocess
import sys
import tempfile

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
LIB_PATH = os.path.join(PKG_DIR, "libdflash_hip.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the first 64 bytes of a kernel's arguments arrive in scalar registers with the wave instead of through scalar
    # loads it has to wait for at its start (measured on the 40-layer verify: 3.53 -> 3.48 ms, nine dependent kernels a layer)
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-Wall", "-Wno-unused-function",
]


# Kernels that keep loads in flight across many instructions with hand-placed s_waitcnt (the loads are inline asm, so
# the compiler does not know their destination registers are still being filled).  If register pressure makes the
# compiler spill, it can save such a register to scratch BEFORE its data has arrived and restore the stale value
# later: silently wrong activations or weights.  The build therefore refuses any of them that uses scratch at all; so it does where
# the loads go to LDS and only the waits are placed by hand (a spill's own loads and stores would be counted among them).
NO_SCRATCH_BY_FILE = {
    "gemm_fewrow.hip": ("gemm_q4k_stream_kernel", "gemm_q4k_slab_kernel", "gemm_q4k_tiled_kernel", "gemm_q4k_experts_kernel",
                        "gemm_q4k_few_slots_kernel", "gemm_q6k_stream_kernel"),
    "gemm_whole.hip": ("gemm_q6t_loop_kernel", "gemm_q4k_wide_kernel"),
    "attn_verify.hip": ("attn_split_kernel", "attn_split_rope_kernel", "attn_rows_kernel", "attn_rows_pair_kernel"),
    "gemm_rows.hip": ("gemm_rows_kernel",),
    "gemm_dense.hip": ("gemm_q4k_dense_pair_kernel",),
}
NO_SCRATCH_KERNELS = tuple(k for kernels in NO_SCRATCH_BY_FILE.values() for k in kernels)
# Inspected exceptions, by mangled-name fragment -> spilled VGPRs: none at present.  An entry belongs here only after
# the generated code has been read and every spill store found to precede the kernel's first asm load; any other
# count than the recorded one fails the build, so that the code is read again when it changes.
INSPECTED_SPILLS = {}
# Files whose generated code is checked for a register that is touched while a load still fills it (inflight.py): reads from
# LDS in all of their kernels, loads from memory in the kernels named (the others count theirs at run time).
CHECKED_CODE = {"gemm_rows.hip": ("gemm_rows_kernel",), "attn_verify.hip": ("attn_rows_pair_kernel",), "gemm_fewrow.hip": ("gemm_q4k_few_slots_kernel",),
                "gemm_whole.hip": ("gemm_q6t_loop_kernel",), "gemm_dense.hip": ()}
RESOURCE_FLAG = "-Rpass-analysis=kernel-resource-usage"
REMARK = r"remark: (?:\S+:\d+:\d+: )?\s*"  # (the place stands ahead of the word, or behind it where the assembly is kept)


def check_no_scratch(compiler_output: str, expect=NO_SCRATCH_KERNELS) -> list:
    """Complaints about the guarded kernels in one compiler run: a kernel that spills VGPRs or has a scratch frame, and
    - so that the guard cannot pass vacuously when the remark format changes or the flag is dropped - a guarded kernel
    (of ``expect``) that the resource-usage remarks do not report at all.  This covers spills only; a plain
    register copy of an asm load's output ahead of the hand-placed wait is the same hazard without a spill: CHECKED_CODE
    covers that, and for the asm loads whose waits are counted at run time the bit-exact GEMM tests are the backstop."""
    bad, name, seen = [], None, set()
    for line in compiler_output.splitlines():
        m = re.search(REMARK + r"Function Name: (\S+)", line)
        if m:
            name = m.group(1)
            seen.update(k for k in NO_SCRATCH_KERNELS if k in name)
            continue
        guarded = name and any(k in name for k in NO_SCRATCH_KERNELS)
        m = re.search(REMARK + r"VGPRs Spill: (\d+)", line)
        if m and guarded:
            allowed = next((n for frag, n in INSPECTED_SPILLS.items() if frag in name), 0)
            if int(m.group(1)) != allowed:
                bad.append(f"{name}: {m.group(1)} VGPRs spilled (inspected: {allowed})")
        m = re.search(REMARK + r"ScratchSize \[bytes/lane\]: (\d+)", line)
        if m and guarded and int(m.group(1)) != 0 and not any(frag in name for frag in INSPECTED_SPILLS):
            bad.append(f"{name}: {m.group(1)} bytes of scratch per lane")
    bad += [f"{k}: no resource-usage remark found (is {RESOURCE_FLAG} still passed, has the remark format changed?)"
            for k in expect if k not in seen]
    return bad


def strip_remarks(compiler_output: str) -> str:
    """The compiler's text without the resource-usage remarks (with the source line and caret quoted below, if they are) and
    the packed-fp32 notice."""
    out, quoted = [], False
    for line in compiler_output.splitlines():
        if RESOURCE_FLAG in line:
            quoted = True
            continue
        quoted = quoted and re.match(r"\s*\d*\s*\|", line) is not None
        if quoted:
            continue
        if "packed-fp32-ops" in line or re.fullmatch(r"\d+ warnings? generated.*", line.strip()):
            continue
        out.append(line)
    return "\n".join(out)


def sources():
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")))


def is_stale() -> bool:
    if not os.path.exists(LIB_PATH):
        return True
    t = os.path.getmtime(LIB_PATH)
    deps = sources() + glob.glob(os.path.join(CSRC, "*.h")) + \
        glob.glob(os.path.join(PKG_DIR, "..", "include", "*.h"))
    return any(os.path.getmtime(d) > t for d in deps)


def check_code(src: str, folder: str) -> list:
    """Complaints about the device assembly that the compiler has left in ``folder`` for a file of CHECKED_CODE."""
    spec = importlib.util.spec_from_file_location("_dflash_inflight", os.path.join(PKG_DIR, "inflight.py"))
    inflight = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(inflight)
    name = os.path.basename(src)
    path = os.path.join(folder, name[:-4] + "-hip-amdgcn-amd-amdhsa-gfx950.s")
    if not os.path.exists(path):
        return [f"{name}: no device assembly at {os.path.basename(path)}"]
    with open(path) as f:
        return inflight.check_assembly(f.read(), CHECKED_CODE[name])


def build(verbose: bool = False) -> str:
    """Compile every HIP source into one shared library; always recompiles."""
    with tempfile.TemporaryDirectory() as folder:
        return _build(folder, verbose)


def _build(folder: str, verbose: bool) -> str:
    objs = []
    procs = []
    for src in sources():
        obj = src[:-4] + ".o"
        cmd = [HIPCC] + [f for f in FLAGS if f != "-shared"] + [RESOURCE_FLAG, "-c", src, "-o", obj]
        if os.path.basename(src) in CHECKED_CODE:
            cmd.append("-save-temps=cwd")  # (the device assembly; the code is the same)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, cwd=folder)))
        objs.append(obj)
    failed = False
    for src, p in procs:
        raw, _ = p.communicate()
        out = strip_remarks(raw)
        if p.returncode != 0:
            failed = True
            sys.stderr.write(f"hipcc failed for {src}:\n{out}\n")
            continue
        # (a guarded kernel's absence from the remarks is a failure in the file it lives in)
        bad = check_no_scratch(raw, NO_SCRATCH_BY_FILE.get(os.path.basename(src), ()))
        if bad:
            failed = True
            sys.stderr.write(f"{src}: kernels with loads in flight must not use scratch:\n  " + "\n  ".join(bad) + "\n")
        if os.path.basename(src) in CHECKED_CODE:
            bad = check_code(src, folder)
            if bad:
                failed = True
                sys.stderr.write(f"{src}: registers touched while a load still fills them:\n  " + "\n  ".join(bad[:40]) + "\n")
        if verbose and out.strip():
            sys.stderr.write(out + "\n")
    if failed:
        raise RuntimeError("hipcc compilation failed")
    link = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc", "-o", LIB_PATH] + objs
    r = subprocess.run(link, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout)
        raise RuntimeError("hipcc link failed")
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True))

"""Build libcornserve_amd.so (the C-ABI kernel library) in-tree with hipcc for gfx950, and libcornserve_amd_torch.so
(host code: native implementations of torch operators over that ABI) with g++.

Usage: ``python -m cornserve_amd.build`` or ``cornserve_amd.build.build_library()``.  The library is
written next to the sources so that it travels with the tree; nothing is JIT-compiled at import.
"""

from __future__ import annotations

import os
import re
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
INCLUDE = PKG_DIR.parent / "include"
LIB_PATH = PKG_DIR / "libcornserve_amd.so"
TORCH_LIB_PATH = PKG_DIR / "libcornserve_amd_torch.so"
OBJ_DIR = CSRC / "build"

ARCH = "gfx950"
# Packed-FP32 instructions are disabled for every device translation unit (see the project notes on
# v_pk_*_f32); the host pass prints a harmless "not a recognized feature" note for the same flag.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{INCLUDE}",
    f"-I{CSRC}",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; cannot build libcornserve_amd.so")
    return exe


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(line for line in proc.stdout.splitlines() if "packed-fp32-ops" not in line and "--hip-link" not in line)
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{out}")
    if out.strip():
        print(out, file=sys.stderr)


# Sources with this marker keep their accumulators in accumulation registers that only inline assembly
# touches; the compiler does not know they are occupied, so its output is checked after every build.
HAND_MANAGED_ACC_MARKER = "CS_ALL_ACC_REGS"
_ACC_REG = re.compile(r"\ba(\d+|\[)")


def check_hand_managed_acc_registers(asm_text: str) -> list[str]:
    """Return the kernels that use inline-assembly accumulation registers AND in which compiler-generated
    code touches an accumulation register too (a register spill or a staging copy would corrupt the
    accumulators).  An empty list means the convention holds."""
    offenders = []
    for m in re.finditer(r"^(_Z\S+):.*?s_endpgm", asm_text, re.S | re.M):
        in_asm, uses_inline, outside = False, False, 0
        for line in m.group(0).splitlines():
            if "#ASMSTART" in line:
                in_asm = True
                continue
            if "#ASMEND" in line:
                in_asm = False
                continue
            code = line.split(";")[0]
            if _ACC_REG.search(code):
                if in_asm:
                    uses_inline = True
                else:
                    outside += 1
        if uses_inline and outside:
            offenders.append(f"{m.group(1)}: {outside} compiler-generated accumulation-register references")
    return offenders


def _compile_checked(hipcc: str, src: Path, obj: Path) -> None:
    """Compile a source with hand-managed accumulation registers; its object appears only once the assembly that it was made
    from, which the same compilation leaves behind, has passed the check (a second compilation for the listing doubles the
    time of a build: 29 minutes of CPU time against 13)."""
    tmp = OBJ_DIR / (src.stem + ".tmp")
    shutil.rmtree(tmp, ignore_errors=True)
    tmp.mkdir()
    try:
        _run([hipcc, *HIPCC_FLAGS, "-save-temps=obj", "-c", str(src), "-o", str(tmp / obj.name)])
        listing = next(tmp.glob(f"*{ARCH}.s"), None)
        if listing is None:   # (a compiler that keeps no listing)
            listing = tmp / (src.stem + f".{ARCH}.s")
            _run([hipcc, *HIPCC_FLAGS, "-S", "--cuda-device-only", str(src), "-o", str(listing)])
        offenders = check_hand_managed_acc_registers(listing.read_text())
        if offenders:
            raise RuntimeError(f"{src.name}: the compiler used accumulation registers that inline assembly owns:\n  "
                               + "\n  ".join(offenders))
        os.replace(tmp / obj.name, obj)
    finally:
        shutil.rmtree(tmp, ignore_errors=True)


def _check_no_missing_kernels(lib: Path) -> None:
    """A shared library links with undefined symbols; a kernel whose host-side launch stub the compiler
    dropped would only show up as a load error on the GPU box.  Every undefined symbol must be external
    (HIP runtime, libc/libstdc++): none may come from this library's own (anonymous) namespaces."""
    nm = shutil.which("nm")
    if nm is None:
        return
    out = subprocess.run([nm, "-D", "--undefined-only", str(lib)], stdout=subprocess.PIPE, text=True).stdout
    own = [line.split()[-1] for line in out.splitlines() if "GLOBAL__N" in line or " cs_" in line]
    if own:
        raise RuntimeError(f"{lib.name} has undefined symbols of its own (dropped kernels?):\n  " + "\n  ".join(own))


def _build_torch_ops() -> None:
    import torch

    root = Path(torch.__file__).resolve().parent
    gxx = shutil.which("g++")
    if gxx is None:
        raise RuntimeError("g++ not found; cannot build libcornserve_amd_torch.so")
    system = [root / "include", root / "include/torch/csrc/api/include", "/opt/rocm/include", sysconfig.get_paths()["include"]]
    _run([gxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}", f"-I{INCLUDE}",
          *(arg for d in system for arg in ("-isystem", str(d))), str(CSRC / "torch_ops.cpp"), "-o", str(TORCH_LIB_PATH),
          f"-L{PKG_DIR}", f"-l:{LIB_PATH.name}", f"-L{root / 'lib'}", "-ltorch_cpu", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"])


def build_library(force: bool = True, jobs: int = 8) -> Path:
    """Compile every .hip source under csrc/ and link the shared library. Returns its path."""
    hipcc = _hipcc()
    OBJ_DIR.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    headers = list(CSRC.glob("*.h")) + list(INCLUDE.glob("*.h"))
    newest_hdr = max(h.stat().st_mtime for h in headers)
    objs, stale_objs = [], []
    todo = []
    for src in sources:
        obj = OBJ_DIR / (src.stem + ".o")
        objs.append(obj)
        stale = force or not obj.exists() or obj.stat().st_mtime < max(src.stat().st_mtime, newest_hdr)
        if stale:
            stale_objs.append(obj)
            if HAND_MANAGED_ACC_MARKER in src.read_text():
                todo.append(lambda src=src, obj=obj: _compile_checked(hipcc, src, obj))
            else:
                todo.append(lambda cmd=[hipcc, *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)]: _run(cmd))
    try:
        with ThreadPoolExecutor(max_workers=max(1, min(jobs, len(todo) or 1))) as pool:
            list(pool.map(lambda job: job(), todo))
    except BaseException:   # (here every job has ended) no later incremental build may link what was not checked
        for obj in stale_objs:
            obj.unlink(missing_ok=True)
        raise
    TORCH_LIB_PATH.unlink(missing_ok=True)   # (an older one must not stay beside the new kernel library if its own step fails)
    _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(LIB_PATH), *map(str, objs)])
    _check_no_missing_kernels(LIB_PATH)
    _build_torch_ops()
    return LIB_PATH


if __name__ == "__main__":
    incremental = "--incremental" in sys.argv
    print(build_library(force=not incremental))

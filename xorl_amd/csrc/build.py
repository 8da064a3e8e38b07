"""Compile the HIP sources in this directory into xorl_amd/lib/libxq_hip.so (gfx950), and the host path of the modules
(xq_torch.cpp, host code against torch's C++ API) into xorl_amd/lib/xq_torch.so."""

from __future__ import annotations

import glob
import os
import re
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_DIR = os.path.join(os.path.dirname(HERE), "lib")
OBJ_DIR = os.path.join(HERE, "_obj")
SO_PATH = os.path.join(LIB_DIR, "libxq_hip.so")
TORCH_SO_PATH = os.path.join(LIB_DIR, "xq_torch.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    # packed fp32 VALU forms are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the first 16 dwords of a kernel's scalar arguments arrive in registers with the wave (where the platform does it)
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-Wall", "-Wno-unused-function",
    "-Rpass-analysis=kernel-resource-usage",
]


def kernels_in(text: str) -> list[str]:
    """Names of the __global__ functions of a source, whatever their attributes and parameters."""
    text = re.sub(r"//[^\n]*|/\*.*?\*/", "", text, flags=re.S)
    text = re.sub(r"\b__launch_bounds__\s*\((?:[^()]|\([^()]*\))*\)|\b__attribute__\s*\(\((?:[^()]|\([^()]*\))*\)\)", "", text)
    names = re.findall(r"\b__global__\s+(?:\w+\s+)*?void\s+(\w+)\s*\(", text)
    if len(names) != len(re.findall(r"\b__global__\b", text)):
        raise RuntimeError(f"__global__ functions whose names are not found beside {names}")
    return names


def kernels_with(statement: str) -> list[str]:
    """Names of the kernels in files that have such an inline assembly statement (a pattern of its text)."""
    names = []
    for path in sorted(glob.glob(os.path.join(HERE, "*.h")) + glob.glob(os.path.join(HERE, "*.hip"))):
        with open(path) as f:
            text = f.read()
        if re.search(r'asm volatile\("' + statement, text):
            here = kernels_in(text)
            if not here:
                raise RuntimeError(f"{path}: inline assembly that is checked by kernel, and no kernel")
            names += here
    return names


def asm_read_kernels() -> list[str]:
    """Names of the kernels in files that read LDS into registers from inline assembly with waits of their own.  The compiler takes
    such a register as written at once: a spill before the wait would store what it held before."""
    return kernels_with("ds_read")


def asm_m0_kernels() -> list[str]:
    """Names of the kernels in files whose direct-to-LDS loads are assembly statements that take M0 as another statement left it."""
    return kernels_with("global_load_lds")


def check_m0(assembly: str, guarded: list[str]) -> None:
    """Raise if the compiler uses M0 by itself in one of the guarded kernels, by its assembly."""
    for name, body in re.findall(r"^(_Z\w+):(.*?)^\s*\.size\s+\1,", assembly, re.S | re.M):
        kernel = next((k for k in guarded if re.search(rf"\d{k}(?![a-z])", name)), None)
        if not kernel:
            continue
        own = re.sub(r";[^\n]*", "", re.sub(r";\s*#?ASMSTART.*?;\s*#?ASMEND", "", body, flags=re.S))
        use = re.search(r"^.*\bm0\b.*$", own, re.M)
        if use:
            raise RuntimeError(f"{name}: {use[0].strip()} beside loads that expect M0 as {kernel} left it")


def check_scratch(remarks: str, guarded: list[str]) -> None:
    """Raise if one of the guarded kernels uses scratch memory, by the compiler's resource remarks."""
    for name, usage in re.findall(r"Function Name: (\S+)(.*?)(?=Function Name: |\Z)", remarks, re.S):
        kernel = next((k for k in guarded if re.search(rf"\d{k}(?![a-z])", name)), None)
        scratch = re.search(r"ScratchSize \[bytes/lane\]: (\d+)", usage)
        if kernel and (scratch is None or int(scratch[1])):
            raise RuntimeError(f"{name}: {scratch[1] if scratch else 'unknown'} bytes of scratch a lane; {kernel} reads LDS from inline "
                               "assembly and may not spill")


def _split_remarks(text: str) -> tuple[str, str]:
    """(the resource remarks, everything else) of a compiler's output; a remark's place of inclusion and excerpt of the source are dropped"""
    remarks, rest, included, excerpt = [], [], [], False
    for line in text.splitlines():
        if line.startswith("In file included from"):
            included.append(line)
        elif "[-Rpass-analysis=kernel-resource-usage]" in line:
            remarks.append(line)
            included, excerpt = [], True
        elif not (excerpt and re.match(r"\s*\d* \| ", line)):
            if "is not a recognized feature for this target" not in line:
                rest += [*included, line]
            included, excerpt = [], False
    return "\n".join(remarks), "\n".join(rest)


def _compile(src: str, force: bool) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src).replace(".hip", ".o"))
    deps = [src] + glob.glob(os.path.join(HERE, "*.h")) + glob.glob(os.path.join(HERE, "..", "..", "include", "*.h"))
    if not force and os.path.exists(obj) and all(os.path.getmtime(obj) >= os.path.getmtime(d) for d in deps):
        return obj
    cmd = [HIPCC, *FLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    remarks, err = _split_remarks(r.stderr)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    try:
        check_scratch(remarks, asm_read_kernels())
        m0 = asm_m0_kernels()
        if any(re.search(rf"\d{k}(?![a-z])", remarks) for k in m0):
            listing = obj[:-2] + ".s"
            r = subprocess.run([HIPCC, *FLAGS, "--cuda-device-only", "-S", src, "-o", listing], capture_output=True, text=True)
            if r.returncode != 0:
                raise RuntimeError(f"hipcc -S failed for {src}:\n{_split_remarks(r.stderr)[1]}")
            with open(listing) as f:
                check_m0(f.read(), m0)
    except RuntimeError:
        os.remove(obj)
        raise
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _build_torch(force: bool) -> None:
    """xq_torch.so: a CPython extension linked to torch and, beside it, to libxq_hip.so."""
    src, hdr = os.path.join(HERE, "xq_torch.cpp"), os.path.join(HERE, "..", "..", "include", "xq.h")
    if not force and os.path.exists(TORCH_SO_PATH) and all(os.path.getmtime(TORCH_SO_PATH) >= os.path.getmtime(d) for d in (src, hdr)):
        return
    import torch

    t = os.path.dirname(torch.__file__)
    rocm = os.path.dirname(os.path.dirname(HIPCC))
    includes = [os.path.join(t, "include"), os.path.join(t, "include", "torch", "csrc", "api", "include"),
                os.path.join(rocm, "include"), sysconfig.get_paths()["include"]]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wno-unused-parameter", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *[f for i in includes for f in ("-isystem", i)], src, "-o", TORCH_SO_PATH, f"-L{os.path.join(t, 'lib')}",
           "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip", f"-L{LIB_DIR}", "-lxq_hip",
           "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for {src}:\n{r.stderr}")
    if r.stderr.strip():
        sys.stderr.write(r.stderr)


def build(force: bool = False, jobs: int = 8) -> str:
    os.makedirs(LIB_DIR, exist_ok=True)
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(HERE, "*.hip")))
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(lambda s: _compile(s, force), srcs))
    if force or not os.path.exists(SO_PATH) or any(os.path.getmtime(o) > os.path.getmtime(SO_PATH) for o in objs):
        r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", SO_PATH, *objs],
                           capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{r.stderr}")
    _build_torch(force)
    return SO_PATH


if __name__ == "__main__":
    print(build(force="--force" in sys.argv))

"""Compiles the HIP sources under based_amd/csrc into based_amd/libbased_hip.so for gfx950.

Usage:  python -m based_amd.build          (cross-compiles; no GPU needed)
"""
from __future__ import annotations

import concurrent.futures as cf
import glob
import hashlib
import json
import os
import re
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
OBJDIR = os.path.join(CSRC, "build")
LIB = os.path.join(HERE, "libbased_hip.so")
BINDING = os.path.join(HERE, "_binding" + sysconfig.get_config_var("EXT_SUFFIX"))
TENSORS = os.path.join(HERE, "_tensors" + sysconfig.get_config_var("EXT_SUFFIX"))

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    "-Wall",
    "-Wno-unused-command-line-argument",
    # packed-fp32 VALU forms are disabled for all device code built here
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", INCLUDE,
    "-I", CSRC,
]


RESOURCES = os.path.join(OBJDIR, "resource_usage.json")
_REMARK = re.compile(r"remark:\s+(Function Name|VGPRs|AGPRs|VGPRs Spill|SGPRs Spill|ScratchSize \[bytes/lane\]|"
                     r"Occupancy \[waves/SIMD\]|LDS Size \[bytes/block\]):\s+(\S+)")


_SNIPPET = re.compile(r"^\s*\d*\s*\|")   # the source lines clang shows under a remark


def interface() -> int:
    """The number of include/based_hip.h that everything built of it carries (never 0)."""
    with open(os.path.join(INCLUDE, "based_hip.h"), "rb") as f:
        return int.from_bytes(hashlib.sha256(f.read()).digest()[:8], "little") >> 1 | 1


def _compile(src: str):
    """Compiles one source; returns (object file, {kernel: resource figures the compiler reports})."""
    obj = os.path.join(OBJDIR, os.path.basename(src).rsplit(".", 1)[0] + ".o")
    cmd = [HIPCC, *FLAGS, f"-DBASED_HIP_INTERFACE={interface()}LL", "-Rpass-analysis=kernel-resource-usage", "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    noise = "unknown target-feature"  # host pass does not know the gfx feature name; harmless
    usage, cur, other = {}, None, []
    for line in r.stderr.splitlines():
        m = _REMARK.search(line)
        if m:
            if m.group(1) == "Function Name":
                cur = usage.setdefault(m.group(2), {})
            elif cur is not None:
                cur[m.group(1)] = int(m.group(2))
        elif ("-Rpass-analysis" not in line and line.strip() and noise not in line and "packed-fp32-ops" not in line
              and not _SNIPPET.match(line)):
            other.append(line)
    if other:
        sys.stderr.write("\n".join(other) + "\n")
    return obj, usage


# Sources a group of models needs, for a machine that serves nothing else: `build_part`.
PARTS = {
    "streaming": ("capi", "decay_scan", "decode_linear", "experts", "gated_conv", "gated_delta", "gated_delta_chunk", "greedy", "latent_attn",
                  "prompt_linear", "rglru", "stream_norm_conv", "token_mix", "window_attn"),
}


def _link(objs, out: str) -> None:
    # linked beside its final place and moved there, so that a library that exists is whole
    tmp = f"{out}.{os.getpid()}.tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, out)


def _build_binding(out: str = BINDING, number: int | None = None, compiler: str = "g++") -> bool:
    """csrc/binding.cpp, the entry points of LIB as Python callables.  Without a compiler or Python's headers there is none, and calls go
    through ctypes."""
    if os.path.exists(out):
        os.remove(out)
    tmp = f"{out}.{os.getpid()}.tmp"
    cmd = [compiler, "-O2", "-std=c++17", "-shared", "-fPIC", "-fvisibility=hidden", "-Wall", "-I", INCLUDE, "-I", sysconfig.get_paths()["include"],
           f"-DBASED_HIP_INTERFACE={interface() if number is None else number}LL", os.path.join(CSRC, "binding.cpp"), "-L", HERE, "-l:libbased_hip.so",
           "-Wl,-rpath,$ORIGIN", "-o", tmp]
    try:
        r = subprocess.run(cmd, capture_output=True, text=True)
    except OSError as e:
        r = subprocess.CompletedProcess(cmd, 1, "", str(e))
    if r.returncode != 0:
        sys.stderr.write(f"note: no binding was built, calls go through ctypes:\n{r.stdout}{r.stderr}\n")
        return False
    os.replace(tmp, out)
    return True


def _build_tensors(out: str = TENSORS, compiler: str = "g++") -> bool:
    """csrc/tensors.cpp, against the torch that is installed.  Without a compiler or the headers there is none, and tensors are asked from Python."""
    if os.path.exists(out):
        os.remove(out)
    tmp = f"{out}.{os.getpid()}.tmp"
    try:
        import torch
        from torch.utils import cpp_extension

        headers = [x for path in cpp_extension.include_paths() for x in ("-isystem", path)]
        libraries = [x for path in cpp_extension.library_paths()[:1] for x in ("-L", path)]
        cmd = [compiler, "-O2", "-std=c++17", "-shared", "-fPIC", "-fvisibility=hidden", "-Wall", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
               *headers, "-I", sysconfig.get_paths()["include"], os.path.join(CSRC, "tensors.cpp"), *libraries, "-ltorch_python", "-ltorch_cpu", "-lc10",
               "-o", tmp]
        r = subprocess.run(cmd, capture_output=True, text=True)
    except (OSError, ImportError, AttributeError) as e:
        r = subprocess.CompletedProcess([], 1, "", str(e))
    if r.returncode != 0:
        sys.stderr.write(f"note: tensors are asked from Python:\n{r.stdout}{r.stderr}\n")
        return False
    os.replace(tmp, out)
    return True


def build_part(part: str) -> str:
    """Compiles the sources of one part into a library of its own (based_amd/_lib.py: use_part)."""
    from ._lib import part_path

    os.makedirs(OBJDIR, exist_ok=True)
    srcs = [os.path.join(CSRC, f"{name}.hip") for name in PARTS[part]]
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = [o for o, _ in ex.map(_compile, srcs)]
    out = part_path(part)
    _link(objs, out)
    return out


def build(verbose: bool = False) -> str:
    os.makedirs(OBJDIR, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    if not srcs:
        raise RuntimeError("no HIP sources found")
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        tensors = ex.submit(_build_tensors)
        done = list(ex.map(_compile, srcs))
        tensors.result()
    objs = [o for o, _ in done]
    # what the compiler says each kernel needs (registers, spills, LDS): kept beside the objects; a
    # kernel that spills vector registers is named, because a few spilled registers in a loop have
    # cost a hot kernel 5 % here without any other sign
    usage = {os.path.basename(src): u for src, (_, u) in zip(srcs, done)}
    with open(RESOURCES, "w") as f:
        json.dump(usage, f, indent=1, sort_keys=True)
    for src, kernels in usage.items():
        for name, u in kernels.items():
            if u.get("VGPRs Spill", 0) > 0:
                sys.stderr.write(f"note: {src}: {name} spills {u['VGPRs Spill']} vector registers\n")
    if os.path.exists(BINDING):  # (one of a library before must not lie beside this one)
        os.remove(BINDING)
    _link(objs, LIB)
    _build_binding()
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources")
    return LIB


if __name__ == "__main__":
    build(verbose=True)

"""Build recipe for libaxon_amd.so (HIP, gfx950 only) and for _torch_ext.so, the native host side of the small
operators (plain C++ against torch's headers, linked to the former).

``build()`` always recompiles both; ``ensure_built()`` compiles only when libaxon_amd.so is missing, and
``ensure_extension_built()`` the extension alone when that is what is missing.  hipcc cross-compiles without a GPU.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import tempfile

_HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(_HERE, "csrc")
LIB_PATH = os.path.join(_HERE, "libaxon_amd.so")
EXT_PATH = os.path.join(_HERE, "_torch_ext.so")
SOURCES = ("capi.hip", "rows.hip", "loss.hip", "owned.hip", "diag.hip", "returns.hip", "cov.hip", "logits.hip", "step.hip", "lmhead.hip")

HIPCC_FLAGS = (
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    "-munsafe-fp-atomics",  # native global_atomic_add_f32 instead of a CAS loop
    # packed-fp32 VALU forms are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
)


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; libaxon_amd.so cannot be built")
    return exe


def _run(cmd, cwd) -> str:
    proc = subprocess.run(cmd, cwd=cwd, capture_output=True, text=True)
    log = "\n".join(
        line for line in (proc.stdout + proc.stderr).splitlines()
        if "is not a recognized feature" not in line  # host pass does not know the GPU feature
    )
    if proc.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed ({proc.returncode}): {' '.join(cmd)}\n{log}")
    return log


def _ext_commands(obj: str, out: str, lib_dir: str):
    """Compile and link commands of the torch extension; HIP's runtime is the one that torch brings."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths

    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    includes = [*include_paths("cuda"), sysconfig.get_paths()["include"]]
    compile_cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-w", "-D__HIP_PLATFORM_AMD__=1",
                   "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
                   "-DTORCH_EXTENSION_NAME=_torch_ext", f'-DAXON_TORCH_VERSION="{torch.__version__}"',
                   *(a for i in includes for a in ("-isystem", i)),
                   "-c", os.path.join(CSRC, "torch_ext.cpp"), "-o", obj]
    link_cmd = ["g++", "-shared", "-o", out, obj, f"-L{torch_lib}", "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu",
                "-ltorch_python", f"-L{lib_dir}", "-l:libaxon_amd.so", "-Wl,-rpath,$ORIGIN"]
    return compile_cmd, link_cmd


def build(verbose: bool = False) -> str:
    """Compile every HIP source into ``axon_amd/libaxon_amd.so`` and return its path.  One hipcc per source,
    side by side (the file with the most kernel instantiations takes a minute alone), then one link; the torch
    extension beside them."""
    from concurrent.futures import ThreadPoolExecutor

    hipcc = _hipcc()
    compile_flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    with tempfile.TemporaryDirectory(prefix="axon_amd_build_") as tmp:
        objs = [os.path.join(tmp, os.path.splitext(s)[0] + ".o") for s in SOURCES]
        cmds = [[hipcc, *compile_flags, "-c", os.path.join(CSRC, s), "-o", o] for s, o in zip(SOURCES, objs)]
        ext = os.path.join(tmp, "_torch_ext.so")
        ext_compile, ext_link = _ext_commands(os.path.join(tmp, "torch_ext.o"), ext, tmp)
        cmds.append(ext_compile)
        with ThreadPoolExecutor(max_workers=min(len(cmds), os.cpu_count() or 1, 8)) as pool:
            logs = list(pool.map(lambda c: _run(c, tmp), cmds))
        out = os.path.join(tmp, "libaxon_amd.so")
        logs.append(_run([hipcc, "--offload-arch=gfx950", "-fPIC", "-shared", "-o", out, *objs], tmp))
        logs.append(_run(ext_link, tmp))
        if verbose and any(l.strip() for l in logs):
            print("\n".join(l for l in logs if l.strip()))
        shutil.move(out, LIB_PATH)
        shutil.move(ext, EXT_PATH)
    return LIB_PATH


def ensure_built() -> str:
    if not os.path.exists(LIB_PATH):
        build()
    return LIB_PATH


def ensure_extension_built() -> str:
    """The extension beside a library that is there: g++ and torch's headers, no hipcc."""
    if not os.path.exists(EXT_PATH):
        with tempfile.TemporaryDirectory(prefix="axon_amd_build_") as tmp:
            ext = os.path.join(tmp, "_torch_ext.so")
            for cmd in _ext_commands(os.path.join(tmp, "torch_ext.o"), ext, os.path.dirname(LIB_PATH)):
                _run(cmd, tmp)
            shutil.move(ext, EXT_PATH)
    return EXT_PATH

"""Builds libfta.so (HIP kernels + C ABI) in-tree for gfx950 with hipcc.

    python flash-triangle-attention_amd/build.py [--force]

hipcc cross-compiles without a GPU, so this runs anywhere the ROCm toolchain is installed.  The extension module
fta_native.so (the C++ host path from torch tensors) is built for the torch at hand; without torch the C library and its
demo are built alone.
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
if HERE not in sys.path:
    sys.path.insert(0, HERE)

import fta_lib  # noqa: E402

CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
LIB = os.path.join(HERE, "libfta.so")
SOURCES = ["fta_api.hip", "fta_fwd.hip", "fta_fwd1.hip", "fta_fwd1_slabs.hip", "fta_fwd2.hip", "fta_fwd_feat.hip", "fta_bwd.hip", "fta_bwd_feat.hip", "fta_bwd_dq1.hip", "fta_bwd_dq1_bf16.hip",
           "fta_bwd_dkdv1.hip", "fta_bwd_dkdv1_bf16.hip", "fta_bwd_short.hip", "fta_block.hip"]

DEMO_SOURCE = "fta_c_demo.cpp"
DEMO = os.path.join(HERE, "fta_c_demo")

# the C++ host path between torch and the library: a Python extension module
NATIVE_SOURCE = "fta_torch.cpp"
NATIVE = os.path.join(HERE, "fta_native.so")

OBJDIR = os.path.join(HERE, "build")

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # packed fp32 VALU forms are kept off for every device translation unit
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-inline-asm",
]


def torch_version() -> "str | None":
    try:
        import torch
    except ImportError:
        return None
    return torch.__version__


def needs_build() -> bool:
    version = torch_version()
    built = [LIB, DEMO] + ([NATIVE] if version is not None else [])
    if not all(os.path.exists(f) for f in built) or (version is not None and fta_lib.native_torch_version(NATIVE) != version):
        return True
    t = min(os.path.getmtime(f) for f in built)
    deps = [os.path.join(CSRC, f) for f in os.listdir(CSRC)] + [os.path.join(INCLUDE, "fta.h")]
    return any(os.path.getmtime(d) > t for d in deps)


def native_commands(hipcc: str, obj: str) -> "tuple[list, list] | None":
    """Compile and link commands of the extension module (host code only); None without torch."""
    import sysconfig

    if torch_version() is None:
        return None
    import torch
    root = os.path.dirname(torch.__file__)
    inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
           sysconfig.get_paths()["include"], os.path.join(os.path.dirname(os.path.dirname(hipcc)), "include"), INCLUDE]
    compile_cmd = [hipcc, "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=fta_native",
                   f'-DFTA_TORCH_VERSION="{torch.__version__}"', f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-Wno-everything"]
    for d in inc:
        compile_cmd += ["-I", d]
    compile_cmd += ["-c", os.path.join(CSRC, NATIVE_SOURCE), "-o", obj]
    lib = os.path.join(root, "lib")
    link_cmd = [os.environ.get("CXX", "g++"), "-shared", "-o", NATIVE, obj, "-L", HERE, "-lfta", "-L", lib, "-lc10", "-lc10_hip", "-ltorch",
                "-ltorch_cpu", "-ltorch_hip", "-ltorch_python", "-Wl,-rpath,$ORIGIN", "-Wl,--no-as-needed"]
    return compile_cmd, link_cmd


def build(force: bool = True, verbose: bool = False) -> str:
    if not force and not needs_build():
        return LIB
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    # one object per source, compiled side by side (each is an independent hipcc run), then one link
    os.makedirs(OBJDIR, exist_ok=True)
    objs = [os.path.join(OBJDIR, os.path.splitext(s)[0] + ".o") for s in SOURCES]
    cmds = [[hipcc] + FLAGS + ["-I", INCLUDE, "-I", CSRC, "-c", os.path.join(CSRC, s), "-o", o] for s, o in zip(SOURCES, objs)]
    if verbose:
        for c in cmds:
            print(" ".join(c))
    native_obj = os.path.join(OBJDIR, "fta_torch.o")
    native = native_commands(hipcc, native_obj)
    if native is not None:
        cmds.append(native[0])
    else:
        print("no torch: building libfta.so and the demo without fta_native.so", file=sys.stderr)
    procs = [subprocess.Popen(c, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True) for c in cmds]
    failed = False
    for pr in procs:
        out, _ = pr.communicate()
        if pr.returncode != 0:
            sys.stderr.write(out)
            failed = True
    if failed:
        raise RuntimeError("hipcc failed compiling libfta.so")
    link = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs
    if verbose:
        print(" ".join(link))
    res = subprocess.run(link, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError("hipcc failed linking libfta.so")
    if native is not None:
        res = subprocess.run(native[1], capture_output=True, text=True)
        if res.returncode != 0:
            sys.stderr.write(res.stdout + res.stderr)
            raise RuntimeError("linking fta_native.so failed")
    # the C-ABI demo: a plain C++ program (HIP runtime only) linked against the library next to it
    demo = [hipcc, "--offload-arch=gfx950", "-O2", "-std=c++17", "-Wno-unused-command-line-argument", "-I", INCLUDE,
            os.path.join(CSRC, DEMO_SOURCE), "-o", DEMO, "-L", HERE, "-lfta", "-Wl,-rpath,$ORIGIN"]
    if verbose:
        print(" ".join(demo))
    res = subprocess.run(demo, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError("hipcc failed building fta_c_demo")
    return LIB


if __name__ == "__main__":
    print(build(force=True, verbose=True))

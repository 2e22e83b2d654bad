"""Compiles the HIP sources under csrc/ into libchop_costvol.so (gfx950 only) and the host path
between it and torch into _chop_torch.so.

Run as ``python -m custom_helper_op_amd.build``.  hipcc cross-compiles without a GPU.
Flags that are part of the numerical contract:
  -ffp-contract=off   no implicit multiply-add fusion (coordinates must be bit-exact);
  -packed-fp32-ops disabled, so the compiler emits no packed fp32 arithmetic.
"""
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libchop_costvol.so")
TORCH_LIB = os.path.join(HERE, "_chop_torch.so")
SOURCES = ["tiled_f32_fwd_wide.hip", "tiled_f32_bwd_wide.hip", "tiled_f32_fwd_narrow.hip",
           "tiled_f32_bwd_narrow.hip", "tiled_f16_fwd.hip", "tiled_f16_bwd.hip",
           "tiled_bf16_fwd.hip", "tiled_bf16_bwd.hip", "api.hip", "general.hip", "v3_feature.hip",
           "epilogue.hip", "strip.hip", "tiled_f64_fwd_wide.hip", "tiled_f64_bwd_wide.hip",
           "tiled_f64_fwd_narrow.hip", "tiled_f64_bwd_narrow.hip"]
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-ffp-contract=off", "-fno-fast-math",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-attributes",
]


def torch_module_commands():
    """(compile, link) of csrc/torch_ops.cpp: plain host C++ against torch's headers."""
    import torch
    from torch.utils import cpp_extension
    obj = os.path.join(CSRC, "torch_ops.o")
    include = cpp_extension.include_paths(device_type="cuda") + [sysconfig.get_path("include")]
    compile_ = ["g++", "-O2", "-std=c++17", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI,
                *[x for p in include for x in ("-isystem", p)],
                "-c", os.path.join(CSRC, "torch_ops.cpp"), "-o", obj]
    link = ["g++", "-shared", obj, "-o", TORCH_LIB, "-L" + HERE, "-l:" + os.path.basename(LIB),
            *["-L" + p for p in cpp_extension.library_paths(device_type="cuda")],
            "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    return compile_, link


def build(verbose=False, extra=()):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objs = []
    procs = []
    for src in SOURCES:
        obj = os.path.join(CSRC, src.replace(".hip", ".o"))
        cmd = [hipcc, *[f for f in FLAGS if f != "-shared"], *extra, "-c",
               os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
        objs.append(obj)
    compile_torch, link_torch = torch_module_commands()
    if verbose:
        print(" ".join(compile_torch), flush=True)
    procs.append(("torch_ops.cpp", subprocess.Popen(compile_torch, stdout=subprocess.PIPE,
                                                    stderr=subprocess.STDOUT)))
    failed = False
    for src, p in procs:
        out = p.communicate()[0].decode()
        # the host pass warns that it does not know the packed-fp32 feature: harmless
        out = "\n".join(l for l in out.splitlines() if "packed-fp32-ops" not in l)
        if out.strip():
            print(out, flush=True)
        failed |= p.returncode != 0
    if failed:
        raise RuntimeError("compilation failed")
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", LIB]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    if verbose:
        print(" ".join(link_torch), flush=True)
    subprocess.run(link_torch, check=True)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))

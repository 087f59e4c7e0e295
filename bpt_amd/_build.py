"""Compiles the four native libraries in-tree:

  bpt_amd/csrc/libbptgraph.so  host C++ (g++)            <- bptgraph.cpp
  bpt_amd/csrc/libbptattn.so   gfx950 HIP (hipcc)        <- bptattn.hip
  bpt_amd/csrc/libbptplan.so   gfx950 HIP (hipcc)        <- bptplan.hip  (plans built on the GPU; rocPRIM headers)
  bpt_amd/csrc/bptop.so        host C++ (g++, torch)     <- bptop.cpp    (host side of the ops and their autograd; links both)

hipcc cross-compiles for gfx950 without a GPU.  Run `python -m bpt_amd._build`.
"""
import os
import subprocess
import sys

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")
GRAPH_SO = os.path.join(CSRC, "libbptgraph.so")
ATTN_SO = os.path.join(CSRC, "libbptattn.so")
PLAN_SO = os.path.join(CSRC, "libbptplan.so")
OP_SO = os.path.join(CSRC, "bptop.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
HIP_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    # packed FP32 forms (v_pk_*_f32) are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-variable", "-Wno-unused-but-set-variable",
]


# The target feature above only exists for the GPU; hipcc also hands it to its host pass, which reports it once per
# internal step with exactly this line and ignores it.  The line is dropped so that real diagnostics stand out.
_HOST_PASS_NOTE = "'-packed-fp32-ops' is not a recognized feature for this target (ignoring feature)"


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(line for line in proc.stdout.splitlines() if line.strip() != _HOST_PASS_NOTE)
    if out.strip():
        print(out, flush=True)
    if proc.returncode != 0:
        raise subprocess.CalledProcessError(proc.returncode, cmd)


def build_graph(verbose=True):
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wextra",
          os.path.join(CSRC, "bptgraph.cpp"), "-o", GRAPH_SO], verbose)
    return GRAPH_SO


def build_attn(verbose=True):
    _run([HIPCC] + HIP_FLAGS + [os.path.join(CSRC, "bptattn.hip"), "-o", ATTN_SO], verbose)
    return ATTN_SO


def build_plan(verbose=True):
    _run([HIPCC] + HIP_FLAGS + [os.path.join(CSRC, "bptplan.hip"), "-o", PLAN_SO], verbose)
    return PLAN_SO


def build_op(verbose=True):
    """After build_attn and build_plan, whose libraries it links (found beside it at run time)."""
    import sysconfig
    import torch
    from torch.utils import cpp_extension
    rocm = os.path.dirname(os.path.dirname(HIPCC))
    include = cpp_extension.include_paths() + [os.path.join(rocm, "include"), sysconfig.get_paths()["include"]]
    libs = os.path.join(os.path.dirname(torch.__file__), "lib")
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-DTORCH_EXTENSION_NAME=bptop",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM"]
         + [f"-I{p}" for p in include] + [os.path.join(CSRC, "bptop.cpp"), "-o", OP_SO, f"-L{libs}", f"-L{CSRC}",
                                          "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python", "-ltorch", "-l:libbptattn.so", "-l:libbptplan.so", "-Wl,-rpath,$ORIGIN"], verbose)
    return OP_SO


def build_all(verbose=True):
    """The HIP compilations take most of the time and run side by side."""
    from concurrent.futures import ThreadPoolExecutor
    with ThreadPoolExecutor(2) as pool:
        plan = pool.submit(build_plan, verbose)
        graph, attn = build_graph(verbose), build_attn(verbose)
        return graph, attn, plan.result(), build_op(verbose)


if __name__ == "__main__":
    build_all()
    sys.exit(0)

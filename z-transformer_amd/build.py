"""Builds libzt_attn.so for gfx950 in-tree (z-transformer_amd/_build/).

Steps: each csrc/kernels/*.hip -> a gfx950 code object (hipcc --genco); the
host launcher and holder (csrc/zt_attn.cpp, host/zt_holder.cpp) compiled with
g++ against the HIP runtime API and csrc/noalloc.hip (the fixed device scratch
of the allocation-free decode) by hipcc; then all linked into one shared
library with the code objects embedded by .incbin.  Always rebuilds.
genco / host_objects / link are also used by tests/planted/build.py.

All HIP code is compiled with packed-FP32 instructions disabled.
"""
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
BUILD = os.path.join(HERE, "_build")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
ARCH = "gfx950"
KERNELS = [("fwd", "attn_fwd.hip"), ("bwd", "attn_bwd.hip"), ("dec", "attn_decode.hip"), ("misc", "norm_rope.hip"),
           ("cal", "calibrate.hip"), ("gemm", "gemm.hip")]
HIP_FLAGS = ["-O3", "-std=c++20", f"--offload-arch={ARCH}", "-Xclang", "-target-feature", "-Xclang",
             "-packed-fp32-ops", "-Wall"]
LIB = os.path.join(BUILD, "libzt_attn.so")


def _run(cmd):
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in p.stdout.splitlines() if "packed-fp32-ops" not in l and "--hip-link" not in l)
    if p.returncode != 0:
        raise RuntimeError(f"command failed ({p.returncode}): {' '.join(cmd)}\n{out}")
    return out


def _hipcc():
    return shutil.which("hipcc") or os.path.join(ROCM, "bin", "hipcc")


def genco(src, out, defines=()):
    """One kernel source -> a gfx950 code object (written atomically)."""
    _run([_hipcc(), "--genco", *HIP_FLAGS, *[f"-D{d}" for d in defines], src, "-o", out + ".tmp"])
    os.replace(out + ".tmp", out)
    return out


def link(lib, code_objects, host_objects, embed_path):
    """Links host objects and the given code objects (tag -> path, every tag of
    KERNELS) into the shared library `lib`; the code objects are embedded with
    .incbin under the zt_co_<tag> symbols the launcher loads."""
    with open(embed_path, "w") as f:
        f.write("/* generated by build.py: the gfx950 code objects, embedded */\n")
        f.write('\t.section .rodata\n')
        for tag, _ in KERNELS:
            f.write(f"\t.global zt_co_{tag}\n\t.global zt_co_{tag}_end\n\t.balign 64\n")
            f.write(f'zt_co_{tag}:\n\t.incbin "{code_objects[tag]}"\nzt_co_{tag}_end:\n\t.byte 0\n')
        f.write('\t.section .note.GNU-stack,"",@progbits\n')
    tmp = lib + ".tmp"
    # -Bsymbolic: calls between the library's own entry points bind inside it, also
    # when several builds of it are loaded into one process (the test-only ones).
    _run(["g++", "-shared", "-fPIC", "-Wl,-Bsymbolic", *host_objects, embed_path, f"-L{ROCM}/lib", "-lamdhip64",
          f"-Wl,-rpath,{ROCM}/lib", "-o", tmp])
    os.replace(tmp, lib)
    return lib


def host_objects():
    """The launcher, the holder and the allocation-free decode's scratch, as
    position-independent objects in _build/."""
    objs = []
    for src in (os.path.join(HERE, "csrc", "zt_attn.cpp"), os.path.join(HERE, "host", "zt_holder.cpp")):
        obj = os.path.join(BUILD, os.path.basename(src).replace(".cpp", ".o"))
        _run(["g++", "-O2", "-std=c++17", "-fPIC", "-c", "-Wall", "-Wextra", "-D__HIP_PLATFORM_AMD__",
              f"-I{ROCM}/include", src, "-o", obj])
        objs.append(obj)
    # The allocation-free decode's scratch array (a __device__ global, registered
    # with the HIP runtime by hipcc's host code) and its address lookup.
    scratch_obj = os.path.join(BUILD, "noalloc.o")
    _run([_hipcc(), "-c", "-fPIC", *HIP_FLAGS, os.path.join(HERE, "csrc", "noalloc.hip"), "-o", scratch_obj])
    objs.append(scratch_obj)
    return objs


def build(verbose=False):
    os.makedirs(BUILD, exist_ok=True)
    kdir = os.path.join(HERE, "csrc", "kernels")
    with ThreadPoolExecutor(max_workers=len(KERNELS) + 1) as ex:
        cos = {tag: ex.submit(genco, os.path.join(kdir, src), os.path.join(BUILD, f"{tag}.hsaco"))
               for tag, src in KERNELS}
        objs = ex.submit(host_objects)
        cos = {tag: f.result() for tag, f in cos.items()}
        objs = objs.result()
    link(LIB, cos, objs, os.path.join(BUILD, "co_embed.S"))
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)

"""Build recipe for libfmha_decode.so (gfx950), used by __graft_entry__.build().

Compiles fmha_amd/csrc/fmha_decode_api.hip (the C ABI) and every part of
fmha_amd/csrc/fmha_decode_inst.hip (the kernel instantiations, one slice per
-DFMHA_DECODE_PART) with hipcc, in parallel, and links them into
fmha_amd/libfmha_decode.so, in tree, so the built library travels with the
source tree.  The objects go to fmha_amd/_build/.  build_host() compiles the
tensor interface's native module (fmha_amd/csrc/fmha_decode_torch.cpp, host
code only) against the installed torch into fmha_amd/_host.so.
"""
import concurrent.futures
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(HERE, "libfmha_decode.so")
CSRC = os.path.join(HERE, "csrc")
API_SOURCE = os.path.join(CSRC, "fmha_decode_api.hip")
INST_SOURCE = os.path.join(CSRC, "fmha_decode_inst.hip")
HOST_LIB = os.path.join(HERE, "_host.so")
HOST_SOURCE = os.path.join(CSRC, "fmha_decode_torch.cpp")
OBJ_DIR = os.path.join(HERE, "_build")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    # Packed-FP32 VALU forms are kept out of every build.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA results in VGPRs rather than AGPRs: the matrix-core kernel reads
    # every result with VALU instructions, which cannot take AGPR operands
    # (saves one v_accvgpr_read per value).
    "-mllvm", "-amdgpu-mfma-vgpr-form",
]


def hipcc():
    return os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def inst_parts():
    """Number of FMHA_DECODE_PART slices, as fmha_decode_inst.hip states it."""
    m = re.search(r"FMHA_DECODE_PARTS (\d+)", open(INST_SOURCE).read())
    if not m:
        raise RuntimeError("FMHA_DECODE_PARTS missing from " + INST_SOURCE)
    return int(m.group(1))


def _run(cmd):
    res = subprocess.run(cmd, capture_output=True, text=True)
    # The host pass does not know the packed-fp32 feature name and says so.
    err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
    return res.returncode, err


def build(verbose=False, jobs=None):
    """Compile and link the library; raises CalledProcessError on failure."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    for name in os.listdir(OBJ_DIR):  # objects of an earlier part count
        if name.endswith(".o"):
            os.remove(os.path.join(OBJ_DIR, name))
    inc = ["-I" + os.path.join(ROOT, "include"), "-I" + CSRC]
    units = [(API_SOURCE, [], os.path.join(OBJ_DIR, "fmha_decode_api.o"))]
    units += [(INST_SOURCE, ["-DFMHA_DECODE_PART=%d" % p], os.path.join(OBJ_DIR, "fmha_decode_inst_%d.o" % p))
              for p in range(inst_parts())]
    cmds = [[hipcc()] + HIPCC_FLAGS + inc + defs + ["-c", "-o", obj, src] for src, defs, obj in units]
    if verbose:
        print(" ".join(cmds[0]), flush=True)
        print("... and %d parts of %s" % (len(units) - 1, os.path.basename(INST_SOURCE)), flush=True)
    jobs = jobs or min(16, os.cpu_count() or 1)
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        results = list(pool.map(_run, cmds))
    failed = False
    for cmd, (rc, err) in zip(cmds, results):
        if rc != 0:
            failed = True
            sys.stderr.write(" ".join(cmd) + "\n" + err + "\n")
        elif err.strip() and verbose:
            sys.stderr.write(err + "\n")
    if failed:
        raise subprocess.CalledProcessError(1, "hipcc")
    link = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,--no-undefined", "-o", LIB + ".tmp"]
    link += [obj for _, _, obj in units]
    rc, err = _run(link)
    if rc != 0:
        sys.stderr.write(" ".join(link) + "\n" + err + "\n")
        raise subprocess.CalledProcessError(rc, link)
    os.replace(LIB + ".tmp", LIB)
    return LIB


def build_host(verbose=False):
    """Compile the native module of the tensor interface; raises
    CalledProcessError on failure."""
    import sysconfig
    import torch
    root = os.path.dirname(torch.__file__)
    rocm = os.path.dirname(os.path.dirname(hipcc()))
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI,
           "-I" + os.path.join(ROOT, "include"), "-isystem", os.path.join(root, "include"),
           "-isystem", os.path.join(rocm, "include"), "-isystem", sysconfig.get_paths()["include"],
           HOST_SOURCE, "-o", HOST_LIB + ".tmp", "-L" + os.path.join(root, "lib"),
           "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]
    if verbose:
        print(" ".join(cmd), flush=True)
    rc, err = _run(cmd)
    if rc != 0:
        sys.stderr.write(err + "\n")
        raise subprocess.CalledProcessError(rc, cmd)
    os.replace(HOST_LIB + ".tmp", HOST_LIB)
    return HOST_LIB


if __name__ == "__main__":
    print(build(verbose=True))
    print(build_host(verbose=True))

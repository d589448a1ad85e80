"""CPU checks of the code that hipcc makes of the split-KV kernels: what a
load instruction covers, and where its descriptor comes from, decides their
speed and shows only in the assembly.  A few instantiations are compiled to
gfx950 assembly with the library's own flags."""
import os
import re
import subprocess

import pytest

from fmha_amd import _build

KERNELS = (
    "splitkv_pv_kernel<256, 8, kLayoutPagedBlock, 1>",
    "splitkv_pv_kernel<256, 8, kLayoutPagedBlock, 2>",
    "splitkv_pv_kernel<128, 4, kLayoutPagedBlock, 1>",
    "splitkv_pv_kernel<256, 4, kLayoutPacked, 1>",
    "splitkv_scores_kernel<128, 4, kLayoutPacked>",
    "splitkv_scores_kernel<64, 1, kLayoutStrided>",
    "splitkv_scores_group_kernel<256, kLayoutPacked>",
)


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    """{kernel: its assembly lines}"""
    tmp = tmp_path_factory.mktemp("codegen")
    src = tmp / "kernels.hip"
    src.write_text('#include "fmha_decode_splitkv_pv.hpp"\nnamespace fmha_decode {\n' +
                   "".join("template __global__ void %s(SplitArgs);\n" % k for k in KERNELS) + "}\n")
    out = tmp / "kernels.s"
    subprocess.run([_build.hipcc(), *_build.HIPCC_FLAGS, "-I" + _build.CSRC, "-I" + os.path.join(_build.ROOT, "include"),
                    "-S", "--cuda-device-only", "-o", str(out), str(src)], check=True, capture_output=True)
    found, lines = {}, None
    for line in out.read_text().split("\n"):
        m = re.match(r"_ZN11fmha_decode\d+(\w+?)ILi(\w+?)EEEv", line)
        if m and line.split(";")[0].rstrip().endswith(":"):
            lines = found.setdefault((m.group(1), m.group(2).replace("ELi", ", ")), [])
        elif line.startswith(".Lfunc_end"):
            lines = None
        elif lines is not None:
            lines.append(line.strip())
    layouts = {"kLayoutPacked": "0", "kLayoutStrided": "1", "kLayoutPaged": "2", "kLayoutPagedBlock": "3"}
    by_name = {}
    for k in KERNELS:
        name, args = re.match(r"(\w+)<(.*)>", k).groups()
        for layout, value in sorted(layouts.items(), reverse=True):
            args = args.replace(layout, value)
        by_name[k] = found[(name, args)]
    return by_name


def test_wide_rows_are_read_in_whole_lines(listings):
    """P.V at 256 dims of one workgroup: a lane's second 16 bytes of a V row lie 256 bytes
    after its first, so that each load instruction reads 256 neighbouring
    bytes of a row (16 bytes after them, every instruction took every other
    16 bytes of 512, and every line twice)."""
    for k in KERNELS:
        if not re.match(r"splitkv_pv_kernel<256.* 1>", k):
            continue
        wide = [l for l in listings[k] if l.startswith("buffer_load_dwordx4")]
        assert wide
        assert sum(re.search(r"offset:256\b", l) is not None for l in wide) == len(wide) // 2, k
        assert not any(re.search(r"offset:16\b", l) for l in wide), k


@pytest.mark.parametrize("kernel", KERNELS)
def test_descriptors_are_scalar(listings, kernel):
    """No load goes through a loop over the lanes, which the compiler makes
    of a buffer descriptor that it holds in vector registers."""
    label, start, loops = None, 0, []
    lines = listings[kernel]
    for i, line in enumerate(lines):
        m = re.match(r"(\.LBB\w+):", line)
        if m:
            label, start = m.group(1), i
        elif label and line.startswith("s_cbranch_execnz") and label in line:
            body = lines[start:i]
            if any(l.startswith("v_readfirstlane") for l in body) and any(l.startswith("buffer_") for l in body):
                loops.append(body)
    assert not loops, "%d loops, the first:\n%s" % (len(loops), "\n".join(loops[0]))

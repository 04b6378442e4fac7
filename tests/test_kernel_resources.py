"""What the compiler made of the kernels, read from the built library's own code objects (no GPU needed):
registers kept in memory and scalars kept in the lanes of a vector register are time on the chains these
kernels are bound by, and a change far away in a kernel can bring them about."""
import os
import re
import struct
import subprocess

import pytest

from tests import capi


def _kernels():
    """{demangled name: metadata} of every kernel in the library."""
    msgpack = pytest.importorskip("msgpack")
    if not os.path.exists(capi.LIB_PATH):
        import __graft_entry__
        __graft_entry__.build()
    data = open(capi.LIB_PATH, "rb").read()
    found = {}
    # the notes of an AMDGPU code object: name size, description size, type 32 (metadata), "AMDGPU\0" padded to 8
    for m in re.finditer(re.escape(struct.pack("<I", 32) + b"AMDGPU\0\0"), data):
        size = struct.unpack_from("<I", data, m.start() - 4)[0]
        doc = msgpack.unpackb(data[m.end(): m.end() + size], strict_map_key=False)
        for k in doc["amdhsa.kernels"]:
            found[k[".name"]] = k
    names = subprocess.run(["c++filt"], input="\n".join(found), capture_output=True, text=True, check=True).stdout.split("\n")
    return {n.split("(")[0].replace("void ", ""): k for n, k in zip(names, found.values())}


def test_no_kernel_keeps_registers_in_memory():
    kernels = _kernels()
    assert len(kernels) > 100, "the library's kernels are not where they were looked for"
    bad = {n: (k[".vgpr_spill_count"], k[".private_segment_fixed_size"]) for n, k in kernels.items()
           if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}
    assert not bad, bad


@pytest.mark.parametrize("kernel,most", [("finish_kernel<1024, 8>", 4), ("finish_kernel<256, 4>", 12), ("finish_kernel<256, 8>", 12),
                                         ("finish_kernel<256, 16>", 44)])
def test_the_streaming_finish_keeps_its_scalars(kernel, most):
    """The way almost no row takes (finish_row_slow) shares the finishing kernels with the usual one, a chain of
    dependent steps.  With 36 spilled scalars in the place of 22, brought about by a change to the slow way alone, calls of
    64 rows of 152064 were 1 to 2 % slower.  Bounds: the counts when this was written (0, 5, 7 and 33) with some room."""
    k = _kernels()["rs::" + kernel]
    assert k[".sgpr_spill_count"] <= most, k[".sgpr_spill_count"]


@pytest.mark.parametrize("keep", ["false", "true"])
@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_the_pass_over_slices_of_8192_tokens_shares_a_compute_unit_six_ways(dtype, keep):
    """The library cuts rows into slices of 8192 tokens for calls of up to 1536 slices, six workgroups to each of 256
    compute units.  Six waves share a SIMD's 512 registers up to 80 each; with 82 such calls needed a second round and
    were 3 to 7 % slower (512 rows of 20480).  Calls that keep every token were 2 to 5 % slower with 79 registers than
    with 62: eight share one up to 64."""
    k = _kernels()["rs::stream_kernel<8, 256, %d, %s, false>" % (dtype, keep)]
    assert k[".vgpr_count"] <= (64 if keep == "true" else 80), k[".vgpr_count"]


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("groups", [2, 3, 4])
def test_two_workgroups_of_the_short_row_kernel_share_a_compute_unit(dtype, groups):
    """Sixteen waves and sixteen more, eight to a SIMD, have 64 of its 512 registers each.  With 66 calls of 257 to 512 rows of
    8196 to 16384 tokens were up to 40 % slower than on the path that they had been taken from."""
    k = _kernels()["rs::short_kernel<%d, false, 16, %d>" % (dtype, groups)]
    assert k[".vgpr_count"] <= 64, k[".vgpr_count"]

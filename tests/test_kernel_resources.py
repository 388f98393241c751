"""What the compiler gave the kernels, read from the metadata of the built
library's code objects: kernels whose speed rests on holding everything in
registers have no private (scratch) memory and keep the occupancy their
comments state."""
import os
import struct
import subprocess

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "chimes_calculator_amd", "lib",
                   "libchimescalc.so")


def code_objects(blob):
    at = blob.find(b"\x7fELF")
    while at >= 0:
        if struct.unpack_from("<H", blob, at + 18)[0] == 224:  # EM_AMDGPU
            yield at
        at = blob.find(b"\x7fELF", at + 4)


@pytest.fixture(scope="module")
def kernels():
    """{demangled name: metadata}"""
    blob = open(LIB, "rb").read()
    found = {}
    for o in code_objects(blob):
        phoff, = struct.unpack_from("<Q", blob, o + 0x20)
        size, count = struct.unpack_from("<HH", blob, o + 0x36)
        for p in range(o + phoff, o + phoff + size * count, size):
            if struct.unpack_from("<I", blob, p)[0] != 4:  # PT_NOTE
                continue
            q = o + struct.unpack_from("<Q", blob, p + 8)[0]
            end = q + struct.unpack_from("<Q", blob, p + 0x20)[0]
            while q < end:
                ns, ds, kind = struct.unpack_from("<III", blob, q)
                q += 12 + (ns + 3) // 4 * 4
                if kind == 32:  # NT_AMDGPU_METADATA
                    for k in msgpack.unpackb(blob[q:q + ds])["amdhsa.kernels"]:
                        found[k[".name"]] = k
                q += (ds + 3) // 4 * 4
    names = subprocess.run(["c++filt"], input="\n".join(found), capture_output=True, text=True, check=True).stdout
    return {n.split("(")[0].replace("void ", "").replace("chx::", ""): k
            for n, k in zip(names.split("\n"), found.values())}


def pick(kernels, prefix):
    got = {n: k for n, k in kernels.items() if n.startswith(prefix)}
    assert got, prefix
    return got


@pytest.mark.parametrize("prefix", ["k_lmp_pair<"])
def test_no_scratch(kernels, prefix):
    for n, k in pick(kernels, prefix).items():
        assert k[".private_segment_fixed_size"] == 0, n


@pytest.mark.parametrize("prefix", ["k_lane<", "k_eval2<"])
def test_scalar_spills(kernels, prefix):
    """The force table's probes are a loop: unrolled, each kernel that adds to
    it held the probes' execution masks in spilled scalar registers."""
    for n, k in pick(kernels, prefix).items():
        assert k[".sgpr_spill_count"] <= 2, n


def test_lane_wavefronts(kernels):
    """k_lane's registers allow the wavefronts per SIMD it is compiled for
    (512 registers a lane), with little or no scratch."""
    for n, k in pick(kernels, "k_lane<").items():
        nb, D = (int(v) for v in n[n.index("<") + 1:-1].split(","))
        waves = (4 if D <= 8 else 3 if D <= 11 else 2) if nb == 3 else (3 if D <= 3 else 2)
        assert 512 // ((k[".vgpr_count"] + 7) // 8 * 8) >= waves, n
        assert k[".private_segment_fixed_size"] <= (32 if nb == 3 and D in (8, 11) else 0), n

"""Registers and scratch of kernels in the built library, from the metadata that the compiler writes beside each: a
kernel whose waves per SIMD or whose scratch its speed depends on stays within what it was measured with."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from exl3r import _lib

msgpack = pytest.importorskip("msgpack")

BUNDLE, ELF_NOTE, AMDGPU_METADATA = b"__CLANG_OFFLOAD_BUNDLE__", 7, 32


def notes(elf):
    """The descriptors of an ELF64 image's notes, by type."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entry, count, _ = struct.unpack_from("<HHH", elf, 0x3A)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, shoff + i * entry + 4)
        at, size = struct.unpack_from("<QQ", elf, shoff + i * entry + 0x18)
        end = at + size
        while kind == ELF_NOTE and at < end:
            name, desc, note = struct.unpack_from("<III", elf, at)
            at += 12 + (name + 3) // 4 * 4
            yield note, elf[at:at + desc]
            at += (desc + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    """Demangled name -> metadata of every kernel of the product library."""
    with open(_lib.LIB_PATH, "rb") as f:
        image = f.read()
    found, at = {}, image.find(BUNDLE)
    while at >= 0:
        count, = struct.unpack_from("<Q", image, at + 24)
        p = at + 32
        for _ in range(count):
            off, size, length = struct.unpack_from("<QQQ", image, p)
            target = image[p + 24:p + 24 + length]
            p += 24 + length
            if b"gfx950" in target and size:
                for kind, desc in notes(image[at + off:at + off + size]):
                    if kind == AMDGPU_METADATA:
                        for k in msgpack.unpackb(desc, strict_map_key=False)["amdhsa.kernels"]:
                            found[k[".name"]] = k
        at = image.find(BUNDLE, at + 24)
    if not shutil.which("c++filt"):
        pytest.skip("no c++filt")
    names = sorted(found)
    out = subprocess.run(["c++filt"], input="\n".join(names), capture_output=True, text=True, check=True).stdout.split("\n")
    return {d.replace("exl3r::", ""): found[n] for d, n in zip(out, names)}


def matching(kernels, pattern):
    hits = {n: k for n, k in kernels.items() if re.search(pattern, n)}
    assert hits, pattern
    return hits


# pattern of the instances, VGPRs at most (96: 5 waves per SIMD, 80: 6, 64: 8), spilled VGPRs and scratch bytes per
# lane at most
LIMITS = [
    # argmax, four chunks of aligned logits in flight
    (r"void k_argmax(_ws)?<\w+, true, 4, false>", 96, 0, 0),
    # RoPE with the paged append: nothing in scratch
    (r"void k_rope_nx<\w+, [12], [012], \d, false, 1, true, ", 128, 0, 0),
    # bf16 GPT-J with f32 head norms from the {cos, sin} table, one and two passes per item
    (r"void k_rope_nx<TBF16, 1, 2, 2, false, 1, false, 0, 8, false, [12]>", 80, 0, 0),
    (r"void k_rope_nx<TBF16, 1, 2, 2, false, 2, false, 0, 8, false, 0>", 96, 0, 0),
    # RoPE from the {cos, sin} table with head norms, one item per wave: eight waves per SIMD
    (r"void k_rope_nx<\w+, 2, [12], 2, false, 1, false, 0, 8, false, 1>", 64, 0, 0),
    # norms of eight chunks per lane: no row of outputs held beside the row itself
    (r"void k_rms_norm<(TF16|TBF16), \w+, (TF16|TBF16), 8, 1, 0, 2, false, double>", 98, 0, 0),
    (r"void k_rms_norm<(TF16|TBF16), TF32, TF32, 8, 1, 0, 2, false, double>", 128, 6, 28),
    (r"void k_rms_norm<(TF16|TBF16), \w+, TF32, 8, 1, 0, 2, false, double>", 128, 14, 60),
    (r"void k_rms_norm<TF32, TF32, TF32, 8, 1, 0, 2, false, double>", 128, 56, 164),
    (r"void k_rms_norm<\w+, \w+, TNone, 8, 0, 0, [02], false, double>", 120, 0, 0),
]


@pytest.mark.parametrize("pattern,vgprs,spills,scratch", LIMITS)
def test_resources(kernels, pattern, vgprs, spills, scratch):
    over = {n: (k[".vgpr_count"], k[".vgpr_spill_count"], k[".private_segment_fixed_size"])
            for n, k in matching(kernels, pattern).items()
            if k[".vgpr_count"] > vgprs or k[".vgpr_spill_count"] > spills or k[".private_segment_fixed_size"] > scratch}
    assert not over, over


def test_scalar_registers_of_the_rotating_gptj_append(kernels):
    """Its scalar registers are full: what does not fit is moved to and from vector lanes in the item loop."""
    hits = matching(kernels, r"void k_rope_nx<TF16, 1, 0, 0, false, 1, true, 2, 8, false, 0>")
    assert all(k[".sgpr_spill_count"] <= 84 for k in hits.values()), {n: k[".sgpr_spill_count"] for n, k in hits.items()}

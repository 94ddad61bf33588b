"""Register budgets of the GEMM kernels, read from the built library's own metadata: a source
change that costs a kernel its wavefronts per SIMD, or makes it spill, shows here."""

import os
import re
import struct

import msgpack

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "deepseek-v4-flash-offload_amd", "dsv4_hip", "libdsv4hip.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
NT_AMDGPU_METADATA = 32


def _device_images(data):
    """The gfx950 code objects of every offload bundle in the library."""
    for m in re.finditer(MAGIC, data):
        base, p = m.start(), m.end()
        (n,) = struct.unpack_from("<Q", data, p)
        p += 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if size and name.endswith(b"gfx950"):
                yield data[base + off:base + off + size]


def _kernels():
    out = {}
    for elf in _device_images(open(LIB, "rb").read()):
        (phoff,) = struct.unpack_from("<Q", elf, 32)
        phsize, phnum = struct.unpack_from("<HH", elf, 54)
        for i in range(phnum):
            kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phsize)
            if kind != 4:  # PT_NOTE
                continue
            p = off
            while p < off + size:
                namesz, descsz, ntype = struct.unpack_from("<III", elf, p)
                desc = p + 12 + (namesz + 3) // 4 * 4
                if ntype == NT_AMDGPU_METADATA:
                    for k in msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]:
                        out[k[".name"]] = k
                p = desc + (descsz + 3) // 4 * 4
    assert out, "no kernel metadata found"
    return out


def test_pure_bf16_decode_gemms_of_a_512_reduction_keep_three_waves_per_simd():
    """moe_gemm_kernel<bf16 activations, gate/up or down, 2 stages>: 512 registers per SIMD lane over
    three wavefronts in granules of 8 leave 168 each (two wavefronts: 8 tokens' down GEMM 11.4 -> 12.6 us)."""
    found = {n: k[".vgpr_count"] for n, k in _kernels().items() if re.search(r"15moe_gemm_kernelILi2ELb[01]ELi2ELb0E", n)}
    assert len(found) == 2 and max(found.values()) <= 168, found


def test_gemm_kernels_do_not_spill():
    gemm = {n: k for n, k in _kernels().items() if "moe_gemm" in n}
    assert len(gemm) >= 50
    assert not {n for n, k in gemm.items() if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}

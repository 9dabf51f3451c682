"""Resources of the built kernels, from the metadata that the compiler leaves in libllmoe.so: no kernel keeps registers in
scratch memory (a spill in a GEMM's inner loop is traffic beside the weight stream; the group-products kernels ran 1.4 to
1.7 times as long with 304 bytes of it per lane)."""
from __future__ import annotations

import struct

import msgpack
import pytest

import llmoe

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
SHT_NOTE, NT_AMDGPU_METADATA = 7, 32


def _metadata(elf):
    shoff, = struct.unpack_from("<Q", elf, 40)
    shsize, shnum = struct.unpack_from("<HH", elf, 58)
    for i in range(shnum):
        _, kind, _, _, at, size, *_ = struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * shsize)
        end = at + size
        while kind == SHT_NOTE and at < end:
            name, desc, note = struct.unpack_from("<III", elf, at)
            d = at + 12 + -(-name // 4) * 4
            if note == NT_AMDGPU_METADATA:
                yield from msgpack.unpackb(elf[d:d + desc])["amdhsa.kernels"]
            at = d + -(-desc // 4) * 4


def _kernels(path):
    data = path.read_bytes()
    b = data.find(BUNDLE)
    while b >= 0:
        n, = struct.unpack_from("<Q", data, b + 24)
        p = b + 32
        for _ in range(n):
            off, size, name = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + name]
            p += 24 + name
            if target.endswith(b"gfx950"):
                yield from _metadata(data[b + off:b + off + size])
        b = data.find(BUNDLE, b + 1)


def test_no_kernel_uses_scratch():
    if not llmoe.LIB_PATH.exists():
        pytest.skip("libllmoe.so not built")
    k = {m[".name"]: m[".private_segment_fixed_size"] for m in _kernels(llmoe.LIB_PATH)}
    for part in ("expert_gemm_plan", "expert_gemmILi0E", "expert_gemmILi2E", "tiled_gemmILi0E", "router_mfma_kernel",
                 "select_token_kernel", "plan_kernel"):
        assert any(part in n for n in k), part
    assert {n: s for n, s in k.items() if s} == {}

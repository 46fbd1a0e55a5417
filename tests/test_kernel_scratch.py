"""The built library's own metadata: kernels for runs of rows keep what they work on in registers.  (With what a lane needs
behind the loop kept through it, or a second tile in a loop around the first, the latent prompts' kernel wrote registers
to memory: runs of 33 to 128 rows took up to 1.3 times as long.)"""
import os
import struct

import msgpack
import pytest


def kernels_of(path):
    """{kernel's name: bytes of memory a lane keeps registers in}"""
    data, found = open(path, "rb").read(), {}
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        n, pos = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            start, size, length = struct.unpack_from("<QQQ", data, pos)
            target, pos = data[pos + 24:pos + 24 + length], pos + 24 + length
            if b"gfx950" in target and size:
                found.update(kernels_of_object(data[at + start:at + start + size]))
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)
    return found


def kernels_of_object(elf):
    first, = struct.unpack_from("<Q", elf, 40)                                  # section headers
    each, count = struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        kind, _, _, start, size = struct.unpack_from("<IQQQQ", elf, first + i * each + 4)
        if kind != 7:                                                           # SHT_NOTE
            continue
        name, length, what = struct.unpack_from("<III", elf, start)
        if what == 32:                                                          # NT_AMDGPU_METADATA
            body = start + 12 + (name + 3) // 4 * 4
            meta = msgpack.unpackb(elf[body:body + length])
            return {k[".name"]: k[".private_segment_fixed_size"] for k in meta["amdhsa.kernels"]}
    return {}


@pytest.mark.parametrize("kernel,instances", [
    ("latent_prompt_kernel", 24), ("latent_form_kernel", 2), ("kv_attention_tile_kernel", 64), ("gla_chunk_state_kernel", 12),
    ("gla_chunk_out_kernel", 12), ("delta_block_prepare_kernel", 4), ("delta_block_walk_kernel", 4), ("latent_decode_up_kernel", 8),
    ("16moe_route_kernel", 6), ("q4_gemm_dma2_kernelILi0ELb0ELi3ELi2ELb1E", 1), ("q4_gemm_dma2_kernelILi1ELb0ELi3ELi2ELb1E", 1)])
def test_nothing_is_kept_in_memory(kernel, instances):
    """(The int4 products: those whose last tiles are cut into slices.)"""
    from vllm_legacy_amd import _lib
    path = _lib.LIB_PATH if kernel.startswith("q4") else _lib.SEQ_LIB_PATH
    if not os.path.exists(path):
        pytest.skip("not built")
    kept = {k: v for k, v in kernels_of(path).items() if kernel in k}
    assert len(kept) == instances, sorted(kept)
    assert not any(kept.values()), {k: v for k, v in kept.items() if v}

"""Kernels that keep arrays in registers do so: what the built library's own kernel descriptions say (no GPU calls)."""
import os
import struct

import msgpack
import pytest

LIB = os.environ.get("ADAMAH_LIB_PATH") or os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "adam_amd", "libadamah_hip.so")


def descriptions():
    """name -> its entry of the amdhsa.kernels notes of the bundled code objects."""
    raw, out, at = open(LIB, "rb").read(), {}, -1
    while (at := raw.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 1)) >= 0:
        (n,), p = struct.unpack_from("<Q", raw, at + 24), at + 32
        for _ in range(n if n < 8 else 0):
            off, size, idlen = struct.unpack_from("<QQQ", raw, p)
            name = raw[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" not in name:
                continue
            elf = raw[at + off:at + off + size]
            shoff, = struct.unpack_from("<Q", elf, 40)
            entry, count = struct.unpack_from("<HH", elf, 58)
            for i in range(count):
                kind, = struct.unpack_from("<I", elf, shoff + i * entry + 4)
                if kind != 7:                                            # SHT_NOTE
                    continue
                o, = struct.unpack_from("<Q", elf, shoff + i * entry + 24)
                names, desc, what = struct.unpack_from("<III", elf, o)
                if what == 32:                                           # NT_AMDGPU_METADATA
                    o += 12 + (names + 3) // 4 * 4
                    out.update((k[".name"], k) for k in msgpack.unpackb(elf[o:o + desc])["amdhsa.kernels"])
    return out


@pytest.mark.parametrize("part,most", [("k_attn_f32", 0), ("k_chunk_scan", 0), ("k_space_scan", 0), ("k_linear_tiled", 0), ("k_linear_skinny", 0),
                                       ("k_experts", 0), ("k_operand_rows", 0), ("k_gemm_q4_ring", 16), ("k_gemm_q4_rows", 0), ("k_gemm_q8_f16", 0),
                                       ("k_head_rows", 0), ("k_linear_few", 0), ("k_gemv_bf16", 0), ("k_delta", 0), ("k_rmsnorm_rows", 0), ("k_rope_append_rows", 0), ("k_kv_tile_arrange", 0),
                                       ("k_attn_prefill", 0), ("k_topk_select", 0), ("k_gemm_q4_narrow", 0), ("k_group_topk_rank", 0),
                                       # heads of up to 128 two tiles of queries a wave; wider ones spill at 256 registers, heads of 256 by 256 most
                                       ("k_attn_bf16ILb0ELi4ELi8E", 0), ("k_attn_bf16ILb1ELi4ELi8E", 12), ("k_attn_bf16", 412)])
def test_arrays_stay_in_registers(part, most):
    """An array that a loop indexes and the compiler does not unroll lands in memory and is read from there in every step (the
    float32 attention of heads wider than 128 ran 1.4 times slower than with its loads in place).  `most`: bytes a lane."""
    assert os.path.exists(LIB), "build the library first: python -m adam_amd.build"
    found = {n: k[".private_segment_fixed_size"] for n, k in descriptions().items() if part in n}
    assert found and max(found.values()) <= most, found


@pytest.mark.parametrize("part,most", [("k_chunk_scanILb1ELi1ELi1E", 128), ("k_chunk_scanILb0ELi1ELi1E", 128), ("k_chunk_scanILb0ELi2ELi1E", 128),
                                       ("k_space_scanILi1ELi1E", 128), ("k_space_scanILi2ELi1E", 128),      # two workgroups of five waves a CU
                                       ("k_chunk_scanILb1ELi2ELi0E", 102), ("k_chunk_scanILb0ELi2ELi0E", 64),  # five and eight waves a SIMD
                                       ("k_chunk_scanILb1ELi3ELi2E", 256), ("k_chunk_scanILb0ELi4ELi2E", 256), ("k_space_scanILi4ELi2E", 256),
                                       ("k_attn_prefillILi64E", 128), ("k_attn_prefillILi128E", 168), ("k_attn_prefillILi256E", 256),      # four, three and two waves a SIMD
                                       ("k_gemm_q4_narrow", 256), ("k_group_topk_rankILb0E", 64), ("k_topk_select", 128)])
def test_as_many_workgroups_fit_as_the_rule_counts_on(part, most):
    """The walks' forms are chosen by how many workgroups a CU holds, and what the short prompts' attention gains hangs on how many waves: registers a lane
    of the form."""
    found = {n: k[".vgpr_count"] for n, k in descriptions().items() if part in n}
    assert found and max(found.values()) <= most, found

"""What the compiler gave the kernels of the built library: registers in scratch memory and LDS, from the code objects' own
notes (no GPU needed)."""
import functools
import struct

import pytest

msgpack = pytest.importorskip("msgpack")


@functools.lru_cache(maxsize=None)
def _kernels():
    """Name -> metadata of every gfx950 kernel: the library holds bundles of code objects, each an ELF file whose note of type
    32 ("AMDGPU") is a msgpack map."""
    from vllm_omni_draft_amd import _lib
    data, out, at = open(_lib.load()._name, "rb").read(), {}, -1
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 1)) >= 0:
        n, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            target, p = data[p + 24:p + 24 + length], p + 24 + length
            if b"gfx950" not in target or not size:
                continue
            elf = data[at + offset:at + offset + size]
            table, (entry, sections) = struct.unpack_from("<Q", elf, 40)[0], struct.unpack_from("<HH", elf, 58)
            for i in range(sections):
                if struct.unpack_from("<I", elf, table + i * entry + 4)[0] != 7:   # SHT_NOTE
                    continue
                note = struct.unpack_from("<Q", elf, table + i * entry + 24)[0]
                name, desc, kind = struct.unpack_from("<III", elf, note)
                if kind == 32:
                    notes = msgpack.unpackb(elf[note + 12 + (name + 3) // 4 * 4:][:desc], strict_map_key=False)
                    out.update((k[".name"], k) for k in notes["amdhsa.kernels"])
    return out


def _named(part):
    found = {n: k for n, k in _kernels().items() if part in n}
    assert found, part
    return found


def test_no_product_of_a_prompt_keeps_registers_in_scratch():
    """Blocks of 256 x 256 outputs use every register there is; a spilled one is a store and a load a lane in every block."""
    products = _named("18prompt_gemm_kernel")
    assert len(products) > 80
    assert {n: k[".vgpr_spill_count"] for n, k in products.items() if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]} == {}


def test_two_workgroups_of_prompt_attention_share_a_cu():
    """A workgroup's LDS is its two stages, its page table and, given at launch, 512 bytes a split for the splits' maxima: in splits of 128 keys
    (template argument 1) two have room beside each other up to 11264 keys."""
    split_maxima = 11264 // 128 * 512
    for size in (64, 128):
        (kernel,) = _named(f"18prompt_attn_kernelILi{size}ELi1E").values()
        assert 2 * (kernel[".group_segment_fixed_size"] + split_maxima) <= 160 * 1024, size

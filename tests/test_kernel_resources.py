"""What the compiled kernels take of a compute unit, from the metadata of the built libraries: registers that spill and LDS or registers that
keep a second work-group out do not show in any result, only in time."""

import re
import struct

import msgpack
import pytest

from burn_transformers_amd.kernels import build


def kernels_of(module):
    """The metadata of every kernel of a built module: code objects of the bundle in the library, AMDGPU notes of each."""
    with open(build.ensure(module), "rb") as handle:
        blob = handle.read()
    found, at = [], blob.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        count, place = struct.unpack_from("<Q", blob, at + 24)[0], at + 32
        for _ in range(count):
            offset, size, named = struct.unpack_from("<QQQ", blob, place)
            name = blob[place + 24:place + 24 + named]
            place += 24 + named
            if b"gfx" in name and size:
                found += notes_of(blob[at + offset:at + offset + size])
        at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)
    assert found, module
    return found


def notes_of(elf):
    sections, (entry, count) = struct.unpack_from("<Q", elf, 0x28)[0], struct.unpack_from("<HH", elf, 0x3A)
    kernels = []
    for i in range(count):
        if struct.unpack_from("<I", elf, sections + i * entry + 4)[0] != 7:        # SHT_NOTE
            continue
        place, size = struct.unpack_from("<QQ", elf, sections + i * entry + 24)
        end = place + size
        while place < end:
            named, described, kind = struct.unpack_from("<III", elf, place)
            start = place + 12 + (named + 3) // 4 * 4
            if kind == 32:                                                          # NT_AMDGPU_METADATA
                kernels += msgpack.unpackb(elf[start:start + described])["amdhsa.kernels"]
            place = start + (described + 3) // 4 * 4
    return kernels


def skinny_forms(far=0):
    """(rows' blocks, column blocks, chunks a batch, waves, quads of a norm, epilogue's kind, metadata) of the skinny product's forms (``far``: of
    those with offsets of 64 bits)."""
    for kernel in kernels_of("gemm_mfma"):
        form = re.search(r"gemm_skinny_kernelI(?:f|DF16b)((?:Li\d+E)+)E", kernel[".name"])
        numbers = [int(n) for n in re.findall(r"Li(\d+)E", form.group(1))] if form else []
        if numbers and numbers[8] == far:
            yield (*numbers[:6], kernel)


def test_two_work_groups_of_the_skinny_product_share_a_compute_unit():
    # eight waves are two a SIMD, whose 512 registers a lane then hold two work-groups up to 128.  (Without a norm: its rows are in
    # registers beside the weights.  Four blocks of eight chunks are 128 registers of weights and rows alone.)
    forms = [f for f in skinny_forms() if f[4] == 0 and not (f[0] * f[1] == 4 and f[2] == 8) and f[6][".max_flat_workgroup_size"] == 512]
    assert len(forms) > 20
    assert not [f for f in forms if f[6][".vgpr_count"] + f[6].get(".agpr_count", 0) > 128]


def test_a_ninth_wave_keeps_no_second_work_group_out():
    # nine waves are three on one SIMD, and two work-groups of nine five: 512 / 5 registers each, in eights
    forms = [f for f in skinny_forms() if f[4] == 0 and f[6][".max_flat_workgroup_size"] == 576]
    assert len(forms) > 20
    assert not [f for f in forms if f[6][".vgpr_count"] + f[6].get(".agpr_count", 0) > 96]


def test_lds_leaves_room_for_two_work_groups_of_the_skinny_product():
    # (without a norm, whose rows are LDS of the launch)
    forms = [f for f in skinny_forms() if f[4] == 0]
    assert len(forms) > 100
    assert not [f for f in forms if f[6][".group_segment_fixed_size"] > 160 * 1024 // 2]


def test_no_form_of_the_skinny_product_spills():
    forms = list(skinny_forms())
    assert len(forms) > 100
    forms += skinny_forms(far=1)
    assert not [f for f in forms if f[6][".vgpr_spill_count"] or f[6][".private_segment_fixed_size"]]


@pytest.mark.parametrize("module", ["attention_f32", "attention_f32_softmax", "attention_f32_capped", "attention_f32_sigmoid"])
def test_float32_decode_attention_keeps_its_keys_in_registers(module):
    kernels = [k for k in kernels_of(module) if re.search(r"attention_f32_(decode|join)_kernel", k[".name"])]
    assert len(kernels) == 3                          # heads of up to 64 and of up to 128, and the join of runs
    assert not [k for k in kernels if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]]
    # two work-groups of four waves a compute unit: a wave has half of the 512 registers a lane
    assert not [k for k in kernels if k[".vgpr_count"] + k.get(".agpr_count", 0) > 256]

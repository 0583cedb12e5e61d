"""Registers of the built kernels, read from the library's own metadata: what decides how many waves a SIMD runs, and whether a wave has all it holds in
registers, can change with any line of a kernel and no result shows it."""
import re
import struct

import msgpack
import pytest

from rbitnet_amd.csrc import build


def _sections(elf, at):
    """(type, name, bytes) of the sections of the ELF file of 64 bits at `at`."""
    start, = struct.unpack_from("<Q", elf, at + 40)
    size, count, names = struct.unpack_from("<HHH", elf, at + 58)
    heads = [struct.unpack_from("<IIQQQQ", elf, at + start + i * size) for i in range(count)]      # name, type, flags, address, offset, size
    text = elf[at + heads[names][4]:at + heads[names][4] + heads[names][5]]
    for name, kind, _, _, offset, length in heads:
        yield kind, text[name:text.index(b"\0", name)].decode(), elf[at + offset:at + offset + length] if kind != 8 else b""


def _metadata(note):
    """The kernels' entry of a code object's notes (NT_AMDGPU_METADATA, 32)."""
    at = 0
    while at < len(note):
        name, length, kind = struct.unpack_from("<III", note, at)
        at += 12 + (name + 3) // 4 * 4
        if kind == 32:
            yield from msgpack.unpackb(note[at:at + length], raw=False, strict_map_key=False)["amdhsa.kernels"]
        at += (length + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    """{(kernel, its template's numbers and types as mangled): (registers, bytes of scratch)} of every kernel of gfx950."""
    with open(build.ensure_built(), "rb") as f:
        elf = f.read()
    found, magic = {}, b"__CLANG_OFFLOAD_BUNDLE__"
    fat = next(data for _, name, data in _sections(elf, 0) if name == ".hip_fatbin")
    for bundle in (m.start() for m in re.finditer(magic, fat)):
        at = bundle + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", fat, bundle + len(magic))[0]):
            offset, size, name = struct.unpack_from("<QQQ", fat, at)
            target = fat[at + 24:at + 24 + name]
            at += 24 + name
            if b"gfx950" not in target or size == 0:
                continue
            for kind, _, note in _sections(fat, bundle + offset):
                for k in _metadata(note) if kind == 7 else ():
                    m = re.match(r"_ZN?(?:12_GLOBAL__N_1)?\d+([a-z]\w*?_kernel)(?:I(.*?)EEv|[Ei])", k[".name"])
                    if m:
                        args = tuple(int(n) if n else kind_ for n, kind_ in re.findall(r"L[ib](\d+)E?|(f|6bf16_t)", (m.group(2) or "") + "E"))
                        found[m.group(1), args] = k[".vgpr_count"], k[".private_segment_fixed_size"]
    assert len(found) > 500
    return found


def test_products_of_few_tokens_hold_their_operands_in_registers(kernels):
    few = [k for k in kernels if k[0] in ("gemm_skinny_kernel", "gemm_f32_few_kernel", "gemm_f32_short_kernel", "gemm_group_kernel", "routed_up_few_kernel",
                                          "routed_down_few_kernel")]
    assert len(few) > 300
    assert [k for k in few if kernels[k][1] != 0] == []


# row tiles of a wave, end -> the most registers that the waves a SIMD ran when these kernels were timed leave to each (512 between them)
@pytest.mark.parametrize("tiles,end,most", [(1, 0, 72), (1, 3, 96), (1, 4, 72), (2, 1, 128), (4, 0, 168), (4, 1, 168), (4, 2, 256), (4, 3, 248)])
@pytest.mark.parametrize("out", ["f", "6bf16_t"])
def test_products_of_9_to_16_tokens_leave_room_for_as_many_waves(kernels, tiles, end, most, out):
    """Fragment-major W, whole stages, a block of tokens a load, nothing set aside."""
    key = "gemm_skinny_kernel", (1, tiles, 1, 1, end, out, 0, 1, 1, 0)
    if end in (2, 3) and out != "f":
        assert key not in kernels                            # (these ends add to a float32 stream)
        return
    assert kernels[key][0] <= most

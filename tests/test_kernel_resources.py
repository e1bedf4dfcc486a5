"""What the compiler says the built kernels hold: the metadata of the code objects inside the library (CPU)."""
import struct

import msgpack

from splash_amd import _native

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def kernels():
    """{mangled name: metadata} of every gfx950 kernel of the library, from the notes of its code objects."""
    library = open(_native.lib._name, "rb").read()
    found, at = {}, library.find(MAGIC)
    while at >= 0:
        place = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", library, at + len(MAGIC))[0]):
            offset, size, length = struct.unpack_from("<3Q", library, place)
            if b"gfx950" in library[place + 24:place + 24 + length]:
                found.update(of_code_object(library[at + offset:at + offset + size]))
            place += 24 + length
        at = library.find(MAGIC, at + 1)
    return found


def of_code_object(elf):
    headers, = struct.unpack_from("<Q", elf, 32)
    entry, count = struct.unpack_from("<2H", elf, 54)
    for i in range(count):
        kind, _, offset, _, _, size = struct.unpack_from("<2I4Q", elf, headers + i * entry)
        at = offset
        while kind == 4 and at < offset + size:   # PT_NOTE
            name, length, note = struct.unpack_from("<3I", elf, at)
            text = at + 12 + -(-name // 4) * 4
            if note == 32:   # NT_AMDGPU_METADATA
                return {k[".name"]: k for k in msgpack.unpackb(elf[text:text + length])["amdhsa.kernels"]}
            at = text + -(-length // 4) * 4
    return {}


def test_the_decode_projections_spill_nothing():
    """A register reloaded in the ring's loop waits for every load behind it, and with that empties the ring
    (kernels/gguf_linear.hip, kDecodeWaves)."""
    decode = {n: k for n, k in kernels().items() if "gguf_decode" in n or "gguf_moe_decode" in n}
    assert len(decode) > 150
    assert not [n for n, k in decode.items() if k[".private_segment_fixed_size"] or k[".vgpr_spill_count"]]

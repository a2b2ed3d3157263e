"""What the compiler gave the attention kernels of libparaattn_hip.so, from the metadata notes of the gfx950 code in it.

A vector register spilled in a tile loop goes to memory and back in every tile, and scalar registers spilled by a
kernel's entry cost short workgroups a few per cent of their time; neither shows in a result."""
import os
import re
import struct

import pytest

from paraattention_amd import _lib

msgpack = pytest.importorskip("msgpack")


def _notes(elf):
    """The metadata of an AMDGPU code object (64-bit little-endian ELF): the msgpack map of its note of type 32."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        kind, _, _, off, size = struct.unpack_from("<IQQQQ", elf, shoff + i * shentsize + 4)
        end = off + size
        while kind == 7 and off + 12 <= end:  # SHT_NOTE
            namesz, descsz, what = struct.unpack_from("<III", elf, off)
            at = off + 12 + (namesz + 3) // 4 * 4
            if what == 32 and elf[off + 12 : off + 18] == b"AMDGPU":
                return msgpack.unpackb(elf[at : at + descsz])
            off = at + (descsz + 3) // 4 * 4
    return None


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("the library is not built")
    blob = open(_lib.LIB_PATH, "rb").read()
    found = {}
    for m in re.finditer(rb"\x7fELF\x02\x01\x01", blob):
        if struct.unpack_from("<H", blob, m.start() + 0x12)[0] != 224:  # EM_AMDGPU
            continue
        meta = _notes(blob[m.start() :])
        for k in meta["amdhsa.kernels"] if meta else ():
            found[k[".name"]] = k
    assert len(found) > 100
    return found


def test_pipelined_kernels_spill_no_vector_register(kernels):
    attention = {n: k for n, k in kernels.items() if any(f"{kind}_kernel" in n for kind in ("pipe", "stream", "short"))}
    # (the form with 64 rows per wavefront, which only a tuning knob reaches, spills and is slower for it)
    attention = {n: k for n, k in attention.items() if not re.search(r"stream_kernelI.*ELb[01]ELi2ELb", n)}
    assert len(attention) > 60
    spilled = {n: k[".vgpr_spill_count"] for n, k in attention.items() if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}
    assert not spilled, spilled


@pytest.mark.parametrize("T", ["4BF16", "3F16"])
def test_unsplit_head_dim_64_kernels_pay_nothing_for_the_split(kernels, T):
    """The dense kernel of an unsplit launch spills fewer scalar registers than the one that decodes key shares, for both
    workgroup sizes and with and without a score bound."""
    for wavefronts in (4, 8):
        for bounded in (0, 1):
            name = f"attn_fwd_d64_pipe_kernelINS_{T}ELb0ELi{wavefronts}ELb{bounded}ELi0ELb0ELb%dEEEv"
            whole, cut = (next(k[".sgpr_spill_count"] for n, k in kernels.items() if name % c in n) for c in (0, 1))
            assert whole <= 24 and whole < cut, (name, whole, cut)


def test_resident_key_kernels_spill_nothing(kernels):
    resident = {n: k for n, k in kernels.items() if "attn_fwd_resident_kernel" in n}
    assert len(resident) == 12  # two types, two head_dims; unmasked with a last tile of 64 or 32 keys, and with a bias
    for n, k in resident.items():
        assert not k[".vgpr_spill_count"] and not k[".sgpr_spill_count"] and not k[".private_segment_fixed_size"], n

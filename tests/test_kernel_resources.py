"""What the compiler gave the built kernels, from the code objects' own metadata."""

import struct

import msgpack
import pytest

from moe_dispatch._lib import library_path

_AMDGPU, _PT_NOTE, _AMDGPU_METADATA = 224, 4, 32


def _code_objects(data):
    """Offsets of the gfx950 ELF images embedded in the library."""
    at = data.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == _AMDGPU:
            yield at
        at = data.find(b"\x7fELF", at + 1)


def _kernels(data):
    """Kernel name -> its metadata, over the library's code objects."""
    kernels = {}
    for base in _code_objects(data):
        phoff, = struct.unpack_from("<Q", data, base + 32)
        phentsize, phnum = struct.unpack_from("<HH", data, base + 54)
        for i in range(phnum):
            kind, _, offset, _, _, size = struct.unpack_from("<IIQQQQ", data, base + phoff + i * phentsize)
            at, end = base + offset, base + offset + size
            while kind == _PT_NOTE and at < end:
                namesz, descsz, note = struct.unpack_from("<III", data, at)
                desc = at + 12 + -(-namesz // 4) * 4
                if note == _AMDGPU_METADATA:
                    for kernel in msgpack.unpackb(data[desc:desc + descsz])["amdhsa.kernels"]:
                        kernels[kernel[".name"]] = kernel
                at = desc + -(-descsz // 4) * 4
    return kernels


@pytest.fixture(scope="module")
def kernels():
    found = _kernels(library_path().read_bytes())
    assert len(found) > 100
    return found


def test_routing_and_row_kernels_spill_no_registers(kernels):
    """Every kernel but the grouped GEMMs (whose scalar registers spill to lanes) keeps
    its registers: a spilled router took twice its time."""
    rest = {name: k for name, k in kernels.items() if "grouped_gemm" not in name}
    for part in ("route_small_kernel", "route_planes_kernel", "router_direct_kernel", "pack_kernel", "combine_kernel"):
        assert any(part in name for name in rest), part
    spilled = {name: (k[".vgpr_spill_count"], k[".private_segment_fixed_size"]) for name, k in rest.items()
               if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}
    assert not spilled

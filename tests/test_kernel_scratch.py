"""Per-thread scratch memory of the built kernels, read from the metadata that
the compiler stores with them in libpetjson.so."""
import struct

import msgpack
import pytest

import petjson as pj


def _kernels():
    """{demangled-enough name: scratch bytes per thread} of every kernel."""
    blob = open(pj.lib_path(), "rb").read()
    out, at = {}, 0
    while (at := blob.find(b"AMDGPU\0\0", at)) >= 0:
        namesz, descsz, kind = struct.unpack_from("<III", blob, at - 12)
        if namesz == 7 and kind == 32 and at + 8 + descsz <= len(blob):    # NT_AMDGPU_METADATA
            meta = msgpack.unpackb(blob[at + 8: at + 8 + descsz], strict_map_key=False)
            out.update({k[".name"]: k[".private_segment_fixed_size"] for k in meta["amdhsa.kernels"]})
        at += 8
    return out


@pytest.mark.parametrize("kernel,instances", [("k_mdec_countI", 2), ("k_mdec_writeI", 4), ("k_encode_modelI", 8),
                                              ("k_encode_rowsI", 4)])
def test_per_record_kernels_stage_in_registers(kernel, instances):
    """The kernels that give each record a thread hold no array in scratch: at
    most the frame of the call that skips unknown values (28 bytes) is there.
    (Eight 16-byte loads in flight per thread once were: 128 bytes.)"""
    got = {n: b for n, b in _kernels().items() if kernel in n}
    assert len(got) == instances and max(got.values()) <= 64, got

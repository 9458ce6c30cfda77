"""Registers of the built kernels, from the metadata of the kernel library's code objects (no GPU call)."""
import struct

import pytest


def kernels():
    from pie_amd import _lib

    msgpack = pytest.importorskip("msgpack")
    data, at, found = _lib.KERNEL_LIB_PATH.read_bytes(), -1, []
    while (at := data.find(b"AMDGPU\0\0", at + 1)) >= 0:   # (an ELF note's name; its lengths and type stand before it)
        name_bytes, content, kind = struct.unpack_from("<III", data, at - 12)
        if name_bytes == 7 and kind == 32:
            found += msgpack.unpackb(data[at + 8:at + 8 + content])["amdhsa.kernels"]
    return found


def test_no_gemm_spills_registers():
    """The GEMMs' launch bounds leave each instance the registers it needs: nothing of theirs goes through scratch memory."""
    gemms = [k for k in kernels() if any(n in k[".name"] for n in ("gemm_columns", "gemm_groups", "gemm_waves", "gemm_wide", "gemm_mfma"))]
    assert len(gemms) > 40 and sum("gemm_waves" in k[".name"] for k in gemms) > 40
    assert not [k[".name"] for k in gemms if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]]

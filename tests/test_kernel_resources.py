"""What the built library says of its kernels (the metadata that hipcc writes beside the code): the kernels that count their own loads
in flight keep nothing in scratch memory. A register spilled there comes back behind a wait for every load before it, so a ring of
loads in flight is drained in each step (GEGLU tiles of 192 x 128: 215 to 356 registers per lane once went there unnoticed)."""
import os
import struct

import msgpack
import pytest

ELF_NOTE, AMDGPU_METADATA = 7, 32


def _kernels(path):
    """{kernel name: its metadata} over the gfx950 code objects bundled in the library"""
    data = open(path, "rb").read()
    kernels, magic = {}, b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, n = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24:entry + 24 + n]
            entry += 24 + n
            if b"gfx950" in target and size:
                kernels.update(_of_code_object(data[at + offset:at + offset + size]))
        at = data.find(magic, at + len(magic))
    return kernels


def _of_code_object(elf):
    found = {}
    table, = struct.unpack_from("<Q", elf, 40)
    entry_size, n_sections = struct.unpack_from("<HH", elf, 58)
    for i in range(n_sections):
        _, kind, _, _, at, size = struct.unpack_from("<IIQQQQ", elf, table + i * entry_size)
        end = at + size
        while kind == ELF_NOTE and at < end:
            n_name, n_desc, note = struct.unpack_from("<III", elf, at)
            desc = at + 12 + (n_name + 3) // 4 * 4
            if note == AMDGPU_METADATA:
                found.update({k[".name"]: k for k in msgpack.unpackb(elf[desc:desc + n_desc])["amdhsa.kernels"]})
            at = desc + (n_desc + 3) // 4 * 4
    return found


@pytest.fixture(scope="module")
def kernels():
    from brodiffusion_amd import _capi
    if not os.path.exists(_capi.LIB_PATH):
        from brodiffusion_amd import build
        build.build()
    return _kernels(_capi.LIB_PATH)


@pytest.mark.parametrize("kernel,at_least", [
    ("linear_pipe_kernel", 54),        # 11 plain forms, 5 GEGLU, 7 of INT8 and 4 of both, by two types
    ("linear_dma_kernel", 2),
    ("sdpa_wide_long_kernel", 2),
    *((f"sdpa_fwd_pp_dma_kernelI{t}Li{d}ELb1E", 3) for t in ("DF16_", "DF16b") for d in (72, 128)),      # split launches: dense, ragged, key mask
    *((f"sdpa_fwd_pp_dma_kernelI{t}Li{d}ELb0ELi3E", 1) for t in ("DF16_", "DF16b") for d in (72, 128)),  # a key mask without prefix
])
def test_kernels_with_loads_in_flight_use_no_scratch(kernels, kernel, at_least):
    found = {name: (k[".private_segment_fixed_size"], k[".vgpr_spill_count"]) for name, k in kernels.items() if kernel in name}
    assert len(found) >= at_least
    assert not {name: use for name, use in found.items() if use != (0, 0)}

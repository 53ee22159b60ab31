"""Registers and scratch of the built kernels, read from the metadata that the
compiler wrote into the library: limits on which workgroups per CU depend."""
import os
import re
import struct
import subprocess

import msgpack
import pytest

from masterthesis_amd import LIB_PATH, capi

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
NT_AMDGPU_METADATA = 32


def _device_objects(blob):
    """The gfx950 ELF objects of the offload bundles in the library."""
    at = blob.find(BUNDLE)
    while at >= 0:
        pos = at + len(BUNDLE)
        (count,) = struct.unpack_from("<Q", blob, pos)
        pos += 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24:pos + 24 + n]
            pos += 24 + n
            if b"gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at = blob.find(BUNDLE, at + 1)


def _metadata(elf):
    (phoff,) = struct.unpack_from("<Q", elf, 32)
    entsize, count = struct.unpack_from("<HH", elf, 54)
    for p in range(count):
        kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + p * entsize)
        if kind != 4:  # PT_NOTE
            continue
        end = off + size
        while off < end:
            namesz, descsz, ntype = struct.unpack_from("<III", elf, off)
            off += 12 + (namesz + 3) // 4 * 4
            if ntype == NT_AMDGPU_METADATA:
                return msgpack.unpackb(elf[off:off + descsz])
            off += (descsz + 3) // 4 * 4
    return {}


@pytest.fixture(scope="module")
def kernels():
    capi.load()
    out = {}
    with open(LIB_PATH, "rb") as f:
        for elf in _device_objects(f.read()):
            for k in _metadata(elf).get("amdhsa.kernels", []):
                out[k[".name"]] = k
    assert len(out) > 50
    return out


def test_fp64_one_step_tiles_keep_four_waves(kernels):
    """Six planes in flight: two 8-wave workgroups per CU need 128 registers."""
    tiles = {n: k for n, k in kernels.items() if re.search(r"stream_kernelINS_9HeatVarOpIdLi0E\S*Li6EEEv", n)}
    assert len(tiles) == 3
    for n, k in tiles.items():
        assert k[".vgpr_count"] <= 128 and k[".private_segment_fixed_size"] == 0, (n, k[".vgpr_count"])


def test_two_row_sweeps_do_not_spill(kernels):
    pairs = {n: k for n, k in kernels.items() if "heatvar_pairs_kernel" in n}
    assert len(pairs) > 20
    assert [n for n, k in pairs.items() if k[".private_segment_fixed_size"]] == []


OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_no_empty_lane_regions(tmp_path):
    """A region that selects lanes and then does nothing: what ROCm 7.2's clang left
    of `c ? v : 0` in the FP64 start of the adjoint when c was a chain of
    short-circuit branches; the zero had been written over v on every lane."""
    with open(LIB_PATH, "rb") as f:
        objects = list(_device_objects(f.read()))
    assert objects
    for n, elf in enumerate(objects):
        path = tmp_path / f"{n}.elf"
        path.write_bytes(elf)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(path)], check=True,
                              capture_output=True, text=True).stdout
        code = "\n".join(x.split("//")[0].strip() for x in text.splitlines())
        assert "s_and_saveexec_b64" in code or "s_endpgm" in code
        bad = re.findall(r"s_and_saveexec_b64 (s\[\d+:\d+\]), \S+\ns_or_b64 exec, exec, \1\n", code)
        assert not bad, (n, len(bad))

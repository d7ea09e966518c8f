"""The built library's kernels as the compiler allocated them: the metadata
that each code object carries (register counts and spills). A spilled scalar
costs a lane move at each use, which tests of the results do not show."""
import re
import struct

import pytest

from scriptonait_amd import build

msgpack = pytest.importorskip("msgpack")

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
METADATA_NOTE = 32  # NT_AMDGPU_METADATA


def code_objects(data):
    """The gfx950 code objects of a host library's offload bundles."""
    for m in re.finditer(re.escape(BUNDLE), data):
        at = m.start() + len(BUNDLE)
        (entries,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(entries):
            off, size, n = struct.unpack_from("<QQQ", data, at)
            triple = data[at + 24:at + 24 + n]
            at += 24 + n
            if size and triple.endswith(build.ARCH.encode()):
                yield data[m.start() + off:m.start() + off + size]


def kernels(elf):
    """The kernel entries of one code object's metadata note (ELF64)."""
    (phoff,) = struct.unpack_from("<Q", elf, 32)
    phentsize, phnum = struct.unpack_from("<HH", elf, 54)
    for i in range(phnum):
        kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phentsize)
        if kind != 4:  # PT_NOTE
            continue
        at, end = off, off + size
        while at < end:
            namesz, descsz, note = struct.unpack_from("<III", elf, at)
            desc = at + 12 + (namesz + 3) // 4 * 4
            if note == METADATA_NOTE:
                yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
            at = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def metadata():
    if not build.LIB_PATH.exists():
        pytest.skip("the library is not built")
    found = {k[".name"]: k for elf in code_objects(build.LIB_PATH.read_bytes()) for k in kernels(elf)}
    assert found
    return found


@pytest.mark.parametrize("nch", [1, 2, 4, 8])
@pytest.mark.parametrize("counts", [0, 1])
@pytest.mark.parametrize("masked", [0, 1])
def test_small_k_register_kernels_spill_nothing(metadata, nch, counts, masked):
    """sample_fast_kernel<NCH, GREEDY, CMODE, BIGK, MASKED> for top-k rows of
    K <= 64, the kernel of an ordinary decode step."""
    name = f"sample_fast_kernelILi{nch}ELb0ELb{counts}ELb0ELb{masked}E"
    (k,) = [v for n, v in metadata.items() if name in n]
    assert (k[".sgpr_spill_count"], k[".vgpr_spill_count"]) == (0, 0)

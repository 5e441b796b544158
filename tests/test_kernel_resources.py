"""Registers and scratch of the built kernels, read from the library's own code object metadata
(no GPU): kernels whose loop lives in registers must not spill."""
import re
import struct
import subprocess
from pathlib import Path

import msgpack
import pytest

ROOT = Path(__file__).resolve().parents[1]
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _elf_notes(elf):
    """(name, type, descriptor) of every ELF64 note."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        _, typ, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * shentsize)
        if typ != 7:   # SHT_NOTE
            continue
        end = off + size
        while off < end:
            nsz, dsz, ntype = struct.unpack_from("<III", elf, off)
            name = elf[off + 12:off + 12 + nsz].rstrip(b"\0")
            off += 12 + (nsz + 3) // 4 * 4
            yield name, ntype, elf[off:off + dsz]
            off += (dsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    """Kernel name -> metadata of every gfx950 kernel in libhxq.so."""
    from helix_substrate import _hxq
    if not _hxq.library_path().exists():
        subprocess.run(["make", "-j8", "-C", str(ROOT / "helix-substrate_amd" / "csrc")], check=True)
    blob = _hxq.library_path().read_bytes()
    found = {}
    for m in re.finditer(re.escape(MAGIC), blob):
        p = m.start() + len(MAGIC)
        n, = struct.unpack_from("<Q", blob, p)
        if not 0 < n < 16:
            continue
        p += 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            ident = blob[p + 24:p + 24 + idlen]
            p += 24 + idlen
            elf = blob[m.start() + off:m.start() + off + size]
            if b"gfx950" not in ident or elf[:4] != b"\x7fELF":
                continue
            for name, typ, desc in _elf_notes(elf):
                if name == b"AMDGPU" and typ == 32:
                    for k in msgpack.unpackb(desc)["amdhsa.kernels"]:
                        found[k[".name"]] = k
    assert found, "no gfx950 kernels found in the library"
    return found


def test_few_row_gemm_does_not_spill(kernels):
    rows = {n: k for n, k in kernels.items() if "rows_kernel" in n}
    assert len(rows) > 100
    spilled = {n: k[".private_segment_fixed_size"] for n, k in rows.items()
               if k[".private_segment_fixed_size"] or k[".vgpr_spill_count"]}
    assert not spilled, spilled

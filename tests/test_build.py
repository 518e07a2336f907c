"""The build takes every listed source or fails, and the library needs no symbol
of its own from elsewhere."""
import os
import re
import struct
import subprocess

import pytest

from shady_thinker_amd import build


def test_missing_source_fails(monkeypatch, tmp_path):
    monkeypatch.setattr(build, "SOURCES", ["runtime.hip", "no_such_kernel.hip"])
    monkeypatch.setattr(build, "OBJ", str(tmp_path))
    monkeypatch.setattr(build, "LIB", str(tmp_path / "lib.so"))
    monkeypatch.setattr(build, "_compile", lambda src: pytest.fail(f"compiled {src}"))
    with pytest.raises(RuntimeError, match="no_such_kernel.hip"):
        build.build()


def test_sources_are_the_hip_files():
    assert sorted(build.SOURCES) == sorted(f for f in os.listdir(build.CSRC) if f.endswith(".hip"))


def test_library_defines_its_symbols():
    out = subprocess.run(["nm", "-D", "--undefined-only", build.LIB], check=True, capture_output=True, text=True).stdout
    assert not [l for l in out.split() if l.startswith(("_ZN2st", "st_"))]


def _kernels(path):
    """The metadata of every GPU kernel in the library (the notes of its embedded code objects)."""
    msgpack = pytest.importorskip("msgpack")
    b = open(path, "rb").read()
    i = b.find(b"\x7fELF\x02\x01")
    while i >= 0:
        if struct.unpack_from("<H", b, i + 18)[0] == 224:  # EM_AMDGPU
            shoff, = struct.unpack_from("<Q", b, i + 40)
            for s in range(*struct.unpack_from("<H", b, i + 60)):
                if struct.unpack_from("<I", b, i + shoff + 64 * s + 4)[0] == 7:  # SHT_NOTE
                    off, _ = struct.unpack_from("<QQ", b, i + shoff + 64 * s + 24)
                    name, size = struct.unpack_from("<II", b, i + off)
                    at = i + off + 12 + (name + 3) // 4 * 4
                    yield from msgpack.unpackb(b[at:at + size], strict_map_key=False)["amdhsa.kernels"]
        i = b.find(b"\x7fELF\x02\x01", i + 4)


@pytest.mark.parametrize("kernel,most", [
    ("gemm_kernel", 5),  # (10 in groups of 64 on 256 columns cost a tenth)
    ("i4xs_kernelILi1ELi1E", 4),  # f32 x, one source (6 on four units with zero points: 5-17%)
    ("i4xs_kernel", 10),  # (8-10: gate/up in groups of 64 with zero points, three units; others to 8)
])
def test_register_spills(kernel, most):
    """No variant of a kernel that fills its registers spills more of them than
    was measured as harmless."""
    spills = {k[".name"]: k[".vgpr_spill_count"] for k in _kernels(build.LIB) if re.search(r"\d" + kernel, k[".name"])}
    assert spills and max(spills.values()) <= most, {n: v for n, v in spills.items() if v > most}

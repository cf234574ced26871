"""Registers of the built kernels, read from the code objects' own metadata (no GPU): a GEMM whose epilogue spills
the operands of its loop pays for it on every tile, and no output shows it."""

import pathlib
import re
import shutil
import struct
import subprocess

import pytest

READOBJ = shutil.which("llvm-readobj") or "/opt/rocm/llvm/bin/llvm-readobj"


def _kernels(lib: pathlib.Path, tmp: pathlib.Path) -> dict[str, int]:
    """Mangled kernel name -> spilled vector registers, of every gfx950 code object in ``lib``."""
    data, out, at = lib.read_bytes(), {}, 0
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    while (at := data.find(magic, at)) >= 0:
        count, = struct.unpack_from("<Q", data, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + length].decode()
            p += 24 + length
            if "gfx950" not in name or not size:
                continue
            obj = tmp / "code.o"
            obj.write_bytes(data[at + offset:at + offset + size])
            notes = subprocess.run([READOBJ, "--notes", str(obj)], capture_output=True, text=True, check=True).stdout
            names = re.findall(r"^\s+\.name:\s+(_Z\S+)$", notes, re.M)
            spills = re.findall(r"^\s+\.vgpr_spill_count:\s+(\d+)$", notes, re.M)
            assert len(names) == len(spills)
            out.update(zip(names, map(int, spills)))
        at += 1
    return out


def test_gemm_kernels_do_not_spill(tmp_path):
    from mx_qlinear import _lib

    if not pathlib.Path(READOBJ).exists():
        pytest.skip("no llvm-readobj")
    if not _lib.LIB_PATH.exists():
        from mx_qlinear import build

        build.build()
    gemms = {k: v for k, v in _kernels(_lib.LIB_PATH, tmp_path).items() if "gemm_i8_kernel" in k}
    assert len(gemms) > 20
    # (a few registers around the tile loop; the gated residual epilogue once spilled 67 and then 137)
    assert max(gemms.values()) <= 16, sorted(gemms.items(), key=lambda kv: -kv[1])[:5]

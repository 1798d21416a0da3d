"""What the compiler gave each kernel of the built library: registers, LDS, spills, scratch
(the metadata note of the gfx950 code objects in libkinfu.so)."""
from __future__ import annotations

import functools
import os
import struct
import subprocess
import tempfile

import yaml

from openfusion_amd import kinfu as kf

READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
SIMDS, VGPRS, LDS_BYTES, MAX_WAVES = 4, 512, 160 * 1024, 8  # of a CU; registers per lane and SIMD, waves per SIMD


def _code_objects(data: bytes):
    at = data.find(BUNDLE)
    while at >= 0:
        pos = at + len(BUNDLE)
        count, = struct.unpack_from("<Q", data, pos)
        pos += 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, pos)
            if b"gfx950" in data[pos + 24:pos + 24 + n] and size:
                yield data[at + off:at + off + size]
            pos += 24 + n
        at = data.find(BUNDLE, at + 1)


@functools.lru_cache(maxsize=1)
def kernels() -> dict[str, dict]:
    """Mangled name -> metadata of every kernel of the library."""
    out = {}
    with open(kf.LIB_PATH, "rb") as f:
        data = f.read()
    for obj in _code_objects(data):
        with tempfile.NamedTemporaryFile(suffix=".elf") as t:
            t.write(obj)
            t.flush()
            text = subprocess.run([READELF, "--notes", t.name], check=True, capture_output=True, text=True).stdout
        meta = yaml.safe_load(text[text.index("---"):text.index("\n...")])
        for k in meta["amdhsa.kernels"]:
            out[k[".name"]] = k
    return out


def find(part: str) -> dict:
    """The one kernel whose mangled name holds `part`."""
    hits = [k for n, k in kernels().items() if part in n]
    assert len(hits) == 1, (part, [k[".name"] for k in hits])
    return hits[0]


def waves_by_registers(k: dict) -> int:
    """Waves per SIMD that the kernel's vector registers leave room for."""
    used = (k[".vgpr_count"] + 7) // 8 * 8  # .vgpr_count includes the accumulation registers
    return min(VGPRS // used, MAX_WAVES)


def blocks_by_registers(k: dict, threads: int) -> int:
    return waves_by_registers(k) * SIMDS // (threads // 64)


def blocks_by_lds(k: dict) -> int:
    return LDS_BYTES // max(k[".group_segment_fixed_size"], 1)

"""Scratch memory of the kernels whose loops hold all they can in registers,
read from the metadata of the built library's own code objects: a register
kept in memory there costs a load or store per step."""
import os
import re
import shutil
import struct
import subprocess

import pytest

READELF = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin:" + os.environ.get("PATH", ""))


def scratch_bytes(tmp_path):
    """kernel (mangled name) -> bytes of scratch per lane"""
    import warp_amd.hip as wh
    lib, out, at = open(wh.LIB_PATH, "rb").read(), {}, 0
    while (at := lib.find(b"\x7fELF", at + 1)) > 0:
        if struct.unpack_from("<H", lib, at + 18)[0] != 224:             # EM_AMDGPU
            continue
        end = struct.unpack_from("<Q", lib, at + 40)[0] + 64 * struct.unpack_from("<H", lib, at + 60)[0]
        f = tmp_path / "code.co"
        f.write_bytes(lib[at:at + end])
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        out.update((n, int(b)) for n, b in re.findall(r"\.name:\s+(\S+)\s+\.private_segment_fixed_size:\s+(\d+)", notes))
    return out


@pytest.mark.skipif(READELF is None, reason="llvm-readelf not installed")
def test_hot_kernels_keep_to_registers(tmp_path):
    got = scratch_bytes(tmp_path)
    assert len(got) > 100
    for name, most in (("k_vq_run_f16ILi9", 0), ("k_vq_run_f16ILi5", 0),
                       ("k_vq_run_f16ILi4", 16),                         # three registers, before its loop
                       ("k_vq_mfma_run", 0), ("k_vq_encode", 0), ("k_vq_scan", 0), ("k_kda", 0), ("k_apply_p6", 0),
                       ("k_lut_p6", 0), ("k_shared_h", 0), ("k_rmsnorm", 0)):
        hits = {k: v for k, v in got.items() if name in k}
        assert hits and max(hits.values()) <= most, hits

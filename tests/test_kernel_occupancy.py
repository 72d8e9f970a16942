"""Waves a SIMD that the stage kernels' registers leave room for, from the built library's own kernel descriptions.
A gfx950 SIMD has 512 VGPRs, given out in eights; several N-phase kernels lie within a few registers of the next
lower wave count, where an edit elsewhere in the face arithmetic costs 10 to 30% of their time unseen."""
import os
import re
import struct
import subprocess

import pytest

from compas_amd.build import LIB

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    """The gfx950 code objects of the offload bundles in a host library."""
    at = blob.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", blob, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            p += 24
            if b"gfx950" in blob[p:p + idlen] and size:
                yield blob[at + off:at + off + size]
            p += idlen
        at = blob.find(MAGIC, p)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(LIB):
        from compas_amd.build import build
        build()
    readelf = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
    out = {}
    path = str(tmp_path_factory.mktemp("co") / "co.elf")
    with open(LIB, "rb") as f:
        blob = f.read()
    for co in _code_objects(blob):
        with open(path, "wb") as f:
            f.write(co)
        notes = subprocess.run([readelf, "--notes", path], capture_output=True, text=True, check=True).stdout
        for k in re.split(r"\n  - \.", notes)[1:]:
            name = re.search(r"\.name:\s+(\S+)", k)
            if name:
                out[name[1]] = {q: int(re.search(r"\.%s:\s+(\d+)" % q, k)[1])
                                for q in ("vgpr_count", "vgpr_spill_count")}
    return out


# (kernel, dimension, scheme, Riemann solver or Phase-Field form, THINC, last argument, waves). Schemes: 0 Godunov,
# 1 MUSCL, 5 WENO5, 6 WENO5B; 1 HLL, 2 HLLC, 10 the Phase-Field mixture flux. Last: phases (k_stage), 0 the
# two-phase model, or the direction (k_faces).
STAGE = [("k_stage", 2, 0, 1, 0, 2, 5), ("k_stage", 2, 1, 1, 0, 2, 4), ("k_stage", 2, 1, 2, 0, 2, 4),
         ("k_stage", 2, 5, 2, 0, 2, 4), ("k_stage", 2, 1, 1, 0, 3, 3), ("k_stage", 2, 1, 2, 0, 3, 3),
         ("k_stage", 2, 5, 2, 0, 3, 3), ("k_stage", 3, 5, 1, 0, 2, 4), ("k_stage", 3, 5, 2, 0, 2, 4),
         ("k_stage", 3, 1, 2, 0, 2, 3), ("k_stage", 3, 5, 2, 0, 3, 3), ("k_stage", 2, 1, 10, 0, 2, 4),
         ("k_stage", 2, 1, 10, 0, 3, 3), ("k_stage", 3, 5, 10, 0, 2, 4)]


@pytest.mark.parametrize("name,dim,scheme,riemann,thinc,last,waves", STAGE)
def test_waves_per_simd(kernels, name, dim, scheme, riemann, thinc, last, waves):
    key = "%d%sILi%dELi%dELi%dELb%dELi%dE" % (len(name), name, dim, scheme, riemann, thinc, last)
    found = [v for k, v in kernels.items() if key in k]
    assert len(found) == 1
    vgpr = found[0]["vgpr_count"]
    assert 512 // (-(-vgpr // 8) * 8) >= waves, vgpr
    assert found[0]["vgpr_spill_count"] == 0


def test_work_list_kernels_keep_two_waves(kernels):
    """Every work-list kernel leaves room for two workgroups a CU, whatever occupancy it is built for."""
    lists = {k: v["vgpr_count"] for k, v in kernels.items() if "k_stage_listILi" in k}
    assert len(lists) >= 48 and max(lists.values()) <= 256

"""Registers, scratch and LDS of the sweep kernels in the built library, from
the code object's own metadata (no GPU): a change that makes an instance of
some solver or order spill, or takes a workgroup's LDS past what lets four
into a CU, shows here and not only in a profile of the default scheme."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from qasmhd_amd import build

LLVM = "/opt/rocm/llvm/bin"


def _code_objects(path, tmp):
    """The gfx950 code objects of the library's offload bundles (one per unit)."""
    fat = os.path.join(tmp, "fat")
    subprocess.run([os.path.join(LLVM, "llvm-objcopy"), "--dump-section", ".hip_fatbin=" + fat, path,
                    os.path.join(tmp, "lib")], check=True, capture_output=True)
    data = open(fat, "rb").read()
    out = []
    for at in (m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)):
        p = at + 24
        n, = struct.unpack_from("<Q", data, p)
        p += 8
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + ln].decode()
            p += 24 + ln
            if "gfx950" in name and size:
                f = os.path.join(tmp, "co%d" % len(out))
                open(f, "wb").write(data[at + off:at + off + size])
                out.append(f)
    return out


@pytest.fixture(scope="module")
def sweeps(tmp_path_factory):
    if not os.path.exists(build.lib_path()):
        build.build()
    if not shutil.which(os.path.join(LLVM, "llvm-readelf")):
        pytest.skip("no llvm-readelf")
    res = {}
    for f in _code_objects(build.lib_path(), str(tmp_path_factory.mktemp("co"))):
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", f], check=True, capture_output=True,
                               text=True).stdout
        for k in re.split(r"\n\s+- \.a", notes)[1:]:
            name = re.findall(r"\.name:\s+(_Z\S+)", k)
            if name and "k_sweep" in name[0]:
                res[name[0]] = {m: int(re.search(r"\.%s:\s+(\d+)" % m, k).group(1))
                                for m in ("private_segment_fixed_size", "group_segment_fixed_size", "vgpr_count")}
    return res


def test_all_sweep_instances_found(sweeps):
    # 2D: x and y, single and batch, 4 solvers x 4 orders, FP64, FP32 and
    # contracted FP64; with gravity x and y; 3D: 3 axes in 3 precisions
    assert len(sweeps) == 16 * (4 * 3 + 2 + 3 * 3)


def test_no_sweep_spills(sweeps):
    # 20 bytes: Roe and MLAU with gravity (measured faster than a wave less)
    bad = {k: v for k, v in sweeps.items() if v["private_segment_fixed_size"] > 20}
    assert not bad


def test_lds_lets_four_workgroups_into_a_cu(sweeps):
    # 160 KB per CU, allocated in units of 1280 bytes
    bad = {k: v for k, v in sweeps.items() if -(-v["group_segment_fixed_size"] // 1280) * 1280 * 4 > 160 * 1024}
    assert not bad

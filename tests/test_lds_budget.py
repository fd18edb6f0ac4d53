"""LDS of the lane sums' workgroups, as the compiler reports it: the wave buffers
(dynamic) and whatever a kernel holds beside them (static) let a compute unit
take the sixteen waves its registers allow."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "zccl_amd", "csrc")
LDS_PER_CU, WAVES = 160 * 1024, 16


def test_sixteen_waves_of_a_sum_fit_a_compute_unit(tmp_path):
    from zccl_amd import build as zb

    try:
        hipcc = zb.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    src = open(os.path.join(CSRC, "zccl_lane.hip")).read()
    buf = int(re.search(r"constexpr uint32_t kOutBuf = (\d+);", src).group(1))
    asm = str(tmp_path / "lane.s")
    flags = [f for f in zb.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([hipcc, *flags, "-I", os.path.join(ROOT, "include"), "-I", CSRC, "--cuda-device-only", "-S",
                    os.path.join(CSRC, "zccl_lane.hip"), "-o", asm], check=True, capture_output=True)
    meta = re.findall(r"\.group_segment_fixed_size: (\d+).*?\.max_flat_workgroup_size: (\d+).*?\.name:\s+(\S+)",
                      open(asm).read(), re.S)
    sums = [(n, int(lds), int(threads) // 64) for lds, threads, n in meta if "homsum_lane" in n]
    assert len(sums) >= 11
    for name, static, waves in sums:
        assert (static + waves * buf) * (WAVES // waves) <= LDS_PER_CU, (name, static, waves)

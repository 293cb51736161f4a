"""What the compiler gives the kernels whose speed hangs on their occupancy, from its own
kernel-resource-usage remarks on this library's sources (no GPU)."""
import importlib.util
import re
import shutil
import subprocess

import pytest

from gschism_amd import build


def _usage(source, tmp_path):
    """{demangled kernel name: {"VGPRs": .., "Occupancy": .., "ScratchSize": ..}} of one source."""
    cmd = [build.HIPCC, *build.COMMON, *build.HIP_FLAGS, "-Rpass-analysis=kernel-resource-usage", "--cuda-device-only",
           "-c", str(build.CSRC / source), "-o", str(tmp_path / "device.o")]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    names = subprocess.run(["c++filt"], input=r.stderr, capture_output=True, text=True).stdout
    out, cur = {}, None
    for line in names.splitlines():
        m = re.search(r"remark: +Function Name: (?:void )?(.*?)\(", line)
        if m:
            cur = out.setdefault(m.group(1), {})
        m = re.search(r"remark: +(VGPRs|Occupancy|ScratchSize)(?: \[[^\]]*\])?: (\d+)", line)
        if m and cur is not None:
            cur[m.group(1)] = int(m.group(2))
    return out


needs_compiler = pytest.mark.skipif(not (shutil.which(build.HIPCC) and shutil.which("c++filt")), reason="needs hipcc and c++filt")


@needs_compiler
def test_narrow_jacobi_phases_keep_their_waves(tmp_path):
    """Batched and large Jacobi solves run the 256-thread phases at as many waves a SIMD as their
    registers give: 7 for the FP32 phase A (71 VGPRs), 4 for FP64 up to 4 rows per thread."""
    u = _usage("pcg_kernels.hip", tmp_path)
    for rpt in (1, 2, 4, 8):
        assert u[f"gsh::k_pcg_phase_a<float, {rpt}, false>"]["Occupancy"] >= 7
        assert u[f"gsh::k_pcg_phase_a<double, {rpt}, false>"]["Occupancy"] >= (3 if rpt == 8 else 4)
    for name, k in u.items():
        if "k_pcg_phase" in name or "k_pcg_run" in name:
            assert k["ScratchSize"] == 0, name


@needs_compiler
def test_momentum_of_few_levels_keeps_its_waves(tmp_path):
    """Waves of few levels hold few loads: on up to 4 and 8 levels (2 and 4 items a lane) they leave
    registers for 5 and 4 waves a SIMD, where the 16 items of many levels leave 2."""
    u = _usage("mesh_kernels.hip", tmp_path)
    for items, waves in ((2, 5), (4, 4), (8, 3), (16, 2)):
        k = u[f"gsh::k_momentum<{items}>"]
        assert k["Occupancy"] >= waves and k["ScratchSize"] == 0


@needs_compiler
def test_backtracking_counters_are_of_this_kernel(tmp_path):
    """bench.py divides the committed counters of k_backtrack by its own time: the profile names a
    kernel that these sources build, with its registers and waves."""
    spec = importlib.util.spec_from_file_location("bench", build.CSRC.parents[1] / "bench.py")
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    bound = bench.backtrack_bound()
    text = (build.CSRC.parents[1] / "profiles" / "backtrack_counters_channel-1024x1024.md").read_text()
    k = _usage("mesh_kernels.hip", tmp_path)["gsh::" + re.search(r"`(k_backtrack<[^`]*>)`", text).group(1)]
    assert bound["vgprs"] == k["VGPRs"] and bound["waves_per_simd"] <= k["Occupancy"]


@needs_compiler
def test_backtracking_forms_keep_their_waves(tmp_path):
    """One sigma with the kept velocities in LDS four waves a SIMD, which flows that change element in each
    substep need; in registers, for grids that do not fill the chip and on z columns, three; short lists,
    which keep nothing, four. No scratch on one sigma and flat beds."""
    u = _usage("mesh_kernels.hip", tmp_path)
    for variant in ("0, false, true", "0, false, false"):
        assert u[f"gsh::k_backtrack<{variant}, true>"]["Occupancy"] >= 4
        assert u[f"gsh::k_backtrack<{variant}, false>"]["Occupancy"] >= 3
    assert u["gsh::k_backtrack<1, false, false, false>"]["Occupancy"] >= 3
    assert u["gsh::k_backtrack<2, false, false, false>"]["Occupancy"] >= 4
    for lv in ("true", "false"):
        assert u[f"gsh::k_backtrack<0, false, true, {lv}>"]["ScratchSize"] == 0

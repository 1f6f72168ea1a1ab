"""The build script's own guard: kernels whose K loop is hand-placed register text may not use scratch memory."""
import importlib.util
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _build_module():
    spec = importlib.util.spec_from_file_location("_dfa_build_checks", os.path.join(ROOT, "deeplink.framework_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_scratch_guard_reads_the_resource_usage_remarks():
    b = _build_module()
    remark = "gemm.hip:806:1: remark: {} [-Rpass-analysis=kernel-resource-usage]"
    clean = "\n".join(remark.format(t) for t in ["Function Name: _ZN3amd19gemmMfma4WaveKernelIDF16bLi0EEEvNS_8MfmaArgsE", "    VGPRs: 250",
                                                  "    ScratchSize [bytes/lane]: 0", "    SGPRs Spill: 0", "    VGPRs Spill: 0"])
    assert b.scratch_users(clean, ("gemmMfma4WaveKernel",)) == []
    spilled = clean.replace("ScratchSize [bytes/lane]: 0", "ScratchSize [bytes/lane]: 52").replace("VGPRs Spill: 0", "VGPRs Spill: 13")
    bad = b.scratch_users(spilled, ("gemmMfma4WaveKernel",))
    assert len(bad) == 2 and "ScratchSize" in bad[0] and "VGPRs Spill: 13" in bad[1]
    # scalar registers parked in lanes of a vector register are not scratch
    lanes = clean.replace("SGPRs Spill: 0", "SGPRs Spill: 2")
    assert b.scratch_users(lanes, ("gemmMfma4WaveKernel",)) == []
    # another kernel's scratch is not this guard's business
    other = spilled.replace("gemmMfma4WaveKernel", "gemmFmaKernel")
    assert b.scratch_users(other, ("gemmMfma4WaveKernel",)) == []
    assert "gemm.hip" in b.NO_SCRATCH_KERNELS


def test_libraries_are_linked_where_the_host_module_does_not_build(monkeypatch):
    b = _build_module()
    linked = []

    def run(cmd, **_):
        linked.append(cmd[cmd.index("-o") + 1])
        return subprocess.CompletedProcess(cmd, 0, "", "")

    monkeypatch.setattr(b, "compile_one", lambda src, obj: (src, 0, ""))
    monkeypatch.setattr(b, "build_host", lambda: (b.HOST_SOURCE, 1, "no torch headers"))
    monkeypatch.setattr(b.subprocess, "run", run)
    with pytest.raises(RuntimeError, match="host module"):
        b.build()
    assert linked == [b.TARGETS["impl"]["out"], b.TARGETS["rt"]["out"]]
    linked.clear()
    monkeypatch.setattr(b, "compile_one", lambda src, obj: (src, int(src.endswith("gemm.hip")), ""))
    with pytest.raises(RuntimeError, match="compilation failed"):
        b.build()
    assert linked == []


DYNAMIC_LDS_PROBE = r"""
#include <cstdio>
#include <map>
#include "common.hpp"
// in place of the runtime's: the largest launch that a kernel was allowed on a device, and whether that can be raised
static int device = 0, calls = 0;
static bool refuse = false;
static std::map<std::pair<const void*, int>, int> allowed;
extern "C" hipError_t hipGetDevice(int* d) { return *d = device, hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute, int bytes) {
  ++calls;
  if (refuse) return hipErrorInvalidValue;
  return allowed[{f, device}] = bytes, hipSuccess;
}
int main() {
  static char a, b;  // kernels
  struct { const void* kernel; int device, bytes; bool refuse; } launches[] = {
      {&a, 0, 34880, false}, {&a, 0, 66560, false}, {&a, 0, 40000, false}, {&b, 0, 1000, false}, {&a, 1, 66560, true}, {&a, 1, 50000, false}, {&a, 1, 66560, false}};
  for (auto& l : launches) {
    device = l.device, refuse = l.refuse;
    const hipError_t e = amd::allowDynamicLds(l.kernel, l.bytes);
    if (l.refuse ? e == hipSuccess : e != hipSuccess || allowed[{l.kernel, l.device}] < l.bytes) return printf("%d bytes on device %d\n", l.bytes, l.device), 1;
  }
  const int before = calls;
  for (int i = 0; i < 3; ++i) (void)amd::allowDynamicLds(&a, 66560);
  return calls == before ? 0 : 2;  // what was allowed is not asked for again
}
"""


def test_dynamic_lds_limit_follows_the_largest_launch(tmp_path):
    """A kernel launched with more dynamic LDS than its launches before needs its limit raised, on each device of its own."""
    b = _build_module()
    (tmp_path / "probe.cpp").write_text(DYNAMIC_LDS_PROBE)
    exe = str(tmp_path / "probe")
    src = b.TARGETS["impl"]["dir"]
    cmd = [b.hipcc(), "-O0", "-std=c++17", "-w", "--offload-host-only", f"-I{b.INCLUDE}", f"-I{src}", "-x", "hip", str(tmp_path / "probe.cpp"),
           os.path.join(src, "runtime_glue.cpp"), "-o", exe, "-Wl,--unresolved-symbols=ignore-all"]
    subprocess.run(cmd, check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


NARROW_STAGES_PROBE = r"""
#include <cstdio>
#include "narrow_stream.hip"
// Every copy that a workgroup issues: those of the walk and, as its loads are counted, those past the last stage.
int main() {
  for (int stages = 1; stages <= 40; ++stages)
    for (int start = 0; start < stages; ++start)
      for (int places = 3; places <= 4; ++places)
        for (int c = 0; c < stages + places - 1; ++c) {
          const int at = amd::narrowStage(c, start, stages);
          if (at < 0 || at >= stages) return printf("copy %d of %d stages from %d: stage %d\n", c, stages, start, at), 1;
          if (c < stages && at != (c + start) % stages) return printf("copy %d of %d stages from %d\n", c, stages, start), 2;
        }
  return 0;
}
"""


def test_copies_past_the_last_stage_keep_their_offset_inside_the_buffer(tmp_path):
    """The scalar offset of a buffer load counts against the size in the descriptor: also a copy that fetches nothing
    (its lanes lie past the end) stays at a stage that the rows have."""
    b = _build_module()
    (tmp_path / "probe.cpp").write_text(NARROW_STAGES_PROBE)
    exe = str(tmp_path / "probe")
    src = b.TARGETS["impl"]["dir"]
    cmd = [b.hipcc(), "-O0", "-std=c++17", "-w", "--offload-host-only", f"-I{b.INCLUDE}", f"-I{src}", "-x", "hip", str(tmp_path / "probe.cpp"),
           "-o", exe, "-Wl,--unresolved-symbols=ignore-all"]
    subprocess.run(cmd, check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


RECTANGLES_PROBE = r"""
#include <cstdio>
#include "gemm_weight_stream.hip"
int amd::computeUnits() { return 256; }
int main() {
  long m, n, k, gated;
  while (scanf("%ld %ld %ld %ld", &m, &n, &k, &gated) == 4) {
    amd::WeightStreamArgs a;
    a.siluMul = gated != 0;
    const float us = amd::weightStreamPlan(m, n, k, &a);
    printf("%d %d %d %d\n", us > 0, a.tilesM, a.rowsPerWg, a.tilesPerWg);
  }
}
"""


def test_rectangles_of_the_gpu_tests_reach_every_tile(tmp_path):
    """The cases that the GPU tests give to the kernel whose rectangles are cut to the chip: which tile each takes on 256
    compute units, and that no tile is left out."""
    from tests.test_gpu_attention_gemm import RECTANGLES

    b = _build_module()
    (tmp_path / "probe.cpp").write_text(RECTANGLES_PROBE)
    exe = str(tmp_path / "probe")
    src = b.TARGETS["impl"]["dir"]
    cmd = [b.hipcc(), "-O0", "-std=c++17", "-w", "--offload-host-only", f"-I{b.INCLUDE}", f"-I{src}", "-x", "hip", str(tmp_path / "probe.cpp"),
           "-o", exe, "-Wl,--unresolved-symbols=ignore-all"]
    subprocess.run(cmd, check=True)
    text = "".join(f"{m} {n} {k} {int(form == 'gated')}\n" for _, _, form, m, n, k, _ in RECTANGLES)
    lines = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
    assert len(lines) == len(RECTANGLES)
    for case, line in zip(RECTANGLES, lines):
        found, tiles_m, rows, tiles = map(int, line.split())
        tm, tn = max(4, -(-rows // 32)), next(w for w in (2, 4, 6, 8, 12) if tiles <= w) // 2
        assert found and (tm, tn) == case[:2], (case, line)
        assert tiles_m * rows >= case[3] > (tiles_m - 1) * rows
    tiles = {case[:2] for case in RECTANGLES}
    assert tiles == {(tm, tn) for tm in range(4, 9) for tn in (1, 2, 3, 4, 6) if (tm, tn) != (8, 1) and not (tn == 6 and tm > 5)}


NARROW_FORMS_PROBE = r"""
#include <cstdio>
#include "narrow_stream.hip"
int amd::computeUnits() { return 256; }
int main() {
  amd::NarrowStreamArgs a;
  int int8;
  while (scanf("%d %d %d %d", &int8, &a.M, &a.N, &a.K) == 4) {
    a.int8B = int8 != 0, a.lda = a.ldb = a.K, a.ldo = a.N;
    printf("%d\n", (int)amd::narrowStreamPays(a));
  }
}
"""


def test_narrow_streams_of_the_gpu_tests_reach_every_form(tmp_path):
    """The cases that the GPU tests give to the kernel for few columns a compute unit: that it takes them on 256 units, and that
    no row group, number of column tiles or weight type is left out."""
    from tests.test_gpu_attention_gemm import NARROW_STREAMS

    b = _build_module()
    (tmp_path / "probe.cpp").write_text(NARROW_FORMS_PROBE)
    exe = str(tmp_path / "probe")
    src = b.TARGETS["impl"]["dir"]
    cmd = [b.hipcc(), "-O0", "-std=c++17", "-w", "--offload-host-only", f"-I{b.INCLUDE}", f"-I{src}", "-x", "hip", str(tmp_path / "probe.cpp"),
           "-o", exe, "-Wl,--unresolved-symbols=ignore-all"]
    subprocess.run(cmd, check=True)
    text = "".join(f"{int(int8)} {m} {n} {k}\n" for int8, _, _, m, n, k in NARROW_STREAMS)
    lines = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split()
    assert lines == ["1"] * len(NARROW_STREAMS), [c for c, l in zip(NARROW_STREAMS, lines) if l != "1"]
    for int8, groups, tiles, m, n, k in NARROW_STREAMS:
        assert groups == -(-m // 16) and tiles == -(-(-(-n // 256)) // 16)
    every = {(int8, g, t) for int8 in (False, True) for g in (1, 2, 3, 4) for t in (1, 2)} | {(True, 1, 3)}
    assert {c[:3] for c in NARROW_STREAMS} == every
    assert {c[:3] for c in NARROW_STREAMS if c[5] % 128 == 0 and not c[0]} == {c for c in every if not c[0]}  # (rotated)

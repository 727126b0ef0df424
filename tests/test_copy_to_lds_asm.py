"""CopyToLds (buffer -> LDS copies written as assembly) in code compiled around it (CPU test over the
compiler's assembly): five wait states between a VALU write of a scalar operand and the load that reads
it, which the compiler does not add inside assembly, and m0 declared as overwritten."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "crucible-strix-halo_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
FLAGS = ["--offload-arch=gfx950", "--offload-device-only", "-O3", "-std=c++20", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]

SRC = """
using namespace cx;
// The scalar offset of each copy comes straight from a VALU write.
extern "C" __global__ void OffsetFromLane(const uint32_t* src, uint32_t* out, int n) {
  __shared__ __align__(16) uint32_t s[1024];
  const u32x4_t r = MakeRsrcWords(src, 4096);
  const uint32_t lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)(LdsChar*)s);
  for (int i = 0; i < n; ++i) {
    CopyToLds<4>(r, threadIdx.x * 16, (uint32_t)__builtin_amdgcn_readfirstlane((int)out[2 * i]), lds);
    CopyToLds<1>(r, threadIdx.x * 4, (uint32_t)__builtin_amdgcn_readfirstlane((int)out[2 * i + 1]), lds + 1024);
  }
  WaitLoadsBarrier<0>();
  out[threadIdx.x] = s[threadIdx.x];
}
// Runs of copies.
extern "C" __global__ void Runs(const uint32_t* src, uint32_t* out, int n) {
  __shared__ __align__(16) uint32_t s[2048];
  const uint32_t lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)(LdsChar*)s);
  CopyToLds<4, 6, 1024>(MakeRsrcWords(src, 65536), threadIdx.x * 16, 64, lds, (uint32_t)n);
  CopyToLds<1, 3, 256>(MakeRsrcWords(src, 65536), threadIdx.x * 4, 64, lds + 6144, 256u);
  WaitLoadsBarrier<0>();
  out[threadIdx.x] = s[threadIdx.x];
}
// m0 holds the same value for another instruction before and after the copy (compiled, never run).
extern "C" __global__ void OtherUseOfM0(const uint32_t* src, uint32_t* out, int a) {
  __shared__ __align__(16) uint32_t s[1024];
  __builtin_amdgcn_s_sendmsg(1, a);
  CopyToLds<4>(MakeRsrcWords(src, 4096), threadIdx.x * 16, 0, 0);
  __builtin_amdgcn_s_sendmsg(1, a);
  WaitLoadsBarrier<0>();
  out[threadIdx.x] = s[threadIdx.x];
}
"""


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not Path(HIPCC).exists():
        pytest.skip("no hipcc")
    src = tmp_path_factory.mktemp("asm") / "copies.hip"
    src.write_text(f'#include "{CSRC}/common.hpp"\n{SRC}')
    text = subprocess.run([HIPCC, *FLAGS, "-S", str(src), "-o", "-"], check=True, capture_output=True, text=True).stdout
    out = {}
    for name in ("OffsetFromLane", "Runs", "OtherUseOfM0"):
        body = re.search(rf"^{name}:.*?s_endpgm", text, re.S | re.M).group(0)
        out[name] = [ln.split(";")[0].strip() for ln in body.splitlines() if re.match(r"\s+[sv]_|\s+(buffer|global|ds)_", ln)]
    return out


def _sgprs(text):
    regs = set()
    for lo, hi in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        regs |= set(range(int(lo), int(hi) + 1))
    return regs | {int(n) for n in re.findall(r"\bs(\d+)\b", text)}


def test_wait_states_before_the_load(kernels):
    code = kernels["OffsetFromLane"]
    loads = [i for i, c in enumerate(code) if re.match(r"buffer_load.* lds$", c)]
    assert len(loads) >= 2
    seen = 0
    for i in loads:
        reads, states = _sgprs(code[i]), 0
        for c in reversed(code[:i]):
            if re.match(r"v_readfirstlane|v_readlane", c):
                if _sgprs(c.split(",")[0]) & reads:
                    seen += 1
                    assert states >= 5, (code[i], c, states)
                    break
            m = re.match(r"s_nop (\d+)", c)
            states += int(m.group(1)) + 1 if m else 1
    assert seen >= 2  # both forms were compiled with an offset from a VALU write


def test_runs_advance_offset_and_m0(kernels):
    # Each further copy: m0 and the offset advanced by scalar instructions, one of them between m0's write
    # and the load (m0's wait state); nothing else between the copies of a run.
    code = kernels["Runs"]
    loads = [i for i, c in enumerate(code) if re.match(r"buffer_load.* lds$", c)]
    assert [c.split()[0] for c in code if re.match(r"buffer_load.* lds$", c)] == 6 * ["buffer_load_dwordx4"] + 3 * ["buffer_load_dword"]
    for i, j in zip(loads, loads[1:]):
        if i == loads[5]:
            continue  # from the first run to the second
        off = re.search(r", (s\d+) offen", code[j]).group(1)
        assert j == i + 3
        assert re.match(r"s_add_u32 m0, m0, 0x(400|100)$", code[i + 1]), code[i:j + 1]
        assert re.match(rf"s_add_u32 {off}, {off}, s\d+$", code[i + 2]), code[i:j + 1]


def test_m0_is_set_again_after_a_copy(kernels):
    code = kernels["OtherUseOfM0"]
    load = next(i for i, c in enumerate(code) if re.match(r"buffer_load.* lds$", c))
    msg = next(i for i, c in enumerate(code) if i > load and c.startswith("s_sendmsg"))
    assert any(re.match(r"s_mov_b32 m0", c) for c in code[load + 1:msg]), code[load:msg + 1]

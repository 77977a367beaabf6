"""The load from memory to LDS that the compiler does not know, as it is compiled: no vector memory instruction reads a scalar register fewer than five wait states
after a vector instruction wrote it, and one instruction stands between m0 and the load."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

# the base in lanes of a vector register: a block table's entry, or a scalar register that was spilled
PROBE = """
#include "nv_common.h"
namespace nv {
__global__ void probe(const uint32_t* at, int n, float* out) {
    __shared__ float tile[1024];
    const uint32_t lo = at[threadIdx.x], hi = at[threadIdx.x + 64];
    for (int i = 0; i < n; ++i) {
        const uint64_t base = (uint64_t)__builtin_amdgcn_readlane(hi, i) << 32 | (uint32_t)__builtin_amdgcn_readlane(lo, i);
        lds_load16((const void*)base, threadIdx.x * 16, lds_address(tile) + (i & 3) * 1024);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    out[threadIdx.x] = tile[threadIdx.x];
}
}  // namespace nv
"""


def _scalars(text):
    """Numbers of the scalar registers that an operand list names."""
    out = set()
    for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        out.update(range(int(a), int(b) + 1))
    out.update(int(a) for a in re.findall(r"\bs(\d+)\b", text))
    return out


def hazards(asm):
    """Vector memory instructions that read a scalar register too soon after a vector instruction wrote it, or m0 in the next instruction, in a listing taken line by
    line."""
    written, found, m0, clock = {}, [], -9, 0
    for line in asm.splitlines():
        line = line.split(";")[0].strip()
        if not line or line.startswith((".", "//")) or line.endswith(":"):
            continue
        op, _, rest = line.partition(" ")
        ops = [x.strip() for x in rest.split(",")]
        clock += 1 + (int(ops[0]) if op == "s_nop" else 0)
        if op.startswith(("global_", "buffer_", "flat_", "scratch_")):
            found += [line for r in _scalars(rest) if clock - 1 - written.get(r, -9) < 5]
            if "lds" in op and clock - 1 - m0 < 1:
                found.append(line)
        elif op.startswith("v_"):
            for r in _scalars(ops[0]):
                written[r] = clock
        elif op.startswith("s_"):
            if ops and ops[0] == "m0":
                m0 = clock
            for r in _scalars(ops[0] if ops else ""):
                written.pop(r, None)
    return found


def test_the_listing_is_read():
    soon = "v_readlane_b32 s4, v1, s2\n s_mov_b32 m0, s3\n s_nop 0\n global_load_lds_dwordx4 v0, s[4:5]\n"
    assert len(hazards(soon)) == 1 and not hazards(soon.replace("s_nop 0", "s_nop 4"))
    assert not hazards("v_readlane_b32 s4, v1, s2\n s_mov_b32 m0, s3\n s_mov_b64 s[6:7], s[4:5]\n global_load_lds_dwordx4 v0, s[6:7]\n")
    assert len(hazards("s_mov_b32 m0, s3\n global_load_lds_dwordx4 v0, s[6:7]\n")) == 1


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_addresses_from_vector_registers(tmp_path):
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(PROBE)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-device-only", "-O3", "-std=c++17", "-S", "-w", "-I", os.path.join(ROOT, "nano-vllm_amd", "csrc"),
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", str(src), "-o", str(out)], check=True, capture_output=True, timeout=120)
    asm = out.read_text()
    body = asm[asm.index("probe"):asm.index("s_endpgm")]
    assert "global_load_lds_dwordx4" in body and "v_readlane_b32" in body
    assert hazards(body) == []

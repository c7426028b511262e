"""The inline assembly that moves 16 bytes a lane from global memory to LDS (fastmax_amd/csrc/fm_tiles.h) hides a memory
instruction from the compiler, so what the compiler would see to is checked on the listing of a probe: a base address
that comes out of a lane is followed by five wait states before the instruction that reads it, and m0 is written by the
compiler itself, so that a value it holds there is not taken to survive the transfer.  hipcc cross-compiles for gfx950 without a GPU."""
import os
import re
import subprocess

from fastmax_amd import build

PROBE = """
#include "fm_tiles.h"
using C = tiles::Copy<64, 4>;
__global__ void base_from_a_lane(const uint64_t* p, uint32_t off) {
  const uint64_t b = p[threadIdx.x];
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b), hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
  C::transfer(reinterpret_cast<const void*>(((uint64_t)hi << 32) | lo), off + threadIdx.x * 16u, 0u);
}
__global__ void m0_between(const char* p, uint32_t off, uint32_t x, uint32_t* out) {
  uint32_t a, b;
  asm volatile("s_mov_b32 %0, %1" : "={m0}"(a) : "s"(x));
  C::transfer(p, off + threadIdx.x * 16u, 1024u);
  asm volatile("s_mov_b32 %0, %1" : "=s"(b) : "{m0}"(a));
  out[threadIdx.x] = b;
}
"""


def listing(tmp_path):
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(PROBE)
    subprocess.run([build.HIPCC, *build.HIP_FLAGS, "--cuda-device-only", "-S", f"-I{build.INCLUDE}", f"-I{build.CSRC}", str(src),
                    "-o", str(out)], check=True, capture_output=True)
    bodies = {}
    for name in ("base_from_a_lane", "m0_between"):
        m = re.search(rf"^_Z\d+{name}\w*:.*?s_endpgm", out.read_text(), re.S | re.M)
        bodies[name] = [ln.split(";")[0].strip() for ln in m.group(0).splitlines() if ln.startswith("\t")]
        bodies[name] = [ln for ln in bodies[name] if ln and not ln.startswith(".")]
    return bodies


def test_transfer_waits_for_its_base_and_owns_m0(tmp_path):
    bodies = listing(tmp_path)

    body = bodies["base_from_a_lane"]
    at = next(i for i, ln in enumerate(body) if ln.startswith("global_load_lds"))
    pair = re.search(r"s\[(\d+):(\d+)\]", body[at])
    regs = {f"s{pair.group(1)}", f"s{pair.group(2)}"}
    states, wrote = 0, False
    for ln in reversed(body[:at]):
        op, args = ln.split(None, 1)
        if op.startswith("v_") and args.split(",")[0] in regs:
            wrote = True
            break
        states += int(args, 0) + 1 if op == "s_nop" else 1
    assert wrote and states >= 5, (states, body)

    body = bodies["m0_between"]
    at = next(i for i, ln in enumerate(body) if ln.startswith("global_load_lds"))
    assert any(re.match(r"s_mov_b32 s\d+, m0", ln) for ln in body[:at]), body   # saved before ..
    assert any(re.match(r"s_mov_b32 m0, s\d+", ln) for ln in body[at:]), body   # .. and put back behind the transfer

"""Stores through the L2 are the compiler's, which keeps what may not be written.

A store of more than 8 bytes still reads its data while the next instructions
issue: on gfx950 a vector instruction may rewrite those registers only after two
wait states.  The compiler puts them in behind the stores that it emits, and
sees none in inline assembly.
"""
import glob
import os
import re
import subprocess

import pytest

import poplibs_amd as pa

CSRC = os.path.join(os.path.dirname(pa.__file__), "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

PROBE = r"""
#include "igemm_common.hpp"
using namespace mxk;
// the data change behind each store, in the registers that it reads
__global__ void rewritten(uint32_t *out, const uintx4 *in, int n) {
  const __amdgpu_buffer_rsrc_t to = bufferOf(out, 1u << 30);
  uintx4 v = in[threadIdx.x];
#pragma unroll 1
  for (int i = 0; i != n; ++i) {
    storeThrough(to, threadIdx.x * 16, v);
    v ^= 0x5a5a5a5au;
    storeThrough(to, threadIdx.x * 16 + 16384, v);
    v += 1u;
  }
}
"""


def test_no_memory_access_in_inline_assembly():
    found = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        with open(path) as f:
            text = f.read()
        for block in re.findall(r"\basm\b[^;]*;", text):
            if re.search(r"\b(global|buffer|flat|scratch|ds)_(load|store|read|"
                         r"write|atomic)", block):
                found.append((os.path.basename(path), block.split("\n")[0]))
    assert not found


def registers(text):
    """The vector registers that an operand names."""
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", text)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    m = re.fullmatch(r"v(\d+)", text)
    return {int(m.group(1))} if m else set()


def wait_states_before_rewrite(lines, at):
    """Wait states between the store at lines[at] and the first vector
    instruction behind it that writes what it stores; None without one."""
    operands = lines[at].split(None, 1)[1].replace(" ", "").split(",")
    data, = [r for r in map(registers, operands) if len(r) == 4]
    states = 0
    for line in lines[at + 1:]:
        op, rest = (line.split(None, 1) + [""])[:2]
        if op.startswith("s_cbranch") or op.startswith("s_endpgm"):
            break
        written = registers(rest.split(",")[0].strip())
        if op.startswith("v_") and written & data:
            return states
        states += int(rest) + 1 if op == "s_nop" else 1
    return None


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_two_wait_states_behind_a_store(tmp_path):
    source = tmp_path / "probe.hip"
    source.write_text(PROBE)
    out = tmp_path / "probe.s"
    subprocess.run(
        [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17",
         "-Wno-unused-command-line-argument", "-Xclang", "-target-feature",
         "-Xclang", "-packed-fp32-ops", "-I", CSRC, "--cuda-device-only",
         "-S", str(source), "-o", str(out)],
        check=True, capture_output=True)
    lines = [line.strip() for line in out.read_text().split("\n")]
    lines = [line for line in lines
             if line and line[0] not in ";." and not line.endswith(":")]
    stores = [i for i, line in enumerate(lines)
              if re.match(r"(buffer|global)_store_dwordx4\b", line)]
    assert stores and all("sc1" in lines[i] for i in stores)
    rewrites = [wait_states_before_rewrite(lines, i) for i in stores]
    assert any(r is not None for r in rewrites)
    assert all(r is None or r >= 2 for r in rewrites), rewrites

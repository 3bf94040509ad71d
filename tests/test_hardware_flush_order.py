"""The sums that switch the wave's denormal mode have every operand depend on
the switch: the compiler does not know that the mode changed, so an add it may
move is ordered behind the switch by its operands' addresses alone."""
import os
import re
import subprocess

from tiler_amd import build as tb

KERNELS = os.path.join(tb.CSRC, "kernels")
PROBE = """
#include <hip/hip_runtime.h>
#include "common.h"
extern "C" __global__ void probe(const float* __restrict__ x, float s, float* __restrict__ y) {
  x = tiler::flush_operands_in_hardware(x);
  y[0] = x[0] * s + x[1];
}
"""


def test_loads_depend_on_the_switch(tmp_path):
    src = tmp_path / "probe.hip"
    src.write_text(PROBE)
    ir = subprocess.run([tb.CLANG, *tb.DEVICE_FLAGS, "-S", "-emit-llvm", f"-I{KERNELS}", "-o", "-", str(src)],
                        check=True, capture_output=True, text=True).stdout
    body = ir[ir.index("@probe("):]
    body = body[:body.index("\n}")]
    zero = re.search(r'(%\d+) = tail call i64 asm sideeffect "s_setreg_imm32_b32 hwreg\(HW_REG_MODE, 4, 2\), 2', body)
    assert zero, body
    # every loaded address is reached from the value the switch produces
    reached = {zero.group(1)}
    for line in body.splitlines():
        m = re.match(r"\s*(%[\w.]+) = (\w+)", line)
        if not m:
            continue
        uses = set(re.findall(r"%[\w.]+", line.split("=", 1)[1]))
        if m.group(2) == "load":
            assert uses & reached, line
        if uses & reached:
            reached.add(m.group(1))
    assert len(re.findall(r"= load float", body)) == 2


def test_every_switch_goes_through_the_helper():
    """No other code writes the mode register."""
    sites = 0
    for name in sorted(os.listdir(KERNELS)):
        with open(os.path.join(KERNELS, name)) as fh:
            text = fh.read()
        sites += text.count("s_setreg")
        for call in re.findall(r"[^\n]*flush_operands_in_hardware\([^\n]*", text):
            assert "x = tiler::flush_operands_in_hardware(x)" in call or "const float* flush_operands" in call \
                or call.lstrip().startswith("//"), call
    assert sites == 1

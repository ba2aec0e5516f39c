"""The hand-over of results between blocks (hc_arrives_last): each wave waits for its own stores in front of the
block's barrier.  Read off the code that hipcc makes of it; nothing runs on a GPU."""
import glob
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "history-cache_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

KERNEL = """
#include "hc_common.h"
extern "C" __global__ void arrival(float *part, unsigned *ticket, float *out, float v) {
  __shared__ int flag;
  part[blockIdx.x * blockDim.x + threadIdx.x] = v;
  if (!hc_arrives_last(ticket, gridDim.x, &flag)) return;
  out[threadIdx.x] = part[threadIdx.x];
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_stores_are_waited_for_in_front_of_the_barrier(tmp_path):
    src = tmp_path / "arrival.hip"
    src.write_text(KERNEL)
    flags = re.search(r"HIPFLAGS \?= ((?:.*\\\n)*.*)", open(os.path.join(CSRC, "Makefile")).read()).group(1)
    flags = flags.replace("\\\n", " ").replace("$(ARCH)", "gfx950").replace("../../include",
                                                                            os.path.join(CSRC, "../../include"))
    asm = subprocess.run([HIPCC, *flags.split(), "-I", CSRC, "--cuda-device-only", "-S", str(src), "-o", "-"],
                         check=True, capture_output=True, text=True).stdout
    code = [line.split(";")[0].strip() for line in asm.splitlines()]
    barrier = next(i for i, line in enumerate(code) if line.startswith("s_barrier"))
    store = max(i for i, line in enumerate(code[:barrier]) if re.match(r"(global|flat|buffer)_store", line))
    assert any(re.match(r"s_waitcnt\b.*vmcnt\(0\)", line) for line in code[store:barrier]), code[store:barrier + 1]


def test_every_hand_over_goes_through_it():
    users = [os.path.basename(p) for p in glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))
             if re.search(r'__ATOMIC_(RELEASE|ACQUIRE), "agent"', open(p).read())]
    assert users == ["hc_common.h"]

"""The queue state that model kernels are compiled against (include/gpupq_device.h) keeps its layout: a
kernel built with an earlier header reads the same words, and heap h's state where it lies.  Sizes
and offsets are those of the first header with several heaps per queue."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

LAYOUT = {
    "HqState": (272, dict(last=0, m=4, mcount=8, prefix=12, deq_n=16, rest_n=20, bound_valid=24, select=32, bound=48,
                          mptr=64, chunk_target=72, chunk_n=104)),
    "GaqState": (56, dict(fel=0, front=16, cur=24, n=28, m=32, prefix=36, deq_n=40, rest_n=44)),
    "HqView": (72, dict(enq=0, deq=8, st=16, ws=24, seg_m=32, enq_cap=40, seg_cap=44, num_lps=48, heaps=52,
                        lps_per_heap=56, area=64)),
}


def test_state_layouts(tmp_path):
    lines = ["#include <cstddef>", "#include <hip/hip_runtime.h>", '#include "gpupq_device.h"']
    for name, (size, fields) in LAYOUT.items():
        lines.append("static_assert(sizeof(gpq::%s) == %d, \"%s\");" % (name, size, name))
        lines += ["static_assert(offsetof(gpq::%s, %s) == %d, \"%s.%s\");" % (name, f, at, name, f)
                  for f, at in fields.items()]
    src = tmp_path / "layout.hip"
    src.write_text("\n".join(lines) + "\n")
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    res = subprocess.run([hipcc, "--offload-arch=gfx950", "--offload-host-only", "-std=c++17", "-fsyntax-only",
                          "-Wno-invalid-offsetof", "-I", os.path.join(ROOT, "include"), str(src)],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr

"""Compiled code of the batches' hand-off kernels (cross-compiled for gfx950, no GPU). Where the two sides of a
divergent branch join, the compiler has been seen to spill registers before the instruction that makes all the lanes
active again: the lanes of the other side then read stale values back (job pointers, pixels: wrong images or worse). The
kernels' register budget is chosen so that it does not; this looks for such spills in the assembly."""
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "cuda-wavefront-pathtracer_amd")


def joins_with_early_spills(path):
    """(kernel, line) of joins that store registers to scratch before `s_or_b64 exec` brings their lanes back. A value
    loaded from scratch, changed and stored there belongs to the lanes of the region that ends."""
    out, kernel, head, pend = [], None, False, []
    for n, line in enumerate(open(path), 1):
        s = line.strip()
        if re.match(r"_Z\S+:", line):
            kernel, head, pend = line.split(":")[0], True, []
        elif re.match(r"\.LBB\S+:", line) or line.startswith("; %bb"):
            head, pend = True, []
        elif head and s and s[0] not in ";.":
            if s.startswith("s_or_b64 exec, exec,"):
                if any("Spill" in p for p in pend) and not any("Reload" in p for p in pend):
                    out.append((kernel, n))
                head = False
            elif "exec" in s or s.startswith(("s_cbranch", "s_branch", "s_endpgm")):
                head = False
            else:
                pend.append(s)
    return out


def test_no_spill_before_the_lanes_of_a_join_are_back(tmp_path):
    import sys
    sys.path.insert(0, PKG)
    import build

    def compile_for(tri):
        src, asm = str(tmp_path / ("roll%d.hip" % tri)), str(tmp_path / ("roll%d.s" % tri))
        with open(src, "w") as f:
            f.write('#include "device/kernels.h"\nnamespace cwp { namespace dev {\n')
            for lane in ("false", "true"):
                f.write("template __global__ void k_bounce_roll<8, %d, 8, kHandWaves, false, %s, true>"
                        "(const DevStepTable*, DevPaths, int);\n" % (tri, lane))
                for level in (1, 2):
                    f.write("template __global__ void k_bounce_roll_tail<%d, 8, kHandWaves, false, %s, %d>"
                            "(const DevStepTable*, DevPaths, int);\n" % (tri, lane, level))
            f.write("template __global__ void k_bounce_jobs<8, %d, 8, kHandWaves, false, true>(const DevJobTable*, DevPaths, int);\n"
                    "template __global__ void k_bounce_jobs_tail<%d, 8, kHandWaves, false>(const DevJobTable*, DevPaths, int);\n"
                    % (tri, tri))
            f.write("}}\n")
        subprocess.run([build.hipcc()] + build.HIP_FLAGS + build.INCLUDES + ["--cuda-device-only", "-S", src, "-o", asm], check=True,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
        assert open(asm).read().count("s_endpgm") >= 8
        return joins_with_early_spills(asm)

    with ThreadPoolExecutor(3) as ex:
        assert sum(ex.map(compile_for, (0, 1, 2)), []) == []

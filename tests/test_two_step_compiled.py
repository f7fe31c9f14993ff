"""The two-step kernel as compiled for gfx950, without a GPU.

Registers: a moving wall next to the values held from plane to plane (D3Q27)
must not push registers out to scratch memory in the plane loop.  Tile shapes:
every edge a state may have gets a tile that fits the kernel."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCE = """#include "{csrc}/fused_two.hpp"
namespace plb {{
void launch(const typename Prec<{v}>::S* A, typename Prec<{v}>::S* B, FusedArgs<typename Prec<{v}>::T> a, TwoGeom g) {{
    hipLaunchKernelGGL((k_pull2<{q}, {v}, {nb}, true, 1>), dim3(1), dim3(64), 0, 0, A, B, nullptr, nullptr, a, g);
}}
}}
"""


@pytest.mark.skipif(not shutil.which(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("nb", [0, 1])
@pytest.mark.parametrize("v", ["kF64", "kF32S"])
def test_moving_wall_keeps_its_registers(tmp_path, v, nb):
    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(SOURCE.format(csrc=os.path.join(ROOT, "plbpd_amd", "csrc"), q=27, v=v, nb=nb))
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S", str(src), "-o",
                    str(out)], check=True, stderr=subprocess.DEVNULL)
    spills = [int(n) for n in re.findall(r"\.vgpr_spill_count:\s+(\d+)", out.read_text())]
    # seven or eight registers stored once, before the loop, cost nothing measurable
    assert len(spills) == 1 and spills[0] <= 8, spills


SHAPES = """#include "{csrc}/fused_kernels.hpp"
#include <cstdio>
int main() {{
    const int edges[] = {{1, 2, 3, 7, 8, 9, 31, 33, 100, 331, 1023, 65537, 2147483600, 2147483647}};
    int bad = 0;
    for (int q : {{19, 27}})
        for (int sb : {{8, 4, 2}})
            for (int X : edges)
                for (int Y : edges) {{
                    const plb::TwoShape t = plb::two_shape(q, sb, X, Y);
                    const long cells = (long)(t.bx + 2) * (t.by + 2);
                    if (t.bx < 1 || t.by < 1 || t.bx > X || t.by > Y || cells > plb::two_cap(q, sb)) {{
                        std::printf("%d %d %d %d: %d x %d\\n", q, sb, X, Y, t.bx, t.by);
                        ++bad;
                    }}
                }}
    return bad != 0;
}}
"""


@pytest.mark.skipif(not shutil.which(HIPCC), reason="no hipcc")
def test_tile_shapes_of_all_edges(tmp_path):
    src, exe = tmp_path / "shapes.hip", tmp_path / "shapes"
    src.write_text(SHAPES.format(csrc=os.path.join(ROOT, "plbpd_amd", "csrc")))
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-ffp-contract=off", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", str(src), "-o", str(exe)], check=True,
                   stderr=subprocess.DEVNULL)
    run = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert run.returncode == 0, (run.returncode, run.stdout)

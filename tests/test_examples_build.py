"""The measurement probes under cudanative.jl_amd/examples, whose commands the summaries under
profiles/ give, still compile for gfx950 (device and host code; nothing is run here)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXAMPLES = os.path.join(ROOT, "cudanative.jl_amd", "examples")
PROBES = ["store_patterns.hip", "mfma_lone_wavefront.hip", "mfma_order_power.hip", "valu_issue_rate.hip"]


@pytest.mark.parametrize("name", PROBES)
def test_probe_compiles_for_gfx950(name, tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    out = tmp_path / (name + ".o")
    r = subprocess.run([hipcc, "--offload-arch=gfx950", "-O3", "-std=c++20", "-Wno-unused-result", "-c",
                        os.path.join(EXAMPLES, name), "-o", str(out)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    assert out.stat().st_size > 0


RECORDS = """
#include "gemm_tiled.hpp"
#include <cstdio>
#include <vector>
int main()
{
    struct { long tiles, batch; bool span, walk; } const cases[] = {{12, 1, false, false}, {1, 7, false, false}, {6, 5, true, false}, {300, 1, false, true}, {90, 4, true, true}};
    for (auto c : cases) {
        const long all = c.tiles * c.batch, gx = c.walk ? 256 : c.tiles, gy = c.walk ? 1 : c.batch, span = c.span ? c.tiles : 0;
        std::vector<int> seen((size_t)all, 0);
        for (long y = 0; y < gy; y++)
            for (long x = 0; x < gx; x++) {
                long tile = x + y * span;
                do {
                    const long at = miw::launch_tile((int)tile, (int)span, (unsigned)y, (unsigned)gx);
                    if (at < 0 || at >= all || seen[(size_t)at]++) {
                        std::printf("tile %ld of row %ld: record %ld of %ld", tile, y, at, all);
                        return 1;
                    }
                    tile += gx;
                } while (c.walk && tile < all);
            }
        for (int n : seen)
            if (n != 1) return 1;
    }
    return 0;
}
"""


def test_timestamp_records_stay_inside_one_per_tile(tmp_path):
    """Where the measurement build of the 256x256 ping-pong kernel writes: one record per tile of the launch, in a buffer of
    tiles x batch records, for a single problem, a batch whose members have one tile, a batch in one run, and workgroups that
    walk several tiles (the kernel's own function, on the host)."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "records.hip", tmp_path / "records"
    src.write_text(RECORDS)
    r = subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++20", "-Wno-inline-asm", "-I" + os.path.join(ROOT, "cudanative.jl_amd", "csrc"),
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", str(src), "-o", str(exe)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout

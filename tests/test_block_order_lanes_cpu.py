"""CPU: the order of pass 4's row blocks for every number of lanes a row may take, not the fewest alone (small
volumes and batches take more: plan_lanes, BatchLanes): plan_block_order / apply_block_order is a permutation of
the blocks, taken from the front (batches) as from the end (emit_block), and set by the planner's own lanes for
small volumes (miniisosurface_amd/csrc/fe_rows.h, compiled for the host with hipcc)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

PROGRAM = r"""
#include "fe_rows.h"
#include <cstdio>
#include <vector>
using namespace miso;
static long plans = 0, raised = 0, tiled = 0;
static bool permutation(int64_t W, int64_t ny, int64_t nz, int lg)
{
    const int64_t per_block = 4 * (int64_t)(64 >> lg), n = (ny * nz + per_block - 1) / per_block;
    const BlockOrder o = plan_block_order(ny, nz, W, lg);
    ++plans;
    raised += o.n0 && lg > fewest_lanes(W);
    if ((int64_t)o.n0 > n) return false;
    std::vector<char> seen(n, 0), from_end(n, 0);
    for (int64_t b = 0; b < n; ++b) {
        const int64_t a = b < (int64_t)o.n0 ? apply_block_order(o, (uint32_t)b) : b, e = n - 1 - a;
        if (a < 0 || a >= n || seen[a] || from_end[e]) return false;
        seen[a] = from_end[e] = 1;
        tiled += a != b;
    }
    return true;
}
int main()
{
    for (int64_t W : {1, 2, 3, 4, 5, 7, 8, 12, 16, 17, 31, 32, 33, 64})
        for (int64_t ny : {1, 4, 7, 32, 64, 96, 128, 200, 256, 384, 512, 640, 1000, 1024, 2048, 4096})
            for (int64_t nz : {1, 2, 3, 5, 9, 64, 127}) {
                for (int lg = fewest_lanes(W); lg <= 6; ++lg)
                    if (!permutation(W, ny, nz, lg)) {
                        printf("W=%ld ny=%ld nz=%ld lanes 2^%d\n", W, ny, nz, lg);
                        return 1;
                    }
                if (!permutation(W, ny, nz, plan_lanes(ny, nz, W))) return 1;
            }
    printf("%ld %ld %ld\n", plans, raised, tiled);
    return 0;
}
"""


@pytest.mark.skipif(not shutil.which(HIPCC) and not os.path.exists(HIPCC), reason="hipcc not found")
def test_block_order_of_every_lane_count(tmp_path):
    src, exe = str(tmp_path / "order.hip"), str(tmp_path / "order")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.run([HIPCC, "-O2", "-std=c++17", "--offload-arch=gfx950", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "miniisosurface_amd", "csrc"), "-o", exe, src], check=True,
                   capture_output=True, timeout=300)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout
    plans, raised, tiled = map(int, out.stdout.split())
    assert plans > 5000 and raised > 1000 and tiled > 10 ** 6, out.stdout

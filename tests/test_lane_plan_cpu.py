"""CPU: how many lanes a grid row takes (plan_lanes, BatchLanes, miniisosurface_amd/csrc/fe_rows.h). A batch
of many jobs fills the chip whatever the size of one job, so its rows keep the fewest lanes also where a
job has less than one wavefront of them; a batch of few small jobs takes more, as one volume of all its rows
would. And which rows pass 1 leaves in the caches (keep_from_row): the last 128 MB where pass 4 takes the rows
from the end, else those of a volume that is kept whole, or none. The headers are compiled for the host with
hipcc."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

PROGRAM = r"""
#include "fe_rows.h"
#include <cstdio>
#include <cstdlib>
using namespace miso;
int main(int argc, char** argv)
{
    if (argc == 4) {
        Geom g{};
        g.nx = atoll(argv[1]);
        g.ny = atoll(argv[2]);
        g.nz = atoll(argv[3]);
        const long long R = g.ny * g.nz, end = keep_from_row(g, true), whole = keep_from_row(g, false);
        printf("%lld %lld\n", R - end, R - whole);
        return 0;
    }
    const int64_t n = atoll(argv[1]), ny = atoll(argv[2]), nz = atoll(argv[3]), W = atoll(argv[4]);
    BatchLanes all;
    for (int64_t j = 0; j < n; ++j) all.add(ny, nz, W);
    printf("%d %d %d\n", fewest_lanes(W), all.job(W), plan_lanes(ny, n * nz, W));
    return 0;
}
"""


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    if not shutil.which(HIPCC) and not os.path.exists(HIPCC):
        pytest.skip("hipcc not found")
    tmp = tmp_path_factory.mktemp("lanes")
    src, exe = str(tmp / "lanes.hip"), str(tmp / "lanes")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-arch=gfx950", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "miniisosurface_amd", "csrc"), "-o", exe, src], check=True,
                   capture_output=True, timeout=300)

    def plan(*args):
        out = subprocess.run([exe, *map(str, args)], check=True, capture_output=True, text=True, timeout=60)
        return tuple(int(x) for x in out.stdout.split())
    return plan


# jobs, rows per plane and planes of a job, mask words per row; lg of the lanes
@pytest.mark.parametrize("n,ny,nz,W,lg", [
    (20000, 7, 7, 1, 0),        # 49 rows a job: less than a wavefront each, 15312 of them in all
    (20000, 3, 3, 1, 0),
    (4000, 5, 9, 1, 0),
    (4096, 8, 8, 1, 0),         # one wavefront each
    (1900, 3, 5, 3, 3),         # 15 rows of 4 lanes: 1781 wavefronts, so twice the lanes and no more
    (300, 20, 20, 1, 1),
    (3, 30, 30, 1, 6),
    (1, 2, 2, 1, 6),
    (1, 2000, 2000, 64, 6),
])
def test_batch_lanes(planner, n, ny, nz, W, lg):
    fewest, job, one = planner(n, ny, nz, W)
    assert job == one           # as one volume with the rows of all jobs
    assert job == lg and lg >= fewest


# nx, ny, nz; rows kept where pass 4 starts at the end, and where it does not (all rows or more: the whole volume)
@pytest.mark.parametrize("nx,ny,nz,end,whole", [
    (1024, 1024, 1024, 32768, 0),
    (4097, 64, 64, 8191, 8191),          # 67 MB
    (65536, 128, 16, 512, 0),
    (1 << 25, 2, 2, 1, 0),
    (1 << 23, 2, 2, 4, 4),               # 128 MB
])
def test_kept_rows(planner, nx, ny, nz, end, whole):
    assert planner(nx, ny, nz) == (end, whole)

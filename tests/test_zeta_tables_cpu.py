"""Which tables of the one-launch zeta solve, and of the two-kernel
iteration's halos, the host lays out (host_zeta_tables): those that the
solver reads under the model's settings, and no others."""
import os
import shutil
import subprocess

import pytest

import shyhip

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "shyfemcm-ismar_amd", "csrc")

# rows of a grid of nx by ny nodes with both diagonals of one direction, in
# blocks of brows rows: workgroup size, rows of the halo tables, whether there
# are factor columns
DRIVER = r"""
#include "shyhip_internal.h"
#include <cstdio>
#include <cstdlib>
using namespace shy;
int main(int, char **v) {
    const int nx = atoi(v[1]), ny = atoi(v[2]), brows = atoi(v[3]), esize = atoi(v[4]), exact = atoi(v[5]);
    std::vector<int> ptr{0}, cols;
    for (int y = 0; y < ny; y++)
        for (int x = 0; x < nx; x++) {
            for (int dy = -1; dy <= 1; dy++)
                for (int dx = -1; dx <= 1; dx++)
                    if (dx * dy <= 0 && x + dx >= 0 && x + dx < nx && y + dy >= 0 && y + dy < ny)
                        cols.push_back((y + dy) * nx + x + dx);
            ptr.push_back((int)cols.size());
        }
    BlockSchedule bs;
    host_block_schedule(nx * ny, ptr, cols, brows, bs);
    ZetaTables zt;
    host_zeta_tables(nx * ny, ptr, cols, bs, esize, exact, zt);
    std::printf("%d %d %d %d\n", zt.threads, zt.hmax, (int)!zt.fcol.empty(), (int)!zt.lcol.empty());
    return 0;
}
"""


@pytest.fixture(scope="module")
def tables(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("needs hipcc")
    if not os.path.exists(shyhip.LIBPATH):
        subprocess.run(["make", "-C", os.path.join(ROOT, "shyfemcm-ismar_amd")], check=True)
    d = tmp_path_factory.mktemp("zt")
    src, exe = d / "zt.cpp", str(d / "zt")
    src.write_text(DRIVER)
    obj = str(d / "zt.o")
    subprocess.run([hipcc, "-std=c++17", "-O1", "-w", "-x", "hip", "--offload-host-only", "-I", CSRC, "-c", str(src),
                    "-o", obj], check=True)
    subprocess.run([hipcc, obj, shyhip.LIBPATH, f"-Wl,-rpath,{os.path.dirname(shyhip.LIBPATH)}", "-o", exe], check=True)

    def run(nx, ny, brows, esize, exact):
        r = subprocess.run([exe, *map(str, (nx, ny, brows, esize, int(exact)))], capture_output=True, text=True,
                           check=True, timeout=60)
        return tuple(map(int, r.stdout.split()))
    return run


@pytest.mark.parametrize("nx, ny, brows, esize, exact, threads, factors", [
    (60, 50, 256, 8, False, 256, False),        # swept, one launch
    (60, 50, 256, 4, False, 256, False),
    (250, 160, 256, 8, False, 512, False),
    (200, 600, 256, 8, False, 0, True),         # too many groups: the two-kernel iteration's halos
    (200, 600, 256, 4, False, 0, True),
    (60, 50, 300, 8, False, 0, None),           # sweeps of more than 256 rows: nothing reads tables
    (60, 50, 512, 8, False, 0, None),
    (60, 50, 700, 4, False, 0, None),
    (60, 50, 256, 8, True, 512, False),         # exact in FP64: dense rows, or substitution
    (250, 160, 256, 8, True, 512, False),
    (60, 50, 300, 8, True, 512, False),
    (200, 600, 256, 8, True, 0, None),          # exact on two kernels: blocks are staged
    (60, 50, 256, 4, True, 0, None),            # exact in FP32
    (200, 600, 256, 4, True, 0, None),
])
def test_tables_that_are_read(tables, nx, ny, brows, esize, exact, threads, factors):
    t, hmax, fcol, lcol = tables(nx, ny, brows, esize, exact)
    assert t == threads
    if factors is None:
        assert (hmax, fcol, lcol) == (0, 0, 0)
    else:
        assert lcol and bool(fcol) == factors

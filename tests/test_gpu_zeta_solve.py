"""The zeta solve at the sizes where the one-launch solve changes shape: one
block of up to 1024 rows, workgroups of 256 and 512 work-items with one or
several diagonal blocks each, last workgroups that are partly empty, halos
of one and two entries per work-item, exact and swept triangular solves, and
basins it does not take (halo or block count too large), which the two-kernel
iteration solves.  The assembled system goes in through the system_* entry
points; the answer is a direct solve of the same system in 64 bits."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from shyhip import mesh

from test_gpu_system_plugin import _element_systems

pytestmark = pytest.mark.gpu

# basin, block rows, triangular sweeps (0: exact)
CASES = {
    "one_block_1024": (lambda: mesh.tidal_basin(nx=32, ny=32), 0, 0),
    "one_block_small": (lambda: mesh.tidal_basin(nx=5, ny=4), 0, 0),
    "one_block_sweeps": (lambda: mesh.tidal_basin(nx=14, ny=13), 256, 3),
    "exact_256": (lambda: mesh.tidal_basin(nx=41, ny=30), 0, 0),
    "exact_blocks_of_60": (lambda: mesh.tidal_basin(nx=41, ny=30), 60, 0),
    "exact_no_dense_rows": (lambda: mesh.lagoon(15000, seed=6, nlv=1, tile=32), 0, 0),
    "exact_wide_halo": (lambda: mesh.tidal_basin(nx=230, ny=70), 0, 0),
    "exact_blocks_of_300": (lambda: mesh.tidal_basin(nx=41, ny=31), 300, 0),
    "exact_blocks_of_700": (lambda: mesh.tidal_basin(nx=41, ny=40), 700, 0),
    "sweeps_two_blocks_a_group": (lambda: mesh.lagoon(2000, seed=5, lx=6000.0, ly=3000.0, nlv=1, tile=16), 100, 3),
    "one_sweep": (lambda: mesh.lagoon(2000, seed=5, lx=6000.0, ly=3000.0, nlv=1, tile=16), 256, 1),
    "two_halo_entries": (lambda: mesh.tidal_basin(nx=200, ny=9), 256, 3),
    "halo_too_large": (lambda: mesh.tidal_basin(nx=400, ny=9), 256, 3),
    "groups_of_256": (lambda: mesh.lagoon(32000, seed=6, nlv=1, tile=32), 256, 3),
    "groups_of_512": (lambda: mesh.lagoon(33500, seed=6, nlv=1, tile=32), 256, 4),
    "groups_of_512_exact": (lambda: mesh.lagoon(33500, seed=6, nlv=1, tile=32), 256, 0),
    "too_many_groups": (lambda: mesh.lagoon(140000, seed=7, nlv=1, tile=32), 256, 3),
}


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("case", list(CASES))
def test_zeta_solve_shapes(gpu, case, prec):
    make, brows, sweeps = CASES[case]
    b = make()
    m = gpu.Model(b, prec, params=dict(dt=300.0, ireib=5, block_rows=brows, tri_sweeps=sweeps, rtol=1e-11, atol=0.0,
                                       refine_rtol=1e-12))
    lib, h = m.lib, m.h
    hia, hik = _element_systems(b, 3)
    kn = np.ascontiguousarray(b.nen3v + 1, np.int32)
    hia = np.ascontiguousarray(hia.transpose(0, 2, 1))          # hia(i,j), column-major
    assert lib.shyhip_system_init(h) == 0
    for ie in range(b.nel):
        assert lib.shyhip_system_assemble(h, ie + 1, C.c_void_p(kn.ctypes.data + 12 * ie),
                                          C.c_void_p(hia.ctypes.data + 36 * ie),
                                          C.c_void_p(hik.ctypes.data + 12 * ie)) == 0
    rows = np.repeat(b.nen3v, 3, axis=1).reshape(-1)
    cols = np.tile(b.nen3v, (1, 3)).reshape(-1)
    A = sp.coo_matrix((hia.transpose(0, 2, 1).astype(np.float64).reshape(-1), (rows, cols)),
                      shape=(b.nkn, b.nkn)).tocsc()
    rhs = np.zeros(b.nkn)
    np.add.at(rhs, b.nen3v.reshape(-1), hik.astype(np.float64).reshape(-1))
    ref = spla.spsolve(A, rhs)
    z = np.zeros(b.nkn, np.float32)
    zp = z.ctypes.data_as(C.c_void_p)
    for rep in range(2):                                        # exact, then warm-started block factors
        z0 = np.full(b.nkn, 0.01 * rep, np.float32)
        assert lib.shyhip_system_solve(h, b.nkn, z0.ctypes.data_as(C.c_void_p)) == 0, lib.shyhip_last_error(h)
        assert lib.shyhip_system_get(h, b.nkn, zp) == 0
        err = np.abs(z - ref).max() / np.abs(ref).max()
        print(case, prec, "rel err", err)
        # 32-bit result (6e-8) and a residual of 1e-11 times a condition of
        # at most a few thousand
        assert err < 1e-6
    assert m.stats()["solver_retries"] == 0
    m.close()

"""The transport's element phase and the momentum columns over element orders.

The element phase reads the tracers from LDS where the elements of a
workgroup share their node-layers, and from memory where a workgroup's list
of node-layers would be too long: elements numbered at random reach that.
Both against the oracle on the same basin, one and two tracers per launch,
element-layer counts that leave the last workgroup part empty.  Bars as in
the parity tests: FP64, tracers 1e-6 of the field scale, levels 1e-6 m."""
import dataclasses

import numpy as np
import pytest

from shyhip import mesh

pytestmark = pytest.mark.gpu

SCALE = dict(temp=25.0, salt=38.0)


def _shuffled(b, seed):
    p = np.random.default_rng(seed).permutation(b.nel)
    return dataclasses.replace(b, nen3v=b.nen3v[p], hm3v=b.hm3v[p], hev=b.hev[p], ilhv=b.ilhv[p])


@pytest.mark.parametrize("shuffle", [False, True])
@pytest.mark.parametrize("ntr,nlv,n", [(2, 6, 3000), (1, 20, 1500)])
def test_element_orders_fp64(gpu, shuffle, ntr, nlv, n):
    import pyoracle
    b = mesh.lagoon(n, seed=7, lx=8000.0, ly=4000.0, nlv=nlv, tile=16)
    if shuffle:
        b = _shuffled(b, 3)
    tr = dict(temp=mesh.smooth_tracer(b, 8, 15.0, 25.0), salt=mesh.smooth_tracer(b, 9, 25.0, 38.0))
    tr = {k: tr[k] for k in list(tr)[:ntr]}
    params = dict(dt=60.0, ireib=5, itpre=1, itvd=2, itvdv=1, aapar=0.0, block_rows=0)
    om = pyoracle.OracleModel(b, "f64", params=params, visv=1e-3, difv=1e-4, tracers=tr)
    gm = gpu.Model(b, "fp64", params=params, visv=1e-3, difv=1e-4, tracers=tr)
    for m in (om, gm):
        m.set_wind(*mesh.wind_stress(12.0, 0.7))
        for k in range(6):
            m.step(mesh.tide_level((k + 1) * 60.0, amps=(0.4, 0.1), periods=(mesh.M2_PERIOD, mesh.K1_PERIOD)) - 0.3,
                   istot=2)
    valid = np.arange(b.nlv)[None, :] < b.ilhkv[:, None]
    assert np.array_equal(gm.pull("iwegv"), om.a["iwegv"])
    assert float(np.max(np.abs(gm.pull("znv") - om.a["znv"]))) < 1e-6
    for name in tr:
        d = float(np.max(np.abs(gm.pull(name) - om.tracers[name])[valid]))
        print(name, "shuffled" if shuffle else "in order", "max diff", d)
        assert d < 1e-6 * SCALE[name]
    gm.close()

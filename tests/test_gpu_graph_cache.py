"""A run with more distinct launch sequences than a model keeps graphs of (256):
substep counts 1 .. 90 over the three rotating buffers of the pipelined
transport, so the graphs are dropped while the streams have work, and made
again.  Bit-identical to direct launches."""
import numpy as np
import pytest

from shyhip import mesh

pytestmark = pytest.mark.gpu


def test_more_graphs_than_are_kept(gpu):
    b = mesh.lagoon(1500, seed=21, lx=6000.0, ly=3000.0, nlv=4, tile=16)
    tr = dict(temp=mesh.smooth_tracer(b, 22, 15.0, 25.0), salt=mesh.smooth_tracer(b, 23, 25.0, 38.0))
    out = []
    for graphs in (True, False):
        m = gpu.Model(b, "fp64", params=dict(dt=60.0, ireib=5, itvd=2, itvdv=1, aapar=0.0, block_rows=256, tri_sweeps=3),
                      visv=1e-3, difv=1e-4, tracers=tr)
        m.set_graphs(graphs)
        m.set_deferred_checks(True)
        n = 0
        for istot in range(1, 91):
            for _ in range(3):
                n += 1
                m.step(0.1 * np.sin(n / 20.0), istot=istot)
        m.sync()
        builds = m.graph_stats()[0]
        assert builds > 256 if graphs else builds == 0
        out.append({k: m.pull(k) for k in ("znv", "utlnv", "salt", "temp")})
        m.close()
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k

"""Fields between the host and the device: what is pushed comes back, in both
host types, for every shape a field has (vertex, element and node layers,
interfaces, the two planes of ddxv), at column counts that are no multiple of
the transposing workgroup's; and a member's state copied into a model of the
same basin, whole and inside a union whose members start at odd offsets."""
import numpy as np
import pytest

from shyhip import ensemble, mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nlv", [1, 5, 32])
def test_push_pull(gpu, prec, nlv):
    b = mesh.lagoon(333, seed=3, lx=4000.0, ly=2000.0, nlv=nlv, tile=8)
    m = gpu.Model(b, prec, tracers=dict(salt=np.zeros((b.nkn, b.nlv))))
    rng = np.random.default_rng(1)
    for name in ("zenv", "utlnv", "wlnv", "hdknv", "ddxv", "znv", "unv", 100):
        a = rng.uniform(-1.0, 1.0, m._shape(name)).astype(np.float32)      # exact in both types
        m.push(name, a)
        for dt in (np.float32, np.float64):
            got = m.pull(name, dt)
            assert got.dtype == dt and np.array_equal(got, a.astype(dt)), (name, dt)
        a64 = rng.uniform(-1.0, 1.0, m._shape(name))
        m.push(name, a64)
        want = a64 if prec == "fp64" else a64.astype(np.float32).astype(np.float64)
        assert np.array_equal(m.pull(name), want), name
        assert np.array_equal(m.pull(name, np.float32), a64.astype(np.float32)), name
    m.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_member_state_copies(gpu, prec):
    bs = [mesh.lagoon(n, seed=s, lx=4000.0, ly=2000.0, nlv=4, tile=8) for n, s in ((301, 5), (450, 6))]
    u = ensemble.union_basin(bs)
    names = ("znv", "zenv", "utlnv", "wlnv", "hdenv", "iwegv", "salt")
    rng = np.random.default_rng(2)

    def model(b, members=None):
        m = gpu.Model(b, prec, members=members, tracers=dict(salt=rng.uniform(20.0, 30.0, (b.nkn, b.nlv))))
        m.push("utlnv", rng.uniform(-1.0, 1.0, (b.nel, b.nlv)))
        m.push("wlnv", rng.uniform(-1.0, 1.0, (b.nkn, b.nlv + 1)))
        return m

    union = model(u.basin, (u.node_start, u.elem_start))
    before = {k: union.pull(k) for k in names}
    alone = model(bs[1])
    src = {k: alone.pull(k) for k in names}
    union.copy_member_state(1, alone, 0)
    for k in names:
        got = union.pull(k)
        lo = u.node_start[1] if got.shape[0] == u.basin.nkn else u.elem_start[1]
        assert np.array_equal(got[lo:], src[k]) and np.array_equal(got[:lo], before[k][:lo]), k
    alone.copy_member_state(0, union, 1)
    for k in names:
        assert np.array_equal(alone.pull(k), src[k]), k
    union.close()
    alone.close()

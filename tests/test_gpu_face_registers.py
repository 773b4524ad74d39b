"""GPU checks of the per-face registers (fluxes and CT weights), which a mesh keeps packed
over the computed faces only: what a caller sets comes back whole, the computed faces hold
the oracle's values in the array extents the caller sees, and the rest stays as set."""
import ctypes

import numpy as np
import pytest

from athena_amd.gpu import Ensemble, GpuMesh
from athena_amd.mesh import MeshDesc
from athena_amd.pgen.blast import Blast
from athena_amd.pgen.sr import ShearLayer
from oracle_bind import OracleMesh
from test_gpu_smr import compare, load_both, smr_wave

pytestmark = pytest.mark.gpu
REGS = ("flux1", "flux2", "flux3", "wght1", "wght2", "wght3")


def _mesh(nx, bnx, ng):
    m = MeshDesc(nx=nx, bnx=bnx, xmin=(-0.5,) * 3, xmax=(0.5,) * 3, gamma=5.0 / 3.0, cfl=0.3,
                 xorder=3 if ng > 2 else 2, ng=ng, rsolver="hlld")
    return m, Blast(m)


def _shape(m, reg):
    d = int(reg[-1]) - 1
    ext = [m.bnx[q] + 2 * m.ng + (q == d) for q in (2, 1, 0)]
    return ([5] if reg.startswith("flux") else []) + ext


@pytest.mark.parametrize("nx,bnx,ng", [((4, 4, 4), (2, 2, 2), 2), ((10, 6, 7), (5, 3, 7), 2),
                                       ((17, 16, 5), (17, 8, 5), 3), ((15, 8, 5), (15, 4, 5), 4)])
def test_face_registers(nx, bnx, ng):
    m, ic = _mesh(nx, bnx, ng)
    print("case face registers", nx, bnx, ng, flush=True)
    d = GpuMesh(m)
    rng = np.random.default_rng(7)
    put = {}
    for reg in REGS:
        for g in (0, m.nblocks - 1):
            put[g, reg] = rng.standard_normal(_shape(m, reg))
            d.set(g, reg, put[g, reg])
    for (g, reg), a in put.items():
        assert np.array_equal(d.get(g, reg).reshape(a.shape), a), (g, reg)

    blocks = [ic.block(g) for g in range(m.nblocks)]
    o = OracleMesh(m)
    o.load(blocks)
    o.initialize(1e300)
    o.run(2, 1e300)
    d.load(blocks)
    d.initialize(1e300)
    d.run(2)
    lo, n = ng, m.bnx
    for (g, reg), a in put.items():
        x = int(reg[-1]) - 1
        got = d.get(g, reg).reshape(a.shape)
        want = o.get(g, reg).reshape(a.shape)
        # the faces of active cells; then everything the flux kernel does not compute
        act = tuple(slice(lo, lo + n[q] + (q == x)) for q in (2, 1, 0))
        assert np.array_equal(got[(...,) + act], want[(...,) + act]), (g, reg)
        comp = tuple(slice(lo - (q != x), lo + n[q] + 1) for q in (2, 1, 0))
        rest = np.ones(a.shape, bool)
        rest[(...,) + comp] = False
        assert np.array_equal(got[rest], a[rest]), (g, reg)


class _Mallinfo2(ctypes.Structure):
    _fields_ = [(n, ctypes.c_size_t) for n in ("arena", "ordblks", "smblks", "hblks", "hblkhd",
                                               "usmblks", "fsmblks", "uordblks", "fordblks",
                                               "keepcost")]


def _host_bytes():
    """Bytes the process holds from malloc."""
    f = ctypes.CDLL(None).mallinfo2
    f.restype = _Mallinfo2
    s = f()
    return s.uordblks + s.hblkhd


def test_host_memory_of_set_registers():
    """Setting the flux registers keeps on the host what lies outside the packed arrays, and
    nothing where that is zero."""
    m, _ = _mesh((96, 96, 96), (48, 48, 48), 2)
    print("case host memory of face registers", flush=True)
    d = GpuMesh(m)
    n = m.bnx
    regs = ("flux1", "flux2", "flux3")
    full, zeroed, outside = {}, {}, 0
    rng = np.random.default_rng(3)
    for reg in regs:
        x = int(reg[-1]) - 1
        full[reg] = rng.standard_normal(_shape(m, reg))
        zeroed[reg] = np.zeros_like(full[reg])
        comp = tuple(slice(m.ng - (q != x), m.ng + n[q] + 1) for q in (2, 1, 0))
        zeroed[reg][(...,) + comp] = full[reg][(...,) + comp]
        outside += full[reg].nbytes - full[reg][(...,) + comp].nbytes
    for arrays, keep in ((zeroed, 0), (full, outside * m.nblocks), (zeroed, 0)):
        for reg in regs:       # staging buffers and the like
            d.set(0, reg, zeroed[reg])
            d.get(0, reg)
        before = _host_bytes()
        for g in range(m.nblocks):
            for reg in regs:
                d.set(g, reg, arrays[reg])
        grown = _host_bytes() - before
        assert grown < keep + 2**20, (grown, keep)
        for g in (0, m.nblocks - 1):
            for reg in regs:
                assert np.array_equal(d.get(g, reg).ravel(), arrays[reg].ravel()), (g, reg)
    minus = np.full(_shape(m, "wght1"), -0.0)
    d.set(1, "wght1", minus)
    assert np.signbit(d.get(1, "wght1")).all()


STREAMED = 120 * 2**20   # bytes of per-face outputs above which a launch stores them streaming


def face_bytes(m):
    return 24 * 8 * m.nblocks * np.prod([n + 2 for n in m.bnx])


@pytest.mark.parametrize("bnx,nx,sr,rsolver,xorder",
                         [((24, 24, 24), (96, 96, 72), False, "hlld", 2),
                          ((27, 16, 29), (81, 96, 87), False, "hlle", 3),
                          ((25, 24, 23), (100, 72, 92), True, "hlle", 3),
                          ((24, 24, 24), (96, 96, 72), True, "hlld", 2)])
def test_streamed_faces(bnx, nx, sr, rsolver, xorder):
    """Enough per-face outputs that the flux launches store them past the L2 caches.  A mesh by
    itself and, with a smaller one, in an ensemble."""
    ng = xorder if xorder == 2 else 4
    desc = dict(xmin=(-0.5,) * 3, xmax=(0.5,) * 3, gamma=4.0 / 3.0 if sr else 5.0 / 3.0, cfl=0.3,
                xorder=xorder, ng=ng, rsolver=rsolver, relativistic=sr)
    ic = ShearLayer if sr else Blast
    m = MeshDesc(nx=nx, bnx=bnx, **desc)
    print("case streamed faces", nx, bnx, sr, rsolver, flush=True)
    assert face_bytes(m) > STREAMED
    problem = ic(m)
    blocks = [problem.block(g) for g in range(m.nblocks)]
    o = OracleMesh(m)
    o.load(blocks)
    o.initialize(1e300)
    o.run(2, 1e300)
    dev = [GpuMesh(m), GpuMesh(m)]
    for d in dev:
        d.load(blocks)
        d.initialize(1e300)
    dev[0].run(2)
    small = MeshDesc(nx=bnx, bnx=bnx, **desc)
    s = GpuMesh(small)
    s.load([ic(small).block(0)])
    s.initialize(1e300)
    e = Ensemble([dev[1], s])
    e.run(2)
    for d in dev:
        for g in range(m.nblocks):
            for key in ("u", "b1", "b2", "b3"):
                assert np.array_equal(d.get(g, key).ravel(), o.get(g, key).ravel()), (g, key)


def test_streamed_faces_of_a_refined_mesh():
    """The flux and EMF corrections read and write what the streamed launch stored."""
    m, lw = smr_wave(80, 0, xorder=2, rsolver="hlld", ng=2)
    print("case streamed faces, refined", m.nblocks, flush=True)
    assert face_bytes(m) > STREAMED
    dev, ora = load_both(m, lw)
    dev.initialize(1.0)
    ora.initialize(1.0)
    dev.run(2, 1.0)
    ora.run(2, 1.0)
    compare(dev, ora, m, "after 2 cycles")

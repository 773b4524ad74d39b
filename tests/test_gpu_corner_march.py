"""GPU checks of the corner EMF kernel's z-march (tile options 6, the default, and 7) where
its tiles and segments have edges: rows of edges that fill a work-group, that just fit and
that are split into equal tiles; the smallest MeshBlocks; MeshBlocks whose planes do not
divide into whole segments; and launches of every kind of height: single planes, the two
planes at least of a large launch, and the tallest segments, of tiles of one and of several
rows, with the height each case reaches checked against the launch's rule.  The march evaluates the linear mapping's expressions on the same
values, so whole runs are bit for bit those of one thread per edge (tile 0), which the
parity tests tie to the CPU oracle; the widest case is compared with the oracle directly."""
import numpy as np
import pytest

from athena_amd.gpu import GpuMesh
from athena_amd.mesh import MeshDesc
from athena_amd.pgen.blast import Blast
from athena_amd.pgen.linear_wave import LinearWave, linear_wave_mesh
from athena_amd.pgen.sr import ShearLayer
from harness import compare
from oracle_bind import OracleMesh

pytestmark = pytest.mark.gpu
KEYS = ("u", "w", "bcc", "b1", "b2", "b3")


def _box(nx, bnx, sr=False):
    m = MeshDesc(nx=nx, bnx=bnx, xmin=(-0.5,) * 3, xmax=(0.5,) * 3,
                 gamma=4.0 / 3.0 if sr else 5.0 / 3.0, cfl=0.3, xorder=2, ng=2,
                 rsolver="hlle" if sr else "hlld", relativistic=sr)
    return m, (ShearLayer if sr else Blast)(m)


def _lw(bnx):
    m = linear_wave_mesh(24, bnx=bnx, rsolver="hlld", xorder=2, ng=2)
    return m, LinearWave(m, wave_flag=0, amp=1e-6)


# name: mesh, planes per segment under tile options 6 and 7
CASES = {
    "2x2x2": (lambda: _lw((2, 2, 2)), 2, 2),
    "3x4x6": (lambda: _lw((3, 4, 6)), 1, 1),
    "row_126": (lambda: _box((126, 6, 5), (126, 6, 5)), 1, 1),   # 127 edges: one tile, 128 cells
    "row_127": (lambda: _box((127, 6, 5), (127, 6, 5)), 1, 1),   # 128 edges: two tiles
    "row_260_sr": (lambda: _box((260, 4, 7), (260, 4, 7), sr=True), 1, 1),   # three tiles
    "rows_of_5": (lambda: _box((70, 140, 66), (35, 35, 33)), 3, 4),
    "rows_of_1": (lambda: _box((192, 96, 64), (96, 48, 32)), 11, 17),   # 33 planes in 3 and 2
    "rows_of_7_sr": (lambda: _box((80, 60, 60), (20, 20, 20), sr=True), 2, 3),
}


def heights(m):
    """Planes per segment under tile options 6 and 7 (corner_tile and march_geom)."""
    n = [b + 1 for b in m.bnx]
    ti = n[0] if n[0] < 256 else 255
    if ti > 127:
        ti = -(-n[0] // -(-n[0] // 127))
    nti, tj = -(-n[0] // ti), 256 // (ti + 1) - 1
    ntj = -(-n[1] // tj)
    tj = -(-n[1] // ntj)
    tall = max(2, (32 // tj + 1) // 2)
    short = int(nti * ntj * n[2] * m.nblocks / 768.0 + 0.5)
    out = []
    for cap in (tall, tall + tall // 2):
        h = max(1, min(cap, short))
        out.append(-(-n[2] // -(-n[2] // h)))
    return tuple(out)


def run(m, ic, tiles):
    d = GpuMesh(m)
    d.load([ic.block(g) for g in range(m.nblocks)])
    d.set_tiles(tiles)
    d.initialize()
    d.run(3)
    return d


@pytest.mark.parametrize("name", list(CASES))
def test_corner_march_runs_bit_for_bit_as_one_thread_per_edge(name):
    make, *want = CASES[name]
    m, ic = make()
    print("case corner march", name, flush=True)
    assert heights(m) == tuple(want)
    ref = run(m, ic, [0, 0, 0, 0])
    for tile in (6, 7):
        d = run(m, ic, [0, tile, 0, 0])
        assert d.state() == ref.state(), tile
        for g in range(m.nblocks):
            for key in KEYS:
                assert np.array_equal(d.get(g, key), ref.get(g, key)), (tile, g, key)


def test_corner_march_against_the_oracle():
    m, ic = _box((127, 6, 5), (127, 6, 5))
    print("case corner march vs oracle, 127x6x5", flush=True)
    o = OracleMesh(m)
    o.load([ic.block(g) for g in range(m.nblocks)])
    o.initialize(1e300)
    o.run(3, 1e300)
    d = run(m, ic, [0, 6, 0, 0])
    res = compare(m, lambda g, k: d.get(g, k), lambda g, k: o.get(g, k))
    assert all(eq for _, eq in res.values()), res

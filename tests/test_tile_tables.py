"""The once-per-edge fused kernel's tables (CPU): every cell, node, halo edge
and listed edge that a workgroup reads, replayed against the mesh, and the
kernel's phases (anuga_core_amd/csrc/de_kernels.hip, de_xflux_e) over the LDS
they share. Calls only host-side entry points."""

import ctypes as C
import os
import resource
import subprocess
import sys

import numpy as np
import pytest

from anuga_core_amd import _native
from anuga_core_amd.mesh import Mesh, graded_square, rectangular, rectangular_cross
from tests.test_tiles import BLOCK, tile_layout

# DE_XCELLS_MAX, DE_XHALO_MAX, DE_XNODES_MAX
CELLS, HALO, NODES = min(BLOCK, 1022 - BLOCK), min(BLOCK - 64, 256), 384


def _tables(nb, vertices=None, crowded=False, refused=None, **fields):
    """The tables of packed neighbours nb [N][3], or None beyond the limits;
    crowded: with the tiles beyond them marked instead. refused: the arrays,
    after a call with these fields that returns this error."""
    N = len(nb)
    nt = (N + BLOCK - 1) // BLOCK
    cap = 3 * N + nt * (CELLS + NODES + HALO)
    u = lambda n: np.zeros(n, np.uint32)  # noqa: E731
    i = lambda n: np.zeros(n, np.int32)   # noqa: E731
    a = dict(sizes=np.zeros(4, np.int64), stencil=u(N), across=u(N), nodes=u(N), cstart=i(nt),
             hstart=i(nt), estart=i(nt), esplit=i(nt), nstart=i(nt), cell=i(cap),
             hstencil=u(cap), hcell=u(cap), hnodes=u(cap), edge=u(cap), node=np.zeros(2 * cap))
    if crowded:
        a["crowded"] = np.zeros(nt, np.uint8)
    types = dict(_native.TileTables._fields_)
    given = {k: v.ctypes.data_as(types[k]) for k, v in a.items()}
    t = _native.TileTables(**{**dict(capacity=cap), **given, **fields})
    vx = None if vertices is None else np.ascontiguousarray(vertices, np.float64)
    nb = np.ascontiguousarray(nb, np.int32)
    rc = _native.lib().anuga_tile_tables(
        N, nb.ctypes.data_as(C.POINTER(C.c_int32)),
        None if vx is None else vx.ctypes.data_as(C.POINTER(C.c_double)), C.byref(t))
    if refused is not None:
        assert rc == refused
        return a
    if rc:
        return None
    for name, end, starts in (("cell", 0, "cstart"), ("hstencil", 1, "hstart"),
                              ("edge", 2, "estart"), ("node", 3, "nstart")):
        a[starts] = np.append(a[starts], a["sizes"][end])
    a["node"] = a["node"].reshape(-1, 2)
    return a


def _field(w, i):
    return (w.astype(np.int64) >> (10 * i)) & 1023


def _replay(nb, a, vertices):
    N = len(nb)
    nb = nb.astype(np.int64)
    for b in range((N + BLOCK - 1) // BLOCK):
        k0, k1 = b * BLOCK, min(N, (b + 1) * BLOCK)
        if "crowded" in a and a["crowded"][b]:
            # no entries, so that the kernel's first loads stay in bounds
            assert all(a[s][b] == a[s][b + 1] for s in ("cstart", "hstart", "estart"))
            assert a["esplit"][b] == a["estart"][b]
            assert np.all(a["stencil"][k0:k1] == 0x3fffffff) and not np.any(a["across"][k0:k1])
            continue
        cells = np.full(2 * BLOCK, -1)
        cells[:k1 - k0] = np.arange(k0, k1)
        more = a["cell"][a["cstart"][b]:a["cstart"][b + 1]]
        assert len(more) <= CELLS and len(np.unique(more)) == len(more)
        assert not np.any((more >= k0) & (more < k1))
        cells[BLOCK:BLOCK + len(more)] = more
        es, e0, e1 = a["esplit"][b], a["estart"][b], a["estart"][b + 1]
        h = slice(a["hstart"][b], a["hstart"][b + 1])
        nhe = h.stop - h.start
        assert nhe == e1 - es and nhe <= HALO
        hcell = a["hcell"][h].astype(np.int64)
        halo, hj = cells[hcell & 1023], hcell >> 10
        assert np.all((hcell & 1023) >= BLOCK) and np.all(halo >= 0) and np.all(hj < 3)
        k = np.arange(k0, k1)
        for i in range(3):
            # stencils: the neighbour's cell, 1023 on boundary edges
            for st, tri in ((a["stencil"][k0:k1], k), (a["hstencil"][h], halo)):
                f, v = _field(st, i), nb[tri, i]
                assert np.array_equal(f == 1023, v < 0)
                inner = v >= 0
                assert np.array_equal(cells[f[inner]], v[inner] >> 2)
            # across: the neighbour's edge, and the halo edge that faces it
            f, v = _field(a["stencil"][k0:k1], i), nb[k, i]
            ac = a["across"][k0:k1].astype(np.int64)
            inner = v >= 0
            assert np.array_equal(((ac >> (2 * i)) & 3)[inner], v[inner] & 3)
            out = inner & (f >= BLOCK)
            he = (ac >> (6 + 8 * i)) & 255
            assert np.all(he[out] < nhe)
            assert np.array_equal(halo[he[out]], v[out] >> 2)
            assert np.array_equal(hj[he[out]], v[out] & 3)
            # one listed entry per halo edge, in the halo edges' order
            en = a["edge"][es + he[out]].astype(np.int64)
            assert np.array_equal(en & 1023, k[out] - k0)
            assert np.all((en >> 10) & 3 == i) and np.all((en >> 12) & 1 == 1)
        # in-tile edges: each once, from its lower-numbered triangle
        en = a["edge"][e0:es].astype(np.int64)
        t, i, n, j = en & 1023, (en >> 10) & 3, (en >> 13) & 1023, (en >> 23) & 3
        assert np.all((en >> 12) & 1 == 0) and np.all(t < n)
        assert np.array_equal(nb[k0 + t, i], ((k0 + n) << 2) | j)
        v = nb[k0:k1]
        inside = (v >= 0) & ((v >> 2) >= k0) & ((v >> 2) < k1)
        assert len(np.unique(t * 4 + i)) == len(en) == inside.sum() // 2
        if vertices is None:
            continue
        nd = a["node"][a["nstart"][b]:a["nstart"][b + 1]]
        assert len(nd) <= NODES and len(np.unique(nd, axis=0)) == len(nd)
        for c in range(3):
            assert np.array_equal(nd[_field(a["nodes"][k0:k1], c)], vertices[k0:k1, c])
            assert np.array_equal(nd[_field(a["hnodes"][h], c)], vertices[halo, c])


def _ordered(mesh):
    nb = tile_layout(mesh)[0]
    cen = np.ascontiguousarray(mesh.centroid_coordinates)
    order = np.empty(len(nb), np.int64)
    nbr = np.ascontiguousarray(mesh.neighbours, np.int64)
    p64 = lambda x: x.ctypes.data_as(C.POINTER(C.c_int64))  # noqa: E731
    assert _native.lib().anuga_tile_order(len(nb), cen.ctypes.data_as(C.POINTER(C.c_double)),
                                          p64(nbr), p64(order)) == 0
    return nb, mesh.vertex_coordinates.reshape(-1, 3, 2)[order]


@pytest.mark.parametrize("make", [
    lambda: rectangular_cross(1, 1), lambda: rectangular_cross(8, 8),
    lambda: rectangular_cross(37, 53, 1000.0, 700.0), lambda: rectangular_cross(150, 150),
    lambda: rectangular(1000, 1, 1000.0, 1.0), lambda: rectangular(128, 1), lambda: rectangular(3, 43),
    lambda: graded_square(300.0, 9.0, 40.0, (100.0, 100.0, 200.0, 200.0), seed=3)])
def test_tables_name_every_neighbour_edge_and_vertex(make):
    nb, vertices = _ordered(Mesh(*make()))
    a = _tables(nb, vertices)
    if a is None and BLOCK > 256:
        pytest.skip("a tile of a strip has more than two nodes per three triangles")
    assert a is not None
    _replay(nb, a, vertices)
    plain = _tables(nb)
    for name in ("stencil", "across", "cell", "hstencil", "hcell", "edge"):
        assert np.array_equal(plain[name][:len(a[name])], a[name][:len(plain[name])])


def test_tables_refuse_scattered_tiles():
    """Triangles in a random order: more cells than a tile's LDS holds."""
    mesh = Mesh(*rectangular_cross(30, 30))
    N = mesh.number_of_triangles
    order = np.random.default_rng(0).permutation(N)
    place = np.empty(N, np.int64)
    place[order] = np.arange(N)
    n, e = mesh.neighbours[order], mesh.neighbour_edges[order]
    nb = np.where(n >= 0, (place[np.maximum(n, 0)] << 2) | e, -1)
    assert _tables(nb) is None


def _limits(nb, vertices, b):
    """Cells, halo edges and nodes of tile b."""
    k0, k1 = b * BLOCK, min(len(nb), (b + 1) * BLOCK)
    n = np.where(nb >= 0, nb >> 2, -1).astype(np.int64)
    out = lambda v: v[(v >= 0) & ((v < k0) | (v >= k1))]  # noqa: E731
    edges = out(n[k0:k1].ravel())
    halo = np.unique(edges)
    cells = np.unique(np.concatenate([halo, out(n[halo].ravel())]))
    tri = np.concatenate([np.arange(k0, k1), halo])
    return len(cells), len(edges), len(np.unique(vertices[tri].reshape(-1, 2), axis=0))


@pytest.mark.parametrize("tiles", [(0,), (3, 9, 17), tuple(range(8, 25))])
def test_only_crowded_tiles_go_without_tables(tiles):
    """A few tiles whose triangles are scattered over the mesh: these alone
    are marked; every other tile's tables are whole."""
    if BLOCK != 256:
        pytest.skip("sized for 256-triangle tiles")
    nb, vertices = _ordered(Mesh(*rectangular_cross(53, 41, 53.0, 41.0)))
    N = len(nb)
    among = np.concatenate([np.arange(b * BLOCK, (b + 1) * BLOCK) for b in tiles + (30,)])
    order = np.arange(N)
    order[among] = np.random.default_rng(len(tiles)).permutation(among)
    place = np.empty(N, np.int64)
    place[order] = np.arange(N)
    n = nb[order].astype(np.int64)
    nb = np.where(n >= 0, (place[np.maximum(n, 0) >> 2] << 2) | (n & 3), -1)
    vertices = vertices[order]
    nt = (N + BLOCK - 1) // BLOCK
    sizes = np.array([_limits(nb, vertices, b) for b in range(nt)])
    want = (sizes > (CELLS, HALO, NODES)).any(axis=1)
    assert 2 <= want.sum() < nt
    a = _tables(nb, vertices, crowded=True)
    assert np.array_equal(a["crowded"], want.astype(np.uint8))
    _replay(nb, a, vertices)
    assert _tables(nb, vertices) is None


NO_THREADS = """
import resource, sys
sys.path.insert(0, %r)
from anuga_core_amd.mesh import Mesh, rectangular_cross
from tests.test_tile_tables import _ordered, _replay, _tables
nb, vertices = _ordered(Mesh(*rectangular_cross(60, 60, 60.0, 60.0)))
pages = int(open("/proc/self/statm").read().split()[0])
resource.setrlimit(resource.RLIMIT_AS, (pages * resource.getpagesize() + (1 << 30),) * 2)
import threading
try:
    threading.Thread(target=int).start()
    print("a thread was started")
except RuntimeError:
    pass
_replay(nb, _tables(nb, vertices), vertices)
print("whole")
"""


def test_tables_without_threads():
    """Where no thread can be started the calling one cuts every tile: stacks
    of 4 GiB do not fit the address space that is left."""
    def limit():
        hard = resource.getrlimit(resource.RLIMIT_STACK)[1]
        resource.setrlimit(resource.RLIMIT_STACK, (4 << 30, hard))

    if 0 <= resource.getrlimit(resource.RLIMIT_STACK)[1] < 4 << 30:
        pytest.skip("the stack limit cannot be raised")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", NO_THREADS % root], preexec_fn=limit, text=True,
                       env=dict(os.environ, OMP_NUM_THREADS="1", OPENBLAS_NUM_THREADS="1"),
                       capture_output=True, timeout=120)
    if "a thread was started" in r.stdout:
        pytest.skip("threads start all the same")
    assert r.returncode == 0 and r.stdout == "whole\n", r.stderr[-2000:]


@pytest.mark.parametrize("field,value", [("capacity", -1), ("capacity", 10), ("sizes", None),
                                         ("stencil", None), ("edge", None), ("node", None)])
def test_tables_refuse_a_bad_description(field, value):
    """Negative and small capacities and missing arrays are refused, with
    nothing written behind an array's end."""
    nb, vertices = _ordered(Mesh(*rectangular_cross(30, 30)))
    a = _tables(nb, vertices, refused=-1, **{field: value})
    if field == "capacity":
        assert not any(np.any(v) for v in a.values())


class Lds:
    """The LDS of a workgroup, holding tokens. Between two barriers no address
    that one thread writes may be read or written by another."""

    def __init__(self, size):
        self.size, self.at = size, {}
        self.barrier()

    def barrier(self):
        self.writer, self.readers = {}, {}

    def put(self, thread, a, token):
        assert 0 <= a < self.size
        assert self.writer.setdefault(a, thread) == thread, "two writers of %d" % a
        assert self.readers.get(a, {thread}) == {thread}, "%d is written as it is read" % a
        self.at[a] = token

    def get(self, thread, a):
        assert 0 <= a < self.size
        assert self.writer.get(a, thread) == thread, "%d is read as it is written" % a
        self.readers.setdefault(a, set()).add(thread)
        return self.at[a]


def _phases(nb, a):
    """Every phase of de_xflux_e with tokens in place of values: what each
    thread reads is what the phase needs, from the slots that the tables name.
    Returns the number of edges evaluated."""
    N, nt = len(nb), (len(nb) + BLOCK - 1) // BLOCK
    hecap = max((int(np.diff(a["hstart"]).max()) + 15) // 16 * 16, 16)
    Q, XS, HL, HZ = 3 * BLOCK, 2 * BLOCK, 12 * BLOCK, 12 * BLOCK + 4 * hecap
    a = {k: v.astype(np.int64).tolist() for k, v in a.items() if k not in ("node", "sizes")}
    nb = nb.astype(np.int64).tolist()
    field = lambda w, i: (w >> (10 * i)) & 1023  # noqa: E731
    evaluated = 0
    for b in range(nt):
        if "crowded" in a and a["crowded"][b]:
            continue
        k0, kn = b * BLOCK, min(N - b * BLOCK, BLOCK)
        cells = a["cell"][a["cstart"][b]:a["cstart"][b + 1]]
        h0, nhe = a["hstart"][b], a["hstart"][b + 1] - a["hstart"][b]
        e0, es, e1 = a["estart"][b], a["esplit"][b], a["estart"][b + 1]
        hw = (nhe + 63) // 64
        halo = [(cells[(w & 1023) - BLOCK], w >> 10) for w in a["hcell"][h0:h0 + nhe]]
        lds = Lds(HZ + 2 * BLOCK)
        # 0: the cells; the tile's beds
        for t in range(BLOCK):
            k = k0 + t if t < kn else None
            for q in range(6):
                lds.put(t, q * XS + t, ("cell", k, q))
                if t < len(cells):
                    lds.put(t, q * XS + BLOCK + t, ("cell", cells[t], q))
            lds.put(t, HZ + BLOCK + t, ("bed", k))
        lds.barrier()

        # 1: the stencils of the tile's triangles and of the halo edges'
        def read(t, self, tri, st):
            for place, want in [(self, tri)] + [
                    (self if field(st, i) == 1023 else field(st, i),
                     tri if v < 0 else v >> 2) for i, v in enumerate(nb[tri])]:
                for q in range(6):
                    assert lds.get(t, q * XS + place) == ("cell", want, q)

        for t in range(kn):
            read(t, t, k0 + t, a["stencil"][k0 + t])
            lds.put(t, HZ + t, ("depth", k0 + t))
        for t, (tri, _) in enumerate(halo):
            read(t, a["hcell"][h0 + t] & 1023, tri, a["hstencil"][h0 + t])
        lds.barrier()
        # the edge values take the cells' place
        for t in range(kn):
            for i in range(3):
                for r in range(4):
                    lds.put(t, (3 * r + i) * BLOCK + t, ("value", k0 + t, i, r))
        lds.barrier()

        def edge(thread, e):
            en, he = a["edge"][e], e - es
            t, i, n, j = en & 1023, (en >> 10) & 3, (en >> 13) & 1023, (en >> 23) & 3
            A = i * BLOCK + t
            R, rs = (HL + he, hecap) if he >= 0 else (j * BLOCK + n, Q)
            side = (k0 + t, i)
            other = halo[he] if he >= 0 else (k0 + n, j)
            assert nb[side[0]][i] == (other[0] << 2) | other[1]
            for r in range(4):
                assert lds.get(thread, A + r * Q) == ("value",) + side + (r,)
                assert lds.get(thread, R + r * rs) == ("value",) + other + (r,)
            for m in (t, n) if he < 0 else (t,):
                assert lds.get(thread, HZ + m) == ("depth", k0 + m)
                assert lds.get(thread, HZ + BLOCK + m) == ("bed", k0 + m)
            for r, name in enumerate(("a0", "a1", "a2", "b1")):
                lds.put(thread, A + r * Q, (name,) + side)
            lds.put(thread, R, ("b2",) + side)
            if he < 0:
                lds.put(thread, R + rs, ("c1",) + side)
                lds.put(thread, R + 2 * rs, ("c2",) + side)

        # 2: the halo's edge values; edges inside the tile on the other waves
        done = []
        for t, (tri, j) in enumerate(halo):
            for r in range(4):
                lds.put(t, HL + r * hecap + t, ("value", tri, j, r))
        for t in range(64 * hw, BLOCK):
            e = e0 + t - 64 * hw
            if e < es:
                edge(t, e)
                done.append(e)
        lds.barrier()
        # 3: the edges that are left
        for t in range(BLOCK):
            for e in range(min(es, e0 + BLOCK - 64 * hw) + t, e1, BLOCK):
                edge(t, e)
                done.append(e)
        assert sorted(done) == list(range(e0, e1))
        evaluated += len(done)
        lds.barrier()
        # 4: every triangle's three edges, by the roles that the words give
        for t in range(kn):
            k = k0 + t
            ac = a["across"][k]
            for i in range(3):
                A, f, v = i * BLOCK + t, field(a["stencil"][k], i), nb[k][i]
                if f == 1023:
                    assert v < 0
                    got = [lds.get(t, A + r * Q) for r in range(4)]
                    want = [("value", k, i, r) for r in range(4)]
                elif f > t:
                    far = HL + ((ac >> (6 + 8 * i)) & 255) if f >= BLOCK else \
                        ((ac >> (2 * i)) & 3) * BLOCK + f
                    got = [lds.get(t, A + r * Q) for r in range(4)] + [lds.get(t, far)]
                    want = [(x, k, i) for x in ("a0", "a1", "a2", "b1", "b2")]
                else:
                    far = ((ac >> (2 * i)) & 3) * BLOCK + f
                    got = [lds.get(t, far + r * Q) for r in range(3)] + \
                        [lds.get(t, A + Q), lds.get(t, A + 2 * Q)]
                    want = [(x, v >> 2, v & 3) for x in ("a0", "a1", "a2")] + \
                        [(x, v >> 2, v & 3) for x in ("c1", "c2")]
                assert got == want, (k, i, got, want)
    return evaluated


@pytest.mark.parametrize("make,per_triangle", [
    (lambda: rectangular_cross(40, 40, 1000.0, 700.0), (1.4, 1.8)),
    (lambda: rectangular_cross(37, 53, 1000.0, 700.0), None),
    (lambda: rectangular_cross(1, 1), None), (lambda: rectangular_cross(8, 8), None),
    (lambda: rectangular(128, 1), None),
    (lambda: graded_square(600.0, 40.0, 300.0, (150.0, 150.0, 450.0, 450.0), seed=1), None)])
def test_lds_of_every_phase(make, per_triangle):
    nb, _ = _ordered(Mesh(*make()))
    n = _phases(nb, _tables(nb))
    if per_triangle:   # about 1.6 evaluated edges per triangle instead of 3
        assert per_triangle[0] < n / len(nb) < per_triangle[1]


def test_lds_of_tiles_at_the_limits():
    """Tiles with scattered triangles, up to nearly as many cells as the tables
    take, beside crowded ones that are left out."""
    if BLOCK != 256:
        pytest.skip("sized for 256-triangle tiles")
    nb, _ = _ordered(Mesh(*rectangular_cross(53, 41, 53.0, 41.0)))
    N = len(nb)
    rng = np.random.default_rng(3)
    order = np.arange(N)
    for b in range(0, 30, 2):   # exchange more and more triangles of two tiles
        m = 12 + b
        i, j = (rng.choice(np.arange(t * BLOCK, (t + 1) * BLOCK), m, replace=False)
                for t in (b, b + 1))
        order[i], order[j] = order[j], order[i].copy()
    place = np.empty(N, np.int64)
    place[order] = np.arange(N)
    n = nb[order].astype(np.int64)
    nb = np.where(n >= 0, (place[np.maximum(n, 0) >> 2] << 2) | (n & 3), -1)
    a = _tables(nb, crowded=True)
    assert a["crowded"].any() and np.diff(a["cstart"]).max() > 0.9 * CELLS
    _replay(nb, a, None)
    _phases(nb, a)

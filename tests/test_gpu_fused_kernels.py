"""The fused FP64 kernels that meshes, options and limits choose between give
the same bits: the once-per-edge kernel with its geometry from the vertices,
the same with the stored geometry, and the gather kernel, over every tile or
over the crowded ones only."""

import numpy as np
import pytest
import torch

from anuga_core_amd.boundaries import (Dirichlet_boundary, Reflective_boundary,
                                       Transmissive_boundary)
from anuga_core_amd.domain import Domain
from anuga_core_amd.ensemble import Ensemble
from anuga_core_amd.mesh import Mesh, graded_square, rectangular_cross
from tests.test_tile_tables import _ordered, _tables

pytestmark = pytest.mark.gpu

NAMES = ("stage", "xmomentum", "ymomentum")
KINDS = (lambda d: Reflective_boundary(d), lambda d: Dirichlet_boundary([0.3, 0.2, -0.1]),
         lambda d: Transmissive_boundary(d))


def _inputs(mesh, seed):
    """Hills, partly above the water, and moving water."""
    rng = np.random.default_rng(seed)
    N = mesh.number_of_triangles
    x, y = mesh.centroid_coordinates.T
    z = 0.6 * np.sin(x / 2.3) * np.cos(y / 3.1) - 0.3
    wet = rng.random(N) < 0.9
    return dict(elevation=z, stage=np.where(wet, np.maximum(z, 0.1 * rng.random(N)), z),
                friction=0.03 * rng.random(N), xmomentum=0.2 * wet * rng.standard_normal(N),
                ymomentum=0.2 * wet * rng.standard_normal(N))


def _run(mesh, q, alg, steps, **options):
    d = Domain(mesh=mesh, **options)
    d.set_flow_algorithm(alg)
    d.set_evolve_min_timestep(0.0)
    for n, v in q.items():
        d.set_quantity(n, v, location="centroids")
    d.set_boundary({t: KINDS[i % 3](d) for i, t in enumerate(sorted(d.get_boundary_tags()))})
    for n in steps:
        d.evolve_steps(n)
    return ([d.get_quantity(n).centroid_values for n in NAMES], d.dt_history,
            d.get_boundary_flux_integral())


def _same(a, b):
    assert a[1] == b[1] and a[2] == b[2]
    for x, y in zip(a[0], b[0]):
        assert np.array_equal(x, y)


def _stacked_sheets(n, sheets=25, m=6):
    """A grid of 4 n n triangles and, beside it, a stack of sheets over one
    another: a tile there holds a piece of every sheet, with its surroundings."""
    p0, t0 = (np.asarray(a) for a in rectangular_cross(n, n, float(n), float(n))[:2])
    p1, t1 = (np.asarray(a) for a in rectangular_cross(m, m, float(m), float(m))[:2])
    points = [p0] + [p1 + [n + 10.0, 0.0]] * sheets
    triangles = [t0] + [t1 + len(p0) + i * len(p1) for i in range(sheets)]
    return Mesh(np.concatenate(points), np.concatenate(triangles))


@pytest.mark.parametrize("alg", ["DE0", "DE1", "DE2"])
@pytest.mark.parametrize("n", [40, 460])
def test_crowded_tiles_leave_the_others_on_the_fast_kernel(monkeypatch, n, alg):
    """Below and above the number of tiles from which the crowded ones get a
    launch of their own, against the gather kernel over all tiles."""
    print("case crowded tiles %d %s" % (n, alg), flush=True)
    mesh = _stacked_sheets(n)
    if alg == "DE0":
        a = _tables(*_ordered(mesh), crowded=True)
        assert 0 < a["crowded"].sum() < 40
    q = _inputs(mesh, n)
    runs = []
    for once in ("1", "0"):
        monkeypatch.setenv("ANUGA_HIP_EDGE_ONCE", once)
        runs.append(_run(mesh, q, alg, (3, 67) if n < 100 else (3,)))
    _same(*runs)


def _sloped(mesh, q):
    d = Domain(mesh=mesh)
    d.set_flow_algorithm("DE1")
    for n, v in q.items():
        d.set_quantity(n, v, location="centroids")
    d.set_boundary({t: Reflective_boundary(d) for t in d.get_boundary_tags()})
    d.evolve_steps(2)
    before = torch.cuda.mem_get_info()[0]
    d.set_sloped_mannings_function(True)
    d.evolve_steps(1)
    taken = before - torch.cuda.mem_get_info()[0]
    d.evolve_steps(4)
    return taken, [d.get_quantity(n).centroid_values for n in NAMES]


@pytest.mark.parametrize("mesh", [lambda: Mesh(*rectangular_cross(201, 197, 201.0, 197.0)),
                                  lambda: _stacked_sheets(200)])
def test_vertex_coordinates_are_formed_for_sloped_friction(monkeypatch, mesh):
    """Only sloped friction reads the vertex coordinates per triangle: they
    take their 48 B when it is first set, formed from the nodes of the tiles.
    Meshes without such nodes (here: the gather kernel over all tiles) have
    them from the start, and the same steps."""
    print("case sloped friction set late", flush=True)
    mesh = mesh()
    q = _inputs(mesh, 2)
    crowded = mesh.number_of_triangles != 4 * 201 * 197
    taken, a = _sloped(mesh, q)
    # allocations come in pieces of 2 MiB
    assert abs(taken - (0 if crowded else 48 * mesh.number_of_triangles)) <= 2 << 21
    monkeypatch.setenv("ANUGA_HIP_EDGE_ONCE", "0")
    taken, b = _sloped(mesh, q)
    assert abs(taken) <= 2 << 21
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


# the switches of the two kernels that a mesh within the limits leaves unused:
# stored geometry (vertices that do not reproduce the mesh's arrays) and the
# gather kernel (normals that do not mirror, tiles beyond the limits)
KERNELS = [("ANUGA_HIP_VERTEX_GEOMETRY", "0"), ("ANUGA_HIP_EDGE_ONCE", "0")]
MESHES = {"graded": lambda: Mesh(*graded_square(300.0, 9.0, 40.0, (100.0, 100.0, 200.0, 200.0),
                                                seed=3)),
          "ragged": lambda: Mesh(*rectangular_cross(37, 53, 60.0, 70.0)),
          "tiny": lambda: Mesh(*rectangular_cross(1, 1, 1.0, 1.0))}


@pytest.mark.parametrize("name,value", KERNELS)
@pytest.mark.parametrize("alg", ["DE0", "DE1", "DE2"])
@pytest.mark.parametrize("mesh", sorted(MESHES))
def test_kernels_give_the_same_bits(monkeypatch, mesh, alg, name, value):
    print("case %s %s %s" % (mesh, alg, name), flush=True)
    mesh = MESHES[mesh]()
    q = _inputs(mesh, 7)
    usual = _run(mesh, q, alg, (5, 68))
    monkeypatch.setenv(name, value)
    _same(_run(mesh, q, alg, (5, 68)), usual)


@pytest.mark.parametrize("name,value", KERNELS)
@pytest.mark.parametrize("alg", ["DE0", "DE1"])
def test_ensemble_kernels_give_the_same_bits(monkeypatch, alg, name, value):
    print("case ensemble %s %s" % (alg, name), flush=True)
    meshes = [MESHES[m]() for m in ("tiny", "ragged", "graded", "tiny")]
    runs = []
    for switch in (False, True):
        if switch:
            monkeypatch.setenv(name, value)
        e = Ensemble(meshes, flow_algorithm=alg)
        for s, mesh in enumerate(meshes):
            tags = sorted(mesh.get_boundary_tags())
            kinds = ["reflective", ("dirichlet", [0.3, 0.2, -0.1]), "transmissive"]
            e.set_scenario(s, mesh, _inputs(mesh, s), {t: kinds[i % 3] for i, t in enumerate(tags)})
        e.evolve_steps(3)
        e.evolve_steps(67)
        runs.append(([e.get_quantity(s, n) for s in range(len(meshes)) for n in NAMES],
                     [e.get_time(s) for s in range(len(meshes))],
                     list(e.get_boundary_flux_integrals())))
    _same(*runs)


@pytest.mark.parametrize("alg", ["DE0", "DE1", "DE2"])
@pytest.mark.parametrize("sides", [1, 2])
def test_meshes_whose_geometry_is_their_own(sides, alg):
    """Lengths that the vertices do not give, on both sides of an edge (the
    once-per-edge kernel reads the stored geometry) and on one (an edge has two
    fluxes: the gather kernel), against the separate kernels."""
    print("case own geometry %d %s" % (sides, alg), flush=True)
    mesh = MESHES["graded"]()
    el = mesh.edgelengths.copy()
    for k in range(5, mesh.number_of_triangles, 97):
        n, j = mesh.neighbours[k, 1], mesh.neighbour_edges[k, 1]
        el[k, 1] = np.nextafter(el[k, 1], np.inf)
        if n >= 0 and sides == 2:
            el[n, j] = el[k, 1]
    mesh.edgelengths = el
    q = _inputs(mesh, 11)
    a, b = (_run(mesh, q, alg, (5, 68), reorder=r) for r in ("tiles", "rcm"))
    assert a[1] == b[1]
    for x, y in zip(a[0], b[0]):
        assert np.array_equal(x, y)

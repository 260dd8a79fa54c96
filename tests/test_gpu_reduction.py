"""The per-block partials' reductions at the block counts where their form
changes: one chunk per block (up to 32 blocks), one lane per block of a chunk
(up to 2048 blocks), and chunk workgroups above. Device-controlled steps (the
timestep formed in the update kernel, the boundary flux in the end-of-step
kernel) against host-sequenced ones, bit for bit; volumes against a sum in
extended precision."""

import math

import numpy as np
import pytest

from anuga_core_amd.boundaries import (Dirichlet_boundary, Reflective_boundary,
                                       Transmissive_boundary)
from anuga_core_amd.domain import Domain
from anuga_core_amd.ensemble import Ensemble
from anuga_core_amd.mesh import Mesh, rectangular

pytestmark = pytest.mark.gpu

NAMES = ("stage", "xmomentum", "ymomentum")


def _inputs(mesh, seed):
    rng = np.random.default_rng(seed)
    N = mesh.number_of_triangles
    x, y = mesh.centroid_coordinates.T
    z = -2.0 + 0.3 * np.sin(x / 3.0) + 0.2 * np.cos(y / 2.0)
    return dict(elevation=z, stage=0.2 * rng.random(N), friction=np.full(N, 0.03),
                xmomentum=0.3 * rng.standard_normal(N), ymomentum=0.3 * rng.standard_normal(N))


def _domain(mesh, q, alg):
    d = Domain(mesh=mesh)
    d.set_flow_algorithm(alg)
    for n, v in q.items():
        d.set_quantity(n, v, location="centroids")
    d.set_boundary({"left": Dirichlet_boundary([0.3, 0.1, 0.0]), "right": Transmissive_boundary(d),
                    "top": Reflective_boundary(d), "bottom": Reflective_boundary(d)})
    return d


@pytest.mark.parametrize("alg", ["DE0", "DE1", "DE2"])
@pytest.mark.parametrize("m,n", [(1, 1), (128, 1), (128, 32), (129, 32), (1024, 256),
                                 (1025, 256)])
def test_device_steps_equal_host_steps(m, n, alg):
    mesh = Mesh(*rectangular(m, n, float(m), float(n)))
    q = _inputs(mesh, m + n)
    runs = []
    for device in (True, False):
        d = _domain(mesh, q, alg)
        d.device_timestep = device
        d.evolve_steps(3)
        d.evolve_steps(4)
        runs.append((d.dt_history, d.get_boundary_flux_integral(),
                     [d.get_quantity(k).centroid_values for k in NAMES]))
        v = d.get_water_volume()
        h = np.maximum(runs[-1][2][0] - q["elevation"], 0.0)
        # a tree of sums over all triangles: at most 40 roundings deep
        assert abs(v - math.fsum(mesh.areas * h)) <= 40 * 2.0 ** -53 * v
    a, b = runs
    assert a[0] == b[0]
    assert a[1] == b[1] and (a[1] != 0.0)
    for x, y in zip(a[2], b[2]):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("alg", ["DE0", "DE1", "DE2"])
def test_runs_that_end_at_yields_equal_host_steps(alg):
    """Odd and even step counts, no-op steps behind a yield and long captured
    runs leave the control blocks as host-sequenced steps do."""
    mesh = Mesh(*rectangular(40, 20, 40.0, 20.0))
    q = _inputs(mesh, 5)
    runs = []
    for device in (True, False):
        d = _domain(mesh, q, alg)
        d.device_timestep = device
        out = []
        for t in d.evolve(yieldstep=0.7, finaltime=6.0):
            out.append((t, d.get_boundary_flux_integral(), d.get_water_volume(),
                        d.recorded_min_timestep, d.recorded_max_timestep, d.number_of_steps))
        d.evolve_steps(151)
        out.append((d.get_time(), d.get_boundary_flux_integral(), d.get_water_volume(),
                    d.timestep, d.flux_timestep, d.number_of_steps))
        runs.append((out, d.dt_history, [d.get_quantity(k).centroid_values for k in NAMES]))
    a, b = runs
    assert a[0] == b[0] and a[1] == b[1]
    for x, y in zip(a[2], b[2]):
        assert np.array_equal(x, y)


def test_ensemble_of_large_and_small_scenarios():
    """The large scenario sends every scenario's partials through the chunk
    stage; the small ones still equal their own domains bit for bit."""
    meshes = [Mesh(*rectangular(m, n, float(m), float(n)))
              for m, n in ((9, 7), (1025, 256), (129, 32))]
    qs = [_inputs(mesh, s) for s, mesh in enumerate(meshes)]
    e = Ensemble(meshes, flow_algorithm="DE1")
    bc = {"left": ("dirichlet", [0.3, 0.1, 0.0]), "right": "transmissive", "top": "reflective",
          "bottom": "reflective"}
    for s, mesh in enumerate(meshes):
        e.set_scenario(s, mesh, qs[s], bc)
    e.evolve_steps(3)
    e.evolve_steps(2)
    integrals, volumes = e.get_boundary_flux_integrals(), e.get_water_volumes()
    for s, mesh in enumerate(meshes):
        d = _domain(mesh, qs[s], "DE1")
        d.evolve_steps(3)
        d.evolve_steps(2)
        assert d.get_time() == e.get_time(s)
        assert d.get_boundary_flux_integral() == integrals[s]
        assert d.get_water_volume() == volumes[s]
        for k in NAMES:
            assert np.array_equal(d.get_quantity(k).centroid_values, e.get_quantity(s, k))

"""The recovery's incidence lists and large copies on the GPU: a field past the staging's buffers against
the oracle, bit for bit, and a fan of tetrahedra about one vertex -- 128 of them (lists formed on the
device) and 512 (a node of more slots than the device sorts: the host's lists) -- whose affine
displacement must recover its constant stress everywhere; and bundles of the last count sorted there
and the first past it."""
import time

import numpy as np
import pytest

import refcpu
import solidfem_amd as sf
from workloads import plate_config

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def test_a_recovery_past_the_staging_buffers_is_bit_identical(ctx):
    w = plate_config(divisions=(41, 39, 2))  # 19188 elements: 6.1 MB of point values, 1.8 MB of nodal values
    ref = refcpu.Problem(w)
    u = 1e-3 * np.random.default_rng(5).standard_normal((ref.node_count, 3))
    rp, rn = ref.recover(u)
    model = sf.Model.from_workload(w)
    for _ in range(2):
        dp, dn = model.recover(ctx, u)
        assert np.array_equal(bits(dp), bits(rp)) and np.array_equal(bits(dn), bits(rn))


def fan(subdivisions):
    """The unit octahedron's faces, each split in four `subdivisions` times and moved to the sphere, coned to its centre."""
    points = [np.array(p, dtype=float) for p in ((1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1))]
    faces = [(a, b, c) for a in (0, 1) for b in (2, 3) for c in (4, 5)]
    for _ in range(subdivisions):
        middle, split = {}, []

        def mid(a, b):
            key = (min(a, b), max(a, b))
            if key not in middle:
                m = points[a] + points[b]
                points.append(m / np.linalg.norm(m))
                middle[key] = len(points) - 1
            return middle[key]

        for a, b, c in faces:
            ab, bc, ca = mid(a, b), mid(b, c), mid(c, a)
            split += [(a, ab, ca), (b, bc, ab), (c, ca, bc), (ab, bc, ca)]
        faces = split
    p = np.array(points + [np.zeros(3)])
    tets = []
    for a, b, c in faces:
        if np.linalg.det(np.array([p[a], p[b], p[c]])) < 0:
            b, c = c, b
        tets.append((len(p) - 1, a, b, c))
    return p, np.array(tets)


@pytest.mark.parametrize("subdivisions", [2, 3])
def test_a_fan_recovers_an_affine_fields_stress(ctx, subdivisions):
    mesh = sf.QuadraticTetMesh.from_linear(sf.TetMesh.new(*fan(subdivisions)))
    model = sf.Model.new(mesh, 1000.0, 0.3)
    gradient = np.array([[1.0, 0.4, -0.2], [0.1, -0.5, 0.3], [0.6, 0.2, 0.8]]) * 1e-3
    points, nodal = model.recover(ctx, mesh.nodes() @ gradient.T)
    e = 0.5 * (gradient + gradient.T)
    lam, mu = 1000.0 * 0.3 / (1.3 * 0.4), 1000.0 / 2.6
    s = lam * np.trace(e) * np.eye(3) + 2 * mu * e
    want = np.array([s[0, 0], s[1, 1], s[2, 2], s[0, 1], s[1, 2], s[2, 0]])
    # a constant strain from rounded nodes, and its least-squares fit over the patch: some hundred
    # roundings of values of the stress's size
    bound = 1e3 * np.finfo(float).eps * np.abs(want).max() * 10
    assert np.abs(points[:, :, 3:9] - want).max() < bound
    assert np.abs(nodal[:, :6] - want).max() < bound


def bundle(tets):
    """`tets` tetrahedra about one vertex, between a ring of points and two poles (the last one may be missing)."""
    ring = (tets + 1) // 2
    angle = 2 * np.pi * np.arange(ring) / ring
    p = np.vstack([np.stack([np.cos(angle), np.sin(angle), 0 * angle], axis=1), [[0, 0, 1], [0, 0, -1], [0, 0, 0]]])
    t = [(ring + 2, i, (i + 1) % ring, ring) for i in range(ring)] + [(ring + 2, (i + 1) % ring, i, ring + 1) for i in range(ring)]
    model = sf.Model.new(sf.QuadraticTetMesh.from_linear(sf.TetMesh.new(p, np.array(t[:tets]))), 1000.0, 0.3)
    return model, 1e-3 * np.random.default_rng(tets).standard_normal((len(model.mesh().nodes()), 3))


@pytest.mark.parametrize("tets", [255, 256, 257, 258])
def test_a_vertex_of_many_elements_is_fitted_from_them_in_order(ctx, tets):
    # the lists are filled in the order of atomics and then put in element order: without that the sums
    # over a node's elements, and the fit to their points, would differ from run to run
    model, u = bundle(tets)
    points, nodal = model.recover(ctx, u)
    for _ in range(5):
        again, nodal_again = model.recover(ctx, u)
        assert np.array_equal(bits(points), bits(again)) and np.array_equal(bits(nodal), bits(nodal_again))
    mesh = model.mesh()
    # a constant strain everywhere comes back, at the hub of all elements too
    gradient = np.array([[1.0, 0.4, -0.2], [0.1, -0.5, 0.3], [0.6, 0.2, 0.8]]) * 1e-3
    _, nodal = model.recover(ctx, mesh.nodes() @ gradient.T)
    e = 0.5 * (gradient + gradient.T)
    lam, mu = 1000.0 * 0.3 / (1.3 * 0.4), 1000.0 / 2.6
    s = lam * np.trace(e) * np.eye(3) + 2 * mu * e
    want = np.array([s[0, 0], s[1, 1], s[2, 2], s[0, 1], s[1, 2], s[2, 0]])
    # as the fans', with elements 40 times as wide as thick: their derivatives round 40 times as far
    assert np.abs(nodal[:, :6] - want).max() < 40 * 1e4 * np.finfo(float).eps * np.abs(want).max()


def test_a_vertex_of_many_elements_costs_no_more_on_the_device(ctx):
    # the last count whose lists the device forms against the first that the host does
    def seconds(tets):
        model, u = bundle(tets)
        best = 1e9
        for _ in range(20):
            t = time.perf_counter()
            model.recover(ctx, u)
            best = min(best, time.perf_counter() - t)
        return best

    assert seconds(256) < 1.5 * seconds(258)

"""Assembly and field kernels at the edges of their tiles, lists and splits,
against the FP64 oracle.

Matrix and right-hand side: an entry is a sum of a few dozen FP32 roundings of
6e-8 of its largest partial sum, so 2e-6 relative bounds the whole.  Field: 6 T
images terms summed in chunks of 16 triangles, the same bound.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from hornlab_metal_bem.procedural import HornSpec
from meshes import buffers_from_arrays, horn_buffers, mesh_buffers, rel_l2, sphere_buffers

pytestmark = pytest.mark.gpu


def _session(buffers, plane=None):
    from hornlab_metal_bem.native import HipBemSession

    return HipBemSession.create_session(buffers, symmetry_plane=plane, check_open_edges=False)


def _soup(n_tri, seed=0):
    """Separate triangles with dofs of their own: three rows per test, so a
    wave's table overflows within its run."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(0.02, 0.3, (n_tri, 1, 3))
    V = (c + rng.uniform(-0.01, 0.01, (n_tri, 3, 3))).reshape(-1, 3)
    V[0, :2] = 0.0  # one vertex on the symmetry planes
    E = np.arange(3 * n_tri).reshape(-1, 3)
    return buffers_from_arrays(V.T, E.T, E, 3 * n_tri, np.full(n_tri, 2))


def _fan(valence):
    """Double cone: two vertices shared by ``valence`` triangles each, longer
    than the list words a lane holds."""
    a = 2 * np.pi * np.arange(valence) / valence
    V = np.concatenate([np.stack([0.1 * np.cos(a), 0.1 * np.sin(a), 0 * a], 1),
                        [[0, 0, 0.08], [0, 0, -0.05]]])
    i = np.arange(valence)
    j = (i + 1) % valence
    F = np.concatenate([np.stack([i, j, np.full(valence, valence)], 1),
                        np.stack([j, i, np.full(valence, valence + 1)], 1)])
    return mesh_buffers(V, F.astype(np.int32), np.full(2 * valence, 2, np.int32))


def _check_assembly(b, plane, k, kim=0.0, beta=None):
    rng = np.random.default_rng(1)
    T = b.n_triangles
    q = (rng.standard_normal(T) + 1j * rng.standard_normal(T)).astype(np.complex64)
    walls = {2: beta} if beta is not None else None
    with _session(b, plane) as s:
        A, rhs = s.assemble_standard_neumann(0.0, k, q, k_imag=kim, impedance_sources=walls)
    rows = None if beta is None else np.where(b.physical_tags_i32 == 2, np.complex64(beta), 0)
    Ao, ro, _ = O.assemble(O.Geometry.from_buffers(b, plane), float(np.float32(k)), q,
                           kim=float(np.float32(kim)), beta=rows)
    assert rel_l2(A, Ao) < 2e-6
    assert rel_l2(rhs, ro) < 2e-6


@pytest.mark.parametrize("n_tri", [1, 15, 16, 17, 18, 19, 37, 64, 65])
def test_tables_that_overflow(require_gpu, n_tri):
    _check_assembly(_soup(n_tri), None, 20.0)


@pytest.mark.parametrize("plane", ["xz", "yz+xz"])
def test_tables_that_overflow_with_images(require_gpu, plane):
    _check_assembly(_soup(30), plane, 20.0, 0.3, 0.2 + 0.1j)


@pytest.mark.parametrize("valence", [8, 9, 12, 13, 40])
def test_long_column_lists(require_gpu, valence):
    _check_assembly(_fan(valence), None, 30.0)


@pytest.mark.parametrize("edge,plane", [(0.05, "yz+xz"), (0.03, "yz+xz"), (0.02, "yz+xz")])
def test_quarter_horn_all_sources_and_walls(require_gpu, edge, plane):
    _check_assembly(horn_buffers(edge_length=edge), plane, 60.0)
    _check_assembly(horn_buffers(edge_length=edge), plane, 60.0, 0.5, 0.3 - 0.2j)


def test_entries_of_distant_pairs_at_a_high_wavenumber(require_gpu):
    """k = 300 1/m on a mesh of 8.9 mm edges: an entry is a sum of over a
    thousand evaluations whose own roundings (phase errors of 4e-6, r times
    roundings of 6e-8 times k) average out, so what it keeps is what they
    share.  8.5e-7 admits the point offset of a test triangle rounded with its
    vertex difference (7.5e-7), not the vertex difference rounded by itself
    as well (9.4e-7)."""
    b = horn_buffers(edge_length=0.0089, seed=2, spec=HornSpec(0.0127, 0.150, 0.150, 0.020, "exponential"))
    q = np.ones(b.n_triangles, np.complex64)
    with _session(b, "yz+xz") as s:
        A, _ = s.assemble_standard_neumann(0.0, 300.0, q)
    Ao, _, _ = O.assemble(O.Geometry.from_buffers(b, "yz+xz"), 300.0, q)
    far = np.ones(A.shape, bool)  # entries whose dofs share no triangle
    dofs = b.p1_local2global_i32.reshape(-1, 3)
    for i in range(3):
        for j in range(3):
            far[dofs[:, i], dofs[:, j]] = False
    assert rel_l2(A[far], Ao[far]) < 8.5e-7


@pytest.mark.parametrize("n_sources", [1, 2, 3])
def test_sources_on_every_triangle(require_gpu, n_sources):
    """Each source's right-hand side solves to the same pressure as alone."""
    b = sphere_buffers(subdivisions=2)
    rng = np.random.default_rng(2)
    T, k = b.n_triangles, np.array([8.0], np.float32)
    q = (rng.standard_normal((n_sources, 1, T)) + 1j * rng.standard_normal((n_sources, 1, T))).astype(np.complex64)
    obs = np.array([[0.0], [0.0], [2.0]], np.float32)
    with _session(b) as s:
        r = s.assemble_solve_evaluate_standard_neumann_batch(
            np.array([400.0]), k, q[0], obs, extra_neumann_dp0=q[1:] if n_sources > 1 else None)[0]
    g = O.Geometry.from_buffers(b)
    for i, got in enumerate([r, *r.extra_sources]):
        A, rhs, _ = O.assemble(g, 8.0, q[i, 0])
        assert rel_l2(got.pressure, O.solve(A, rhs)) < 2e-5  # cond(A) ~ 10


def test_split_and_whole_singular_rules_agree(require_gpu):
    """One frequency per call deals the singular rules over eight waves, 18 in
    one call do not; the pressures differ by FP32 rounding times cond."""
    b = sphere_buffers(subdivisions=3)
    f = np.geomspace(100.0, 1200.0, 18)
    k = (2 * np.pi * f / 343.0).astype(np.float32)
    q = np.ones((18, b.n_triangles), np.complex64)
    obs = np.array([[0.0], [0.0], [2.0]], np.float32)
    with _session(b) as s:
        whole = s.assemble_solve_evaluate_standard_neumann_batch(f, k, q, obs)
        for i in (0, 9, 17):
            one = s.assemble_solve_evaluate_standard_neumann_batch(f[i:i + 1], k[i:i + 1], q[i:i + 1], obs)
            assert rel_l2(one[0].pressure, whole[i].pressure) < 2e-5


def _check_sweep(b, plane, n_freq, tol=2e-5, **kw):
    """A sweep in one resident batch; three of its pressures against the FP64
    oracle: entries good to 1e-7 times the condition number with scaled rows
    (soups 5, the fan 14, the horns up to 170)."""
    f = np.geomspace(300.0, 1500.0, n_freq)
    k = (2 * np.pi * f / 343.0).astype(np.float32)
    q = np.ones((n_freq, b.n_triangles), np.complex64)
    obs = np.array([[0.0], [0.0], [2.0]], np.float32)
    with _session(b, plane) as s:
        r = s.assemble_solve_evaluate_standard_neumann_batch(
            f, k, q, obs, batch_frequencies=n_freq, estimate_rcond=False, **kw)
    assert all(x.diagnostics["resident_batch"]["size"] == n_freq for x in r)
    g = O.Geometry.from_buffers(b, plane)
    for i in sorted({0, n_freq // 2, n_freq - 1}):
        A, rhs, _ = O.assemble(g, float(k[i]), q[i])
        assert rel_l2(r[i].pressure, O.solve(A, rhs)) < tol, i


@pytest.mark.parametrize("plane,n_freq", [
    (None, 21), (None, 22), (None, 42), (None, 43),
    ("xz", 21), ("xz", 22), ("xz", 341), ("xz", 342),
    ("yz+xz", 85), ("yz+xz", 86), ("yz+xz", 341), ("yz+xz", 342)])
def test_whole_halved_and_quartered_runs(require_gpu, plane, n_freq):
    """Tables that overflow, three tiles and so six tile pairs per frequency.
    Up to 128 blocks are cut in four (with four images 512), up to 256 in two
    (with images below 2048), more not at all."""
    _check_sweep(_soup(37), plane, n_freq)


@pytest.mark.parametrize("n_freq", [1, 60, 100])
def test_long_column_lists_whole_halved_and_quartered(require_gpu, n_freq):
    """Two tiles, three tile pairs per frequency: 3, 180 and 300 blocks."""
    _check_sweep(_fan(40), None, n_freq)


@pytest.mark.parametrize("body,plane", [("soup", None), ("soup", "xz"), ("soup", "yz+xz"), ("fan", None),
                                        ("horn", None), ("horn", "xz"), ("horn", "yz+xz")])
def test_fp64_geometry_with_full_tables_and_long_lists(require_gpu, body, plane):
    b = {"soup": lambda: _soup(37), "fan": lambda: _fan(40), "horn": lambda: horn_buffers(edge_length=0.03)}[body]()
    _check_sweep(b, plane, 3, precise_geometry=True)


@pytest.mark.parametrize("plane", [None, "xz", "yz+xz"])
def test_group_with_full_tables_and_long_lists(require_gpu, plane):
    """Members in one launch: overflowing tables beside a member whose tables
    do not, and (without planes) long lists."""
    import torch

    from hornlab_metal_bem.native import GroupCase, HipBemGroup

    bodies = [_soup(37), _soup(30, seed=1), horn_buffers(edge_length=0.04)] + ([_fan(40)] if plane is None else [])
    F, dev = 2, torch.device("cuda:0")
    k = np.array([6.0, 20.0], np.float32)
    sessions, cases, held = [], [], []
    try:
        for b in bodies:
            t = dict(k=torch.as_tensor(k, device=dev),
                     q=torch.ones((F, b.n_triangles), dtype=torch.complex64, device=dev),
                     obs=torch.tensor([[0.0], [0.0], [2.0]], device=dev),
                     field=torch.zeros((F, 1), dtype=torch.complex64, device=dev),
                     p=torch.zeros((F, b.p1_dof_count), dtype=torch.complex64, device=dev),
                     tag=torch.zeros((F, 2), dtype=torch.complex128, device=dev))
            held.append(t)
            sessions.append(_session(b, plane))
            a = {n: v.data_ptr() for n, v in t.items()}
            cases.append(GroupCase(F, a["k"], a["k"], a["q"], 1, a["obs"], a["field"], a["tag"], a["p"]))
        torch.cuda.synchronize()
        with HipBemGroup(sessions) as group:
            group.solve_device(cases, source_tags=[2], impedance_source_tag=2)
        for b, t in zip(bodies, held):
            for i in range(F):
                A, rhs, _ = O.assemble(O.Geometry.from_buffers(b, plane), float(k[i]),
                                       np.ones(b.n_triangles, np.complex64))
                assert rel_l2(t["p"][i].cpu().numpy(), O.solve(A, rhs)) < 2e-5  # as in _check_sweep
    finally:
        for s in sessions:
            s.close()


def _field_terms(b, p, q, obs):
    """Sum of the magnitudes of the identity image's field terms per point."""
    X, Y, W = O.rule6()
    v = b.vertices_3xn_f32[:, b.triangles_3xm_i32].astype(float)  # (3, 3, T)
    y = np.einsum("bl,clt->cbt", np.stack([1 - X - Y, X, Y], 1), v)
    r = np.linalg.norm(y[:, :, :, None] - obs[:, None, None, :], axis=0)
    w = W[:, None, None] * (2 * b.triangle_areas_f32)[None, :, None] / (4 * np.pi)
    return (w * (np.abs(p).max() / r ** 2 + np.abs(q)[None, :, None] / r)).sum((0, 1))


@pytest.mark.parametrize("plane", [None, "yz+xz"])
@pytest.mark.parametrize("n_obs", [1, 63, 64, 65, 257])
def test_field_points_near_and_far(require_gpu, plane, n_obs):
    """Points from 1 mm off the surface to 60 m away, k r up to 1.3e3."""
    b = horn_buffers(edge_length=0.03, quarter=plane is not None)
    rng = np.random.default_rng(3)
    d = rng.standard_normal((3, n_obs))
    obs = (d / np.linalg.norm(d, axis=0) * np.geomspace(0.3, 60.0, n_obs)).astype(np.float32)
    tri = b.triangles_3xm_i32[:, rng.integers(0, b.n_triangles, n_obs)]
    near = b.vertices_3xn_f32[:, tri].mean(axis=1) * np.float32(1.01) + np.float32(1e-3)
    obs[:, ::4] = near[:, ::4]
    k = np.array([20.0], np.float32)
    p = (rng.standard_normal(b.p1_dof_count) + 1j * rng.standard_normal(b.p1_dof_count)).astype(np.complex64)
    q = (20 * rng.standard_normal(b.n_triangles)).astype(np.complex64)
    with _session(b, plane) as s:
        got = s.evaluate_standard_exterior_batch(np.array([1000.0]), k, p[None], q[None], obs)[0]
    want = O.field(O.Geometry.from_buffers(b, plane), 20.0, p, q, obs)
    # near points: each term |p| jac w / (4 pi r^2) + |q| jac w / (4 pi r) of
    # the sum carries about ten roundings of 6e-8, and a few dozen the partial
    # sums, so 4e-6 of the terms' sum bounds the error (the identity image's
    # terms; the others are farther)
    terms = _field_terms(b, p, q, obs[:, ::4])
    assert np.all(np.abs(got - want)[::4] < 4e-6 * terms)
    far = np.ones(n_obs, bool)
    far[::4] = False
    if far.any():
        assert rel_l2(got[far], want[far]) < 5e-6


@pytest.mark.parametrize("plane", [None, "yz+xz"])
def test_field_points_close_to_the_surface(require_gpu, plane):
    """Points 0.05 to 20 mm off 30 mm triangles, over any of their points: the
    nearest quadrature point is up to hundreds of times closer than the
    triangle is wide, and its distance still has to be good to FP32."""
    b = horn_buffers(edge_length=0.03, quarter=plane is not None)
    rng = np.random.default_rng(5)
    n_obs, X, Y = 400, *O.rule6()[:2]
    tri = rng.integers(0, b.n_triangles, n_obs)
    at = rng.dirichlet([1, 1, 1], n_obs)
    a = rng.integers(0, 6, n_obs // 2)
    at[::2] = np.stack([1 - X - Y, X, Y], 1)[a]  # straight above a quadrature point
    v = b.vertices_3xn_f32[:, b.triangles_3xm_i32[:, tri]].astype(float)
    off = np.geomspace(5e-5, 2e-2, n_obs) * b.triangle_normals_3xm_f32[:, tri]
    obs = (np.einsum("ol,clo->co", at, v) - off).astype(np.float32)
    p = (rng.standard_normal(b.p1_dof_count) + 1j * rng.standard_normal(b.p1_dof_count)).astype(np.complex64)
    q = (20 * rng.standard_normal(b.n_triangles)).astype(np.complex64)
    with _session(b, plane) as s:
        got = s.evaluate_standard_exterior_batch(
            np.array([1000.0]), np.array([20.0], np.float32), p[None], q[None], obs)[0]
    want = O.field(O.Geometry.from_buffers(b, plane), 20.0, p, q, obs)
    # about ten roundings of 6e-8 per term
    assert np.all(np.abs(got - want) < 6e-7 * _field_terms(b, p, q, obs))


@pytest.mark.parametrize("precise", [False, True])
@pytest.mark.parametrize("plane", [None, "yz+xz"])
def test_growing_waves_stay_finite(require_gpu, plane, precise):
    """Device arrays may hold k_imag < 0 (the host entry points refuse it):
    e^{-k_imag r} then grows with the distance, which must not reach the lanes
    whose pair is left out."""
    import torch

    b = horn_buffers(edge_length=0.03, quarter=plane is not None)
    k, kim = 20.0, -0.25
    q = (b.physical_tags_i32 == 2).astype(np.complex64)
    dev = {n: torch.as_tensor(a, device="cuda:0") for n, a in dict(
        k=np.array([k], np.float32), kim=np.array([kim], np.float32), q=q[None],
        obs=np.array([[0.1], [0.2], [2.0]], np.float32)).items()}
    field = torch.zeros(1, dtype=torch.complex64, device="cuda:0")
    p = torch.zeros(b.p1_dof_count, dtype=torch.complex64, device="cuda:0")
    tag = torch.zeros(2, dtype=torch.complex128, device="cuda:0")
    with _session(b, plane) as s:
        s.solve_batch_device(1, dev["k"].data_ptr(), dev["k"].data_ptr(), dev["q"].data_ptr(), 1,
                             dev["obs"].data_ptr(), field.data_ptr(), tag.data_ptr(),
                             k_imag_ptr=dev["kim"].data_ptr(), p_ptr=p.data_ptr(), source_tags=[2],
                             precise_geometry=precise)
    A, rhs, _ = O.assemble(O.Geometry.from_buffers(b, plane), k, q, kim=kim)
    assert rel_l2(p.cpu().numpy(), O.solve(A, rhs)) < 2e-5  # entries good to 1e-7, condition 110 with scaled rows


def test_coincident_points_with_fp64_geometry(require_gpu):
    """A triangle given twice, with vertices and dofs of its own each time:
    no common index, so the pair is regular and six distances are zero, which
    add nothing (as in the oracle)."""
    one = _soup(12)
    V = np.concatenate([one.vertices_3xn_f32, one.vertices_3xn_f32[:, :3]], axis=1)
    E = np.arange(39).reshape(13, 3)
    b = buffers_from_arrays(V, E.T, E, 39, np.full(13, 2))
    q = np.ones((1, 13), np.complex64)
    with _session(b) as s:
        r = s.assemble_solve_evaluate_standard_neumann_batch(
            np.array([1000.0]), np.array([20.0], np.float32), q, np.array([[0.0], [0.0], [2.0]], np.float32),
            precise_geometry=True)[0]
    A, rhs, _ = O.assemble(O.Geometry.from_buffers(b), 20.0, q[0])
    assert rel_l2(r.pressure, O.solve(A, rhs)) < 2e-5  # condition 4 with scaled rows

"""The work a user has the solver do, as cases that can be timed and compared.

Each case is one call (or one training-like step) through the package's
public entry points: single frequencies and small spheres where latency
counts, the sweeps a horn designer runs, uneven groups, the shape gradient,
field maps and plain dense solves.  ``listed()`` gives the fixed cases,
``draw(rng)`` more of the same ranges, ``prepare``/``run`` what a program
holds before the call and the call itself, ``exact`` the same outputs in
64 bits from plain torch.
"""
import math
import sys
from functools import lru_cache
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "hornlab-metal-bem_amd"))

from hornlab_metal_bem import ObservationConfig, native_config, solve  # noqa: E402
from hornlab_metal_bem.adjoint import (  # noqa: E402
    FieldProblem,
    directivity_ripple_loss,
    exterior_field,
)
from hornlab_metal_bem.geometry import build_geometry_buffers  # noqa: E402
from hornlab_metal_bem.mesh import (  # noqa: E402
    loaded_mesh_from_arrays,
    make_pure_function_spaces,
    make_pure_grid,
)
from hornlab_metal_bem.native import GroupCase, HipBemGroup, HipBemSession, dense_solve  # noqa: E402
from hornlab_metal_bem.procedural import HornSpec, horn_body, icosphere  # noqa: E402

SPEED, DENSITY = 343.0, 1.2041
FLARES = ("exponential", "conical", "tractrix")


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------


def listed():
    return [
        # one frequency of a small body: an interactive call, all latency
        dict(name="sphere_one", kind="host", body="sphere", level=2, nf=1, fmin=700.0, fmax=700.0,
             angles=37, mode="fp32"),
        # closed sphere across its interior resonances, made well posed by
        # CHIEF points (642 dofs, 10 frequencies)
        dict(name="sphere_chief", kind="host", body="sphere", level=3, nf=10, fmin=200.0,
             fmax=4000.0, angles=37, mode="fp32", chief=6),
        # one frequency of a quarter horn with device arrays
        dict(name="quarter_one", kind="device", body="quarter", edge=0.0089, nf=1, fmin=3000.0,
             fmax=3000.0, angles=37, mode="fp32"),
        # the sweep the framework is quoted on: quarter horn, 40 frequencies,
        # FP16 trailing updates + GMRES-IR
        dict(name="quarter_sweep", kind="device", body="quarter", edge=0.0089, nf=40, fmin=500.0,
             fmax=20000.0, angles=37, mode="mixed_fp16"),
        # the same design evaluated with solve(): session set-up, sweep and
        # result from a loaded mesh, as a design loop calls it
        dict(name="quarter_solve", kind="solve", body="quarter", edge=0.0089, nf=40, fmin=500.0,
             fmax=20000.0, angles=37, mode="fp32"),
        # half horn with impedance walls, lossy wavenumbers, near-field
        # quadrature and two drivers sharing each operator
        dict(name="half_robin", kind="host", body="half", edge=0.0121, nf=12, fmin=300.0,
             fmax=9000.0, angles=19, mode="fp32", robin=True, lossy=True, near=1, sources=2),
        # full body without symmetry, a moderate sweep in FP32
        dict(name="full_mid", kind="device", body="full", edge=0.0121, nf=16, fmin=300.0,
             fmax=9000.0, angles=73, mode="fp32"),
        # full body of about 8000 dofs, mixed precision
        dict(name="full_large", kind="device", body="full", edge=0.0063, nf=16, fmin=200.0,
             fmax=16000.0, angles=181, mode="mixed_fp16"),
        # design variants of uneven order solved as one group
        dict(name="group_uneven", kind="group", body="quarter", edge=0.0062, spread=2.2, members=6,
             nf=6, fmin=300.0, fmax=18000.0, angles=37, mode="fp32"),
        # one step of a shape optimisation: field, loss and gradients
        dict(name="adjoint_step", kind="adjoint", body="quarter", edge=0.0065, nf=6, fmin=1000.0,
             fmax=12000.0, angles=37, mode="fp32_ir"),
        # radiation balloon from known surface data
        dict(name="field_balloon", kind="field", body="quarter", edge=0.0089, nf=40, fmin=500.0,
             fmax=20000.0, angles=864, mode="fp32"),
        # dense complex systems of the caller's own
        dict(name="dense_systems", kind="dense", n=1200, nf=4, mode="fp32"),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["host", "host", "device", "device", "device", "solve", "group", "adjoint",
                       "field", "dense"])
    if kind == "dense":
        n = int(_log(rng, 60, 3000))
        nf = max(1, int(_log(rng, 1, 16) * min(1.0, (1200.0 / n) ** 2)))
        return dict(kind=kind, n=n, nf=nf,
                    mode=rng.choice(["fp32", "fp32_ir", "mixed_fp16", "mixed_bf16", "fp64"]))
    fmin = _log(rng, 200.0, 1000.0)
    case = dict(kind=kind, fmin=round(fmin, 3), angles=int(_log(rng, 5, 181)), mode="fp32")
    body = rng.choice(["quarter", "quarter", "half", "full"])
    if kind == "solve" or kind == "group" or kind == "adjoint":
        body = "quarter"
    if kind == "host" and rng.random() < 0.4:
        body = "sphere"
    case["body"] = body
    if body == "sphere":
        case.update(level=rng.choice([1, 2, 3]), nf=int(_log(rng, 1, 24)),
                    fmax=round(_log(rng, 1000.0, 4000.0), 3))
        if case["fmax"] > 1500.0:
            case["chief"] = rng.randint(4, 9)
        return case
    lo = {"quarter": 0.0065, "half": 0.0100, "full": 0.0110}[body]
    hi = {"quarter": 0.0300, "half": 0.0400, "full": 0.0450}[body]
    case["edge"] = round(_log(rng, lo, hi), 5)
    if body == "full" and rng.random() < 0.25:
        case["edge"] = round(_log(rng, 0.0068, 0.0110), 5)
    # the mesh resolves the highest frequency with at least two edges a wavelength
    top = min(20000.0, 0.5 * SPEED / case["edge"])
    case["fmax"] = round(max(fmin * 1.5, _log(rng, 0.4, 1.0) * top), 3)
    case["nf"] = int(_log(rng, 1, 12 if body == "full" else 40))
    if kind == "host":
        case.update(robin=rng.random() < 0.5, lossy=rng.random() < 0.5, near=rng.choice([0, 0, 1]),
                    sources=rng.choice([1, 1, 2, 3]), nf=min(case["nf"], 12))
    elif kind == "device":
        case["mode"] = rng.choice(["fp32", "fp32_ir", "mixed_fp16", "mixed_bf16", "fp64"])
    elif kind == "group":
        case.update(members=rng.randint(2, 6), spread=round(rng.uniform(1.2, 2.5), 3),
                    nf=min(case["nf"], 8))
    elif kind == "adjoint":
        case.update(mode="fp32_ir", nf=min(case["nf"], 8), edge=max(case["edge"], 0.007),
                    angles=min(case["angles"], 73))
    elif kind == "field":
        case["angles"] = int(_log(rng, 1, 1000))
    return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _weld(V, F, T, signs):
    """Mirror images of a body across coordinate planes, shared vertices joined."""
    keys, verts, tris = {}, [], []
    for s in signs:
        remap = np.empty(len(V), np.int64)
        for i, p in enumerate(V * np.asarray(s)):
            key = tuple(np.round(p / 1e-9).astype(np.int64).tolist())
            remap[i] = keys.setdefault(key, len(verts))
            if remap[i] == len(verts):
                verts.append(p)
        t = remap[F]
        tris.append(t[:, [0, 2, 1]] if np.prod(s) < 0 else t)
    return np.array(verts), np.vstack(tris).astype(np.int32), np.concatenate([T] * len(signs))


def _body(case, seed, member=0):
    """(vertices, triangles, tags, symmetry plane) of a case's mesh."""
    body = case["body"]
    if body == "sphere":
        V, F = icosphere(0.1 * (1.0 + 0.02 * np.random.default_rng(seed).uniform(-1, 1)), case["level"])
        return V, F, np.full(len(F), 2, np.int32), None
    h = case["edge"]
    if case["kind"] == "group" and case["members"] > 1:
        h *= case["spread"] ** (member / (case["members"] - 1.0))
    spec = HornSpec(0.0127, 0.150, 0.150, 0.020, FLARES[member % 3])
    V, F, T = horn_body(spec, edge_length=h, quarter=body != "full", jitter=0.05, seed=seed * 64 + member)
    if body == "half":
        V, F, T = _weld(V, F, T, [(1, 1, 1), (-1, 1, 1)])
    return V, F, T, {"quarter": "yz+xz", "half": "xz", "full": None}[body]


def _buffers(V, F, T):
    grid = make_pure_grid(V, F)
    p1, dp0 = make_pure_function_spaces(grid)
    return build_geometry_buffers(grid, T, p1, dp0)


def _points(case):
    """Observation points (3, 3 * angles): three arcs of half circles at 2 m."""
    a = np.linspace(0.0, math.pi, case["angles"])
    z, r = np.cos(a), np.sin(a)
    arcs = [np.stack([2 * r * math.cos(p), 2 * r * math.sin(p), 0.15 + 2 * z])
            for p in (0.0, 0.5 * math.pi, 0.25 * math.pi)]
    return np.ascontiguousarray(np.concatenate(arcs, axis=1), np.float32)


def _inputs(case, seed, member=0):
    """Everything a case's call is given, as numpy arrays."""
    rng = np.random.default_rng([seed, member])
    if case["kind"] == "dense":
        n, S = case["n"], case["nf"]
        A = (rng.standard_normal((S, n, n), np.float32) + 1j * rng.standard_normal((S, n, n), np.float32))
        A *= np.float32(0.5 / math.sqrt(n))
        A[:, np.arange(n), np.arange(n)] += 1.0
        b = rng.standard_normal((S, n)) + 1j * rng.standard_normal((S, n))
        return dict(A=A.astype(np.complex64), b=b.astype(np.complex64))
    V, F, T, plane = _body(case, seed, member)
    b = _buffers(V, F, T)
    nf = case["nf"]
    freqs = np.geomspace(case["fmin"], case["fmax"], nf) if nf > 1 else np.array([case["fmax"]])
    freqs = freqs * (1.0 + 0.002 * rng.uniform(-1, 1))
    k = (2 * np.pi * freqs / SPEED).astype(np.float32)
    tags = b.physical_tags_i32
    n3 = b.triangle_normals_3xm_f32.astype(np.float64)
    S = case.get("sources", 1)
    q = np.zeros((S, nf, b.n_triangles), np.complex64)
    for s in range(S):
        # a driver on the throat: rigid piston, then pistons with a phase
        # gradient; a sphere vibrates along an axis of its own
        c = b.vertices_3xn_f32[:, b.triangles_3xm_i32].mean(axis=1)
        if case["body"] == "sphere":
            axis = rng.standard_normal(3)
            vel = 0.5 + (axis / np.linalg.norm(axis)) @ n3
        else:
            vel = n3[2] * np.exp(40j * s * c[0])
        amp = 1.0 + 0.2 * rng.uniform(-1, 1)
        q[s] = 1j * DENSITY * 2 * np.pi * freqs[:, None] * np.where(tags == 2, amp * vel, 0.0)
    beta = None
    if case.get("robin"):
        # absorbing walls, per frequency
        beta = [{1: complex(0.05 + 0.1 * i / nf, 0.02 * amp)} for i in range(nf)]
    chief = None
    if case.get("chief"):
        d = rng.standard_normal((3, case["chief"]))
        chief = (0.06 * rng.uniform(0.3, 1.0, case["chief"]) * d / np.linalg.norm(d, axis=0)).astype(np.float32)
    p = None
    if case["kind"] == "field":
        p = np.zeros((nf, b.p1_dof_count), np.complex64)
        for f in range(nf):
            phase = k[f] * (rng.standard_normal(3) / 1.8) @ b.vertices_3xn_f32
            p[f] = (400.0 * np.exp(1j * phase))[: b.p1_dof_count]
        q += (400.0 * k[:, None] * np.exp(1j * rng.uniform(0, 6.28, (nf, b.n_triangles)))).astype(np.complex64)
    return dict(V=V, F=F, T=T, plane=plane, buffers=b, freqs=freqs, k=k, q=q, beta=beta, chief=chief,
                obs=_points(case), p=p,
                k_imag=(0.005 * k.astype(np.float64)).astype(np.float32) if case.get("lossy") else None)


class _Device:
    """A sweep's device arrays, as a program with resident inputs keeps them."""

    def __init__(self, x):
        dev = torch.device("cuda:0")
        F, n, m = len(x["k"]), x["buffers"].p1_dof_count, x["obs"].shape[1]
        self.k = torch.from_numpy(x["k"]).to(dev)
        self.q = torch.from_numpy(np.ascontiguousarray(x["q"][0])).to(dev)
        self.obs = torch.from_numpy(x["obs"]).to(dev)
        self.field = torch.zeros((F, m), dtype=torch.complex64, device=dev)
        self.p = torch.zeros((F, n), dtype=torch.complex64, device=dev)
        self.tag = torch.zeros((F, 2), dtype=torch.complex128, device=dev)
        self.F, self.m = F, m


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dense":
        return dict(case=case, **_inputs(case, seed))
    if kind == "group":
        xs = [_inputs(case, seed, i) for i in range(case["members"])]
        sessions = [HipBemSession.create_session(x["buffers"], symmetry_plane=x["plane"]) for x in xs]
        dev = [_Device(x) for x in xs]
        cases = [GroupCase(d.F, d.k.data_ptr(), d.k.data_ptr(), d.q.data_ptr(), d.m, d.obs.data_ptr(),
                           d.field.data_ptr(), d.tag.data_ptr(), d.p.data_ptr()) for d in dev]
        torch.cuda.synchronize()
        return dict(case=case, group=HipBemGroup(sessions), sessions=sessions, dev=dev, cases=cases)
    x = _inputs(case, seed)
    if kind == "solve":
        mesh = loaded_mesh_from_arrays(x["V"], x["F"], x["T"], native_symmetry_plane=x["plane"])
        arcs = dict(zip(("horizontal", "vertical", "diagonal"),
                        x["obs"].T.astype(np.float64).reshape(3, -1, 3)))
        config = native_config(
            freq_min_hz=float(x["freqs"][0]), freq_max_hz=float(x["freqs"][-1]), freq_count=case["nf"],
            native_symmetry_plane=x["plane"], return_surface_pressure=True,
            observation=ObservationConfig(planes=list(arcs), custom_points=arcs))
        return dict(case=case, mesh=mesh, config=config)
    if kind == "adjoint":
        dev = torch.device("cuda:0")
        b = x["buffers"]
        problem = FieldProblem.from_buffers(b, x["k"], x["obs"], symmetry_plane=x["plane"],
                                            solve_mode=case["mode"], source_tags=(2,),
                                            impedance_source_tag=2)
        V = torch.tensor(np.asarray(b.vertices_3xn_f32, np.float64), device=dev, requires_grad=True)
        q = torch.tensor(x["q"][0], device=dev, requires_grad=True)
        return dict(case=case, problem=problem, V=V, q=q)
    session = HipBemSession.create_session(x["buffers"], symmetry_plane=x["plane"])
    if case.get("near"):
        session.set_near_quadrature(case["near"])
    state = dict(case=case, session=session, x=x)
    if kind == "device":
        state["dev"] = _Device(x)
        torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "dense":
        x, _ = dense_solve(state["A"], state["b"], solve_mode=case["mode"])
        return x
    if kind == "group":
        state["group"].solve_device(state["cases"], source_tags=[2], impedance_source_tag=2)
        return [dict(field=d.field, p=d.p, tag=d.tag) for d in state["dev"]]
    if kind == "solve":
        r = solve(state["mesh"], state["config"])
        return dict(pressure=r.pressure_complex, directivity=r.directivity_db, impedance=r.impedance,
                    average=r.surface_pressure_avg[2], surface=r.surface_pressure_complex)
    if kind == "adjoint":
        V, q = state["V"], state["q"]
        V.grad = q.grad = None
        field = exterior_field(V, q, state["problem"])
        loss = directivity_ripple_loss(field, 3, case["angles"])
        loss.backward()
        return dict(loss=loss.detach(), field=field.detach(), grad_vertices=V.grad, grad_q=q.grad)
    s = state["session"]
    if kind == "device":
        d = state["dev"]
        s.solve_batch_device(
            d.F, d.k.data_ptr(), d.k.data_ptr(), d.q.data_ptr(), d.m, d.obs.data_ptr(),
            d.field.data_ptr(), d.tag.data_ptr(), p_ptr=d.p.data_ptr(), source_tags=[2],
            impedance_source_tag=2, solve_mode=case["mode"], estimate_rcond=True,
            refine_tolerance=1e-6 if case["mode"].startswith("mixed") else 1e-7,
            refine_max_iterations=20)
        return dict(field=d.field, p=d.p, tag=d.tag)
    x = state["x"]
    if kind == "field":
        return s.evaluate_standard_exterior_batch(x["freqs"], x["k"], x["p"], x["q"][0], x["obs"])
    res = s.assemble_solve_evaluate_standard_neumann_batch(
        x["freqs"], x["k"], x["q"][0], x["obs"], k_imag_f32=x["k_imag"], source_tags=[2],
        impedance_source_tag=2, solve_mode=case["mode"], impedance_sources=x["beta"],
        extra_neumann_dp0=x["q"][1:] if len(x["q"]) > 1 else None, chief_points=x["chief"])
    # [frequency][source]
    rows = [[r, *r.extra_sources] for r in res]
    return dict(field=np.array([[s.field for s in r] for r in rows]),
                p=np.array([[s.pressure for s in r] for r in rows]),
                average=np.array([[s.surface_pressure_avg[2] for s in r] for r in rows]))


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how close two correct passes are
# ---------------------------------------------------------------------------


@lru_cache(maxsize=None)
def _counts(body, edge, level, kind, members, spread):
    case = dict(body=body, edge=edge, level=level, kind=kind, members=members, spread=spread)
    out = []
    for i in range(members if kind == "group" else 1):
        V, F, _, _ = _body(case, 0, i)
        out.append((len(V), len(F)))
    return out


def work(case):
    """Flops: 80 per kernel evaluation (G, its normal derivative and their
    block sums) of the assembly and of the field, 8/3 n^3 per complex LU.
    A shape gradient evaluates every pair once more.  Bytes: inputs and
    outputs once."""
    F = case["nf"]
    if case["kind"] == "dense":
        n = case["n"]
        return dict(bytes=8.0 * F * (n * n + 2 * n), flops=8.0 / 3.0 * F * n ** 3)
    images = {"sphere": 1, "full": 1, "half": 2, "quarter": 4}[case["body"]]
    m = 3 * case["angles"]
    S = case.get("sources", 1)
    flops = total = 0.0
    for n, T in _counts(case["body"], case.get("edge"), case.get("level"), case["kind"],
                        case.get("members"), case.get("spread")):
        field = 80.0 * F * m * T * 6 * images * S
        pairs = 80.0 * F * float(T) ** 2 * 36 * images
        if case["kind"] == "field":
            pairs, lu = 0.0, 0.0
        else:
            lu = 8.0 / 3.0 * F * float(n) ** 3
        if case["kind"] == "adjoint":
            pairs, field = 2 * pairs, 2 * field
        flops += field + pairs + lu
        total += 8.0 * F * S * (T + n + m) + 60.0 * T
    return dict(bytes=total, flops=flops)


def tolerance(case):
    """Relative 2-norms; about four times the largest distance from the
    64-bit outputs, or between two passes, seen over listed and drawn cases.
    A horn's interior resonances amplify the rounding of a 32-bit matrix
    (condition numbers to 1e5); a vertex gradient is a small remainder of
    large terms; solve() also returns decibels of the nulls of a pattern."""
    rel = {"dense": 4e-6, "field": 1e-6, "adjoint": 3e-3, "solve": 2.5e-4}.get(case["kind"], 2e-4)
    if case.get("body") == "sphere" and case["kind"] != "field":
        rel = 2e-5
    return {"rel": rel}


# ---------------------------------------------------------------------------
# The same outputs in 64 bits, from plain torch
# ---------------------------------------------------------------------------

_R6X = np.array([0.4459484909159651, 0.0915762135097710, 0.1081030181680700,
                 0.4459484909159651, 0.8168475729804590, 0.0915762135097710])
_R6Y = np.array([0.4459484909159651, 0.0915762135097700, 0.4459484909159651,
                 0.1081030181680700, 0.0915762135097700, 0.8168475729804580])
_R6W = 0.5 * np.array([0.2233815896780110, 0.1099517436553220, 0.2233815896780110,
                       0.2233815896780110, 0.1099517436553220, 0.1099517436553220])
_MASKS = {None: [0], "xz": [0, 2], "yz+xz": [0, 1, 2, 3]}


def _bary(x, y):
    return np.stack([1.0 - x - y, x, y], axis=-1)


def _singular_rule(kind):
    """Sauter-Schwab points as barycentric weights of test and trial (Q, 3)
    in the order (shared, shared or free, free), and the weights (Q,)."""
    g, w = np.polynomial.legendre.leggauss(4)
    g, w = 0.5 * (g + 1), 0.5 * w
    e1, xi, e2, e3 = (v.ravel() for v in np.meshgrid(g, g, g, g, indexing="ij"))
    wt = np.einsum("a,b,c,d->abcd", w, w, w, w).ravel() * xi ** 3
    e12, e123 = e1 * e2, e1 * e2 * e3
    if kind == 3:
        wt = wt * e1 ** 2 * e2
        regions = [(1, 1 - e1 + e12, 1 - e123, 1 - e1, wt), (1 - e123, 1 - e1, 1, 1 - e1 + e12, wt),
                   (1, e1 - e12 + e123, 1 - e12, e1 - e12, wt), (1 - e12, e1 - e12, 1, e1 - e12 + e123, wt),
                   (1 - e123, e1 - e123, 1, e1 - e12, wt), (1, e1 - e12, 1 - e123, e1 - e123, wt)]
    elif kind == 2:
        wt = wt * e1 ** 2
        regions = [(1, e1 * e3, 1 - e12, e1 * (1 - e2), wt), (1, e1, 1 - e123, e12 * (1 - e3), wt * e2),
                   (1 - e12, e1 * (1 - e2), 1, e123, wt * e2), (1 - e123, e12 * (1 - e3), 1, e1, wt * e2),
                   (1 - e123, e1 * (1 - e2 * e3), 1, e12, wt * e2)]
    else:
        wt = wt * e2
        regions = [(1, e1, e2, e2 * e3, wt), (e2, e2 * e3, 1, e1, wt)]
    t, s, ws = [], [], []
    for a1, a2, b1, b2, ww in regions:
        t.append(_bary(xi * a1 - xi * a2, xi * a2))
        s.append(_bary(xi * b1 - xi * b2, xi * b2))
        ws.append(ww)
    return np.concatenate(t), np.concatenate(s), np.concatenate(ws)


def _subdivided(level):
    """Barycentric points (Q, 3) and weights of the six-point rule on the
    4**level equal parts of a triangle."""
    tris = [np.eye(3)]
    for _ in range(level):
        tris = [np.array(p) for t in tris for a, b, c in [t]
                for p in ((a, (a + b) / 2, (c + a) / 2), ((a + b) / 2, b, (b + c) / 2),
                          ((c + a) / 2, (b + c) / 2, c), ((a + b) / 2, (b + c) / 2, (c + a) / 2))]
    r6 = _bary(_R6X, _R6Y)
    return np.concatenate([r6 @ t for t in tris]), np.concatenate([_R6W / len(tris)] * len(tris))


class _Exact:
    """One mesh's system in complex128 on the GPU."""

    def __init__(self, x, vertices=None):
        b = x["buffers"]
        self.d = torch.device("cuda:0")
        self.tri = torch.as_tensor(b.triangles_3xm_i32.T.astype(np.int64), device=self.d)
        self.dof = torch.as_tensor(b.p1_local2global_i32.reshape(-1, 3).astype(np.int64), device=self.d)
        self.n, self.T = b.p1_dof_count, b.n_triangles
        self.masks = _MASKS[x["plane"]]
        self.rw = float(len(self.masks))
        self.sign = {m: torch.tensor([-1.0 if m >> c & 1 else 1.0 for c in range(3)],
                                     dtype=torch.float64, device=self.d) for m in self.masks}
        f64 = lambda a: torch.as_tensor(np.asarray(a, np.float64), device=self.d)  # noqa: E731
        if vertices is None:
            self.P = f64(b.vertices_3xn_f32).T[self.tri]  # (T, 3, 3)
            self.area = f64(b.triangle_areas_f32)
            self.nrm = f64(b.triangle_normals_3xm_f32).T.contiguous()
        else:
            self.P = vertices.T[self.tri]
            N = torch.linalg.cross(self.P[:, 1] - self.P[:, 0], self.P[:, 2] - self.P[:, 0])
            self.area = 0.5 * torch.linalg.norm(N, dim=1)
            self.nrm = N / (2 * self.area)[:, None]
        self.tag = torch.as_tensor(b.physical_tags_i32.astype(np.int64), device=self.d)
        self.B6, self.W6 = f64(_bary(_R6X, _R6Y)), f64(_R6W)
        self.y = torch.einsum("bl,tlc->tbc", self.B6, self.P)
        self.pairs = self._touching(np.round(b.vertices_3xn_f32.astype(np.float64).T / 1e-6).astype(np.int64))
        self.f64 = f64

    def _touching(self, key):
        """{mask: (test, trial, [N, 3, 3] equal vertices)} of touching pairs."""
        tri = self.tri.cpu().numpy()
        out = {}
        for m in self.masks:
            if m == 0:
                kt = ks = tri
            else:
                sg = np.array([-1 if m >> c & 1 else 1 for c in range(3)])
                _, inv = np.unique(np.concatenate([key, key * sg]), axis=0, return_inverse=True)
                inv = inv.reshape(-1)
                kt, ks = inv[: len(key)][tri], inv[len(key):][tri]
            at = {}
            for s in range(len(tri)):
                for v in ks[s]:
                    at.setdefault(int(v), []).append(s)
            found = {(t, s) for t in range(len(tri)) for v in kt[t] for s in at.get(int(v), ())}
            ts = np.array(sorted(found), np.int64).reshape(-1, 2)
            out[m] = (ts[:, 0], ts[:, 1], kt[ts[:, 0]][:, :, None] == ks[ts[:, 1]][:, None, :])
        return out

    def _blocks(self):
        """Yields (test, trial, test dofs, trial dofs, image points' rule) of
        the singular pairs, one batch per kind and pair of masks."""
        for m, (t, s, eq) in self.pairs.items():
            for tm in self.masks:
                sm = tm ^ m
                pt = [0, 2, 1] if bin(tm).count("1") & 1 else [0, 1, 2]
                ps = [0, 2, 1] if bin(sm).count("1") & 1 else [0, 1, 2]
                e = eq[:, pt][:, :, ps].reshape(-1, 9)
                count = e.sum(1)
                for kind in (1, 2, 3):
                    sel = np.flatnonzero(count == kind)
                    if sel.size == 0:
                        continue
                    if kind == 3:
                        ot = os_ = np.tile(np.arange(3), (sel.size, 1))
                    else:
                        first = e[sel].argmax(1)
                        l1, r1 = first // 3, first % 3
                        if kind == 2:
                            last = 8 - e[sel][:, ::-1].argmax(1)
                            l2, r2 = last // 3, last % 3
                            ot = np.stack([l1, l2, 3 - l1 - l2], 1)
                            os_ = np.stack([r1, r2, 3 - r1 - r2], 1)
                        else:
                            table = np.array([[0, 1, 2], [1, 0, 2], [2, 1, 0]])
                            ot, os_ = table[l1], table[r1]
                    lt = torch.as_tensor(np.array(pt)[ot], device=self.d)
                    ls = torch.as_tensor(np.array(ps)[os_], device=self.d)
                    yield (kind, tm, sm, torch.as_tensor(t[sel], device=self.d),
                           torch.as_tensor(s[sel], device=self.d), lt, ls)

    def _near(self, threshold=1.5):
        """{mask: (test, trial)} of close pairs that do not touch."""
        P = self.P
        edge = torch.stack([(P[:, i] - P[:, i - 2]).norm(dim=1) for i in range(3)]).amax(0)
        cut2 = (threshold * torch.maximum(edge[:, None], edge[None])) ** 2
        out = {}
        for m in self.masks:
            Q = P * self.sign[m]
            gap = torch.clamp(torch.maximum(Q.amin(1)[None] - P.amax(1)[:, None],
                                            P.amin(1)[:, None] - Q.amax(1)[None]), min=0)
            near = (gap ** 2).sum(-1) <= cut2
            near &= ((P.mean(1)[:, None] - Q.mean(1)[None]) ** 2).sum(-1) < cut2
            t, s, _ = self.pairs[m]
            near[torch.as_tensor(t, device=self.d), torch.as_tensor(s, device=self.d)] = False
            out[m] = torch.nonzero(near, as_tuple=True)
        return out

    @staticmethod
    def _kernel(d, N, k, kim):
        """4 pi G and 4 pi dG/dn for offsets d (..., 3) and normals N."""
        r = (d * d).sum(-1).sqrt()
        rinv = 1.0 / r
        g = torch.polar(rinv if kim == 0.0 else rinv * torch.exp(-kim * r), k * r)
        return g, g * torch.complex(-kim - rinv, torch.full_like(r, k)) * ((d * N).sum(-1) * rinv)

    def system(self, k, kim, q, beta, near):
        """A (n, n) and right-hand sides (S, n) at one wavenumber; q (S, T)."""
        n, T = self.n, self.T
        A = torch.zeros(n * n, 2, dtype=torch.float64, device=self.d)
        rhs = torch.zeros(len(q), n, dtype=torch.complex128, device=self.d)
        fold = None if beta is None else complex(-kim, k) / 3.0 * beta

        def add(t, s, D, S, dt, ds):
            # blocks D (N, 3, 3), S (N, 3) into rows dt and columns ds
            if fold is not None:
                D = D - (S * fold[s][:, None])[:, :, None]
            A.index_add_(0, (dt[:, :, None] * n + ds[:, None, :]).reshape(-1),
                         torch.view_as_real(D.contiguous()).reshape(-1, 2))
            for i in range(len(q)):
                v = (S * q[i][s][:, None]).contiguous()
                torch.view_as_real(rhs[i]).index_add_(0, dt.reshape(-1), torch.view_as_real(v).reshape(-1, 2))

        def rule(t, s, Pt, Ps, N, bt, bs, w, dt, ds, scale, step):
            # an arbitrary rule: points bt, bs (Q, 3), weights w (Q,)
            for i in range(0, len(t), step):
                j = slice(i, i + step)
                X = torch.einsum("ql,nlc->nqc", bt, Pt[j])
                Y = torch.einsum("ql,nlc->nqc", bs, Ps[j])
                g, D = self._kernel(Y - X, N[j][:, None], k, kim)
                jac = scale * (4 * self.area[t[j]] * self.area[s[j]]) / (4 * math.pi)
                D = torch.einsum("nq,qx->nx", D * w, (bt[:, :, None] * bs[:, None, :]).reshape(-1, 9).to(D.dtype))
                S = (g * w) @ bt.to(g.dtype)
                add(t[j], s[j], D.reshape(-1, 3, 3) * jac[:, None, None], S * jac[:, None], dt[j], ds[j])

        Bw = (self.B6 * self.W6[:, None]).to(torch.complex128)
        step = max(1, int(1.5e7 // (T * 36)))
        ar = torch.arange(T, device=self.d)
        for i in range(0, T, step):
            t = ar[i:i + step]
            D = S = 0.0
            for m in self.masks:
                Y, N = self.y * self.sign[m], self.nrm * self.sign[m]
                tt, ss, _ = self.pairs[m]
                d = Y[None, None] - self.y[t][:, :, None, None]  # (t, a, s, b, 3)
                on = np.flatnonzero((tt >= i) & (tt < i + step))
                it, is_ = (torch.as_tensor(v[on], device=self.d) for v in (tt - i, ss))
                d[it, :, is_] = 1.0
                g, h = self._kernel(d, N[:, None], k, kim)
                g[it, :, is_] = 0
                h[it, :, is_] = 0
                D, S = D + h @ Bw, S + g @ self.W6.to(g.dtype)
            jac = self.rw * 4 * self.area[t][:, None] * self.area[None] / (4 * math.pi)
            D = torch.einsum("taj,ai->tij", D.reshape(len(t), 6, -1), Bw)
            S = torch.einsum("tas,ai->tis", S, Bw)
            D = D.reshape(len(t), 3, T, 3).permute(0, 2, 1, 3) * jac[:, :, None, None]
            S = S.permute(0, 2, 1) * jac[:, :, None]
            tp, sp = t.repeat_interleave(T), ar.repeat(len(t))
            add(tp, sp, D.reshape(-1, 3, 3), S.reshape(-1, 3), self.dof[tp], self.dof[sp])
        for kind, tm, sm, t, s, lt, ls in self._blocks():
            bt, bs, w = (self.f64(v) for v in _singular_rule(kind))
            take = lambda P, l: torch.gather(P, 1, l[:, :, None].expand(-1, -1, 3))  # noqa: E731
            rule(t, s, take(self.P[t], lt) * self.sign[tm], take(self.P[s], ls) * self.sign[sm],
                 self.nrm[s] * self.sign[sm], bt, bs, w, self.dof[t].gather(1, lt),
                 self.dof[s].gather(1, ls), 1.0, 8192)
        if near:
            b, w = (self.f64(v) for v in _subdivided(near))
            both = lambda b, w: (b.repeat_interleave(len(b), 0), b.repeat(len(b), 1),  # noqa: E731
                                 w.repeat_interleave(len(w)) * w.repeat(len(w)))
            for m, (t, s) in self._near().items():
                for (bt, bs, ww), sc in ((both(b, w), 1.0), (both(self.B6, self.W6), -1.0)):
                    rule(t, s, self.P[t], self.P[s] * self.sign[m], self.nrm[s] * self.sign[m], bt, bs,
                         ww, self.dof[t], self.dof[s], sc * self.rw, 8192)
        mass = self.area[:, None, None] * (1 + torch.eye(3, dtype=torch.float64, device=self.d)) / 12
        A[:, 0].index_add_(0, (self.dof[:, :, None] * n + self.dof[:, None]).reshape(-1),
                           (-0.5 * self.rw * mass).reshape(-1))
        return torch.view_as_complex(A).reshape(n, n), rhs

    def rows(self, obs, k):
        """E (m, n) and G (m, T): the field is E p - G q."""
        m = obs.shape[1]
        E = torch.zeros(m, self.n, dtype=torch.complex128, device=self.d)
        G = torch.zeros(m, self.T, dtype=torch.complex128, device=self.d)
        o = self.f64(obs).T
        Bw = (self.B6 * self.W6[:, None]).to(torch.complex128)
        step = max(1, int(1e7 // (self.T * 6)))
        for mask in self.masks:
            Y, N = self.y * self.sign[mask], self.nrm * self.sign[mask]
            for i in range(0, m, step):
                g, D = self._kernel(Y[None] - o[i:i + step, None, None], N[:, None], k, 0.0)
                jac = 2 * self.area / (4 * math.pi)
                G[i:i + step] += (g @ self.W6.to(g.dtype)) * jac
                v = ((D @ Bw) * jac[:, None]).reshape(len(g), -1)
                E[i:i + step].index_add_(1, self.dof.reshape(-1), v)
        return E, G

    def average(self, p):
        w = self.area * (self.tag == 2)
        return (p[..., self.dof].mean(-1) * w).sum(-1) / w.sum()


def _solve_exact(x, near=0):
    """(p [F][S][n], field [F][S][m], average [F][S]) of an input set."""
    e = _Exact(x)
    P, Fd = [], []
    for f, k in enumerate(x["k"].astype(np.float64)):
        kim = 0.0 if x["k_imag"] is None else float(x["k_imag"][f])
        q = torch.as_tensor(x["q"][:, f].astype(np.complex128), device=e.d)
        beta = None
        if x["beta"] is not None:
            beta = (e.tag == 1) * complex(np.complex64(x["beta"][f][1]))
        A, b = e.system(k, kim, q, beta, near)
        if x["chief"] is None:
            p = torch.linalg.solve(A, b.T).T
        else:
            C, g = e.rows(x["chief"], k)
            d = q @ g.T
            s = A.abs().sum(1).amax() / C.abs().sum(1).amax()
            M = torch.cat([A, s * C])
            p = torch.linalg.solve(M.mH @ M, M.mH @ torch.cat([b, s * d], 1).T).T
        qt = q if beta is None else q + complex(-kim, k) * beta * p[:, e.dof].mean(-1)
        E, G = e.rows(x["obs"], k)
        P.append(p)
        Fd.append(p @ E.T - qt @ G.T)
    P, Fd = torch.stack(P), torch.stack(Fd)
    return P, Fd, e.average(P)


def _loss(field, angles):
    spl = 20.0 * torch.log10(torch.clamp(field.abs(), min=20e-6 * 1e-6) / 20e-6)
    spl = spl.reshape(len(field), 3, angles)
    axis = spl[:, 0, 0]
    return ((spl - spl[:, :, :1]) ** 2).mean() + ((axis - axis.mean()) ** 2).mean()


def _adjoint_exact(case, x):
    b = x["buffers"]
    V = torch.tensor(np.asarray(b.vertices_3xn_f32, np.float64), device="cuda:0", requires_grad=True)
    with torch.no_grad():
        e = _Exact(x, V)
        ks = x["k"].astype(np.float64)
        q = torch.as_tensor(x["q"][0].astype(np.complex128), device=e.d)
        LU, P, ER = [], [], []
        for f, k in enumerate(ks):
            A, rhs = e.system(k, 0.0, q[f:f + 1], None, 0)
            LU.append(torch.linalg.lu_factor(A))
            P.append(torch.linalg.lu_solve(*LU[-1], rhs.T)[:, 0])
            ER.append(e.rows(x["obs"], k))
        field = torch.stack([E @ p - G @ qf for (E, G), p, qf in zip(ER, P, q)])
    fl = field.clone().requires_grad_(True)
    loss = _loss(fl, case["angles"])
    loss.backward()
    gq = []
    for f, k in enumerate(ks):
        E, G = ER[f]
        with torch.no_grad():
            lam = torch.linalg.lu_solve(*LU[f], (E.mH @ fl.grad[f])[:, None], adjoint=True)[:, 0]
        gq.append(_vertex_terms(x, V, k, q[f], P[f], lam, fl.grad[f]))
    return dict(loss=loss.detach(), field=field, grad_vertices=V.grad, grad_q=torch.stack(gq))


def _vertex_terms(x, V, k, q, p, lam, g):
    """Adds d/dV Re(g^H (E p - G q) + lam^H (V q - A p)) to V.grad with the
    other factors fixed; returns the gradient with respect to q."""
    base = _Exact(x, V.detach())
    qv = q.clone().requires_grad_(True)
    Bc = base.B6.to(torch.complex128)
    T = base.T

    def done(value):
        value.backward()

    def parts():
        P = V.T[base.tri]
        N = torch.linalg.cross(P[:, 1] - P[:, 0], P[:, 2] - P[:, 0])
        return P, N, torch.linalg.norm(N, dim=1)

    u = lambda l, d: (l[d] @ Bc.T)  # noqa: E731  values at the six points
    lam_c = lam.conj()
    w2 = base.W6[:, None] * base.W6[None]
    step = max(1, int(6e6 // (T * 36)))
    o = base.f64(x["obs"]).T
    ostep = max(1, int(6e6 // (T * 6)))
    for m in base.masks:
        sg = base.sign[m]
        tt, ss, _ = base.pairs[m]
        for i in range(0, T, step):
            P, N, jac = parts()
            y = torch.einsum("bl,tlc->tbc", base.B6, P)
            t = torch.arange(i, min(T, i + step), device=base.d)
            keep = torch.ones(len(t), T, dtype=torch.bool, device=base.d)
            on = np.flatnonzero((tt >= i) & (tt < i + step))
            keep[torch.as_tensor(tt[on] - i, device=base.d), torch.as_tensor(ss[on], device=base.d)] = False
            d = (y * sg)[None, None] - y[t][:, :, None, None]
            d = torch.where(keep[:, None, :, None, None], d, torch.ones_like(d))
            G, D = _Exact._kernel(d, (N * sg)[:, None], k, 0.0)
            c = G * (qv * jac)[:, None] - D * u(p, base.dof)
            c = (c * w2[:, None]).sum(-1) * (keep * jac[t][:, None])[:, None]
            done((c.sum(-1) * u(lam_c, base.dof[t])).sum().real * (base.rw / (4 * math.pi)))
        for i in range(0, len(o), ostep):
            P, N, jac = parts()
            y = torch.einsum("bl,tlc->tbc", base.B6, P) * sg
            G, D = _Exact._kernel(y[None] - o[i:i + ostep, None, None], (N * sg)[:, None], k, 0.0)
            c = (D * u(p, base.dof) - G * (qv * jac)[:, None]) @ base.W6.to(torch.complex128)
            done((c.sum(-1) * g[i:i + ostep].conj()).sum().real / (4 * math.pi))
    for kind, tm, sm, t, s, lt, ls in base._blocks():
        bt, bs, w = (base.f64(v) for v in _singular_rule(kind))
        for i in range(0, len(t), 4096):
            P, N, jac = parts()
            tj, sj, lj, rj = t[i:i + 4096], s[i:i + 4096], lt[i:i + 4096], ls[i:i + 4096]
            take = lambda P, l: torch.gather(P, 1, l[:, :, None].expand(-1, -1, 3))  # noqa: E731
            X = torch.einsum("ql,nlc->nqc", bt, take(P[tj], lj) * base.sign[tm])
            Y = torch.einsum("ql,nlc->nqc", bs, take(P[sj], rj) * base.sign[sm])
            G, D = _Exact._kernel(Y - X, (N[sj] * base.sign[sm])[:, None], k, 0.0)
            lc = lam_c[base.dof[tj].gather(1, lj)] @ bt.T.to(torch.complex128)
            pc = p[base.dof[sj].gather(1, rj)] @ bs.T.to(torch.complex128)
            c = ((G * (qv * jac)[sj][:, None] - D * pc) * lc * w).sum(-1) * jac[tj]
            done(c.sum().real / (4 * math.pi))
    _, _, jac = parts()
    mass = (1 + torch.eye(3, dtype=torch.float64, device=base.d)).to(torch.complex128) / 24
    c = ((lam_c[base.dof] @ mass) * p[base.dof]).sum(-1) * jac
    done(c.sum().real * (0.5 * base.rw))
    return qv.grad


def exact(case, seed):
    kind = case["kind"]
    if work(case)["flops"] > (2.2e12 if kind == "adjoint" else 3e12):
        return None  # longer than about 20 s
    host = lambda v: v.cpu().numpy()  # noqa: E731
    if kind == "dense":
        x = _inputs(case, seed)
        A, b = (torch.as_tensor(x[v].astype(np.complex128), device="cuda:0") for v in "Ab")
        return host(torch.linalg.solve(A, b[..., None])[..., 0])
    if kind == "group":
        out = []
        for i in range(case["members"]):
            p, f, a = _solve_exact(_inputs(case, seed, i))
            out.append(dict(field=f[:, 0], p=p[:, 0], tag=a.expand(-1, 2)))
        return out
    x = _inputs(case, seed)
    if kind == "adjoint":
        return _adjoint_exact(case, x)
    if kind == "field":
        e = _Exact(x)
        q = torch.as_tensor(x["q"][0].astype(np.complex128), device=e.d)
        p = torch.as_tensor(x["p"].astype(np.complex128), device=e.d)
        out = []
        for f, k in enumerate(x["k"].astype(np.float64)):
            E, G = e.rows(x["obs"], k)
            out.append(E @ p[f] - G @ q[f])
        return host(torch.stack(out))
    if kind == "solve":
        # uniform unit acceleration of the throat at the configuration's grid
        freqs = np.geomspace(x["freqs"][0], x["freqs"][-1], case["nf"])
        x["k"] = (2 * np.pi * freqs / SPEED).astype(np.float32)
        x["q"] = np.broadcast_to(np.where(x["buffers"].physical_tags_i32 == 2, np.float32(DENSITY), 0),
                                 x["q"].shape).astype(np.complex64)
        p, f, a = (v[:, 0] for v in _solve_exact(x))
        f = f.reshape(len(freqs), 3, -1)
        spl = 20.0 * torch.log10(torch.clamp(f.abs(), min=20e-6 * 1e-6))
        return dict(pressure=host(f), directivity=host(spl - spl[:, :, :1]), impedance=host(a),
                    average=host(a), surface=host(p))
    p, f, a = _solve_exact(x, case.get("near", 0))
    if kind == "device":
        return dict(field=f[:, 0], p=p[:, 0], tag=a.expand(-1, 2))
    return dict(field=host(f), p=host(p), average=host(a))

"""Performance cases of the solver library: what a finite element program has it do, from the
smallest single solve to a refined mixed-precision factorization, each one pass through the
public entry points (fieldcraft_amd.cholesky, fieldcraft_amd.assembly).

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what the program holds before the call
    run(state)           one pass; returns its outputs
    work(case)           the bytes and operations a pass cannot do without
    exact(case, seed)    the outputs in 64-bit arithmetic by plain torch, where they have such values

The meshes are structured hex8 and tet10 blocks (fieldcraft_amd.problems). The seed sets the
material's stiffness and the loads; the mesh, and with it the pattern, belongs to the case.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from fieldcraft_amd import assembly as AS
from fieldcraft_amd import cholesky as CH
from fieldcraft_amd import problems as P

DEV = "cuda:0"
POISSON = 0.3
STEEL = 210e9
DENSITY = 7850.0
# Refined solves are carried to the accuracy of the FP64 factor's own solutions, so that a reduced
# precision factor can stand in for it.
TARGET_BERR = 1e-14


def listed():
    return [
        # The smallest calls: a factor in hand, one load case from host memory and back (a load
        # step or a time step of a small model). Latency and launches.
        dict(name="solve_host_fp64_small", kind="solve", mesh="hex8", cells_x=8, cells_y=8, cells_z=8,
             precision="fp64", nrhs=1, host=True),
        # One load case of a large model on the device: every step of an implicit time
        # integration or of a Newton iteration with a kept factor.
        dict(name="solve_fp64_large", kind="solve", mesh="hex8", cells_x=36, cells_y=36, cells_z=36,
             precision="fp64", nrhs=1, host=False),
        # Several load cases at once on a medium model.
        dict(name="solve_fp64_8rhs", kind="solve", mesh="hex8", cells_x=20, cells_y=23, cells_z=17,
             precision="fp64", nrhs=8, host=False),
        # The plain FP64 static analysis of the 40 x 8 x 8 cantilever: new values into the
        # analysed pattern, factor, solve.
        dict(name="static_fp64_cantilever", kind="static", mesh="hex8", cells_x=40, cells_y=8, cells_z=8,
             precision="fp64"),
        # The same on the 28^3 cube (70 644 equations), where the matrix cores count.
        dict(name="static_fp64_cube28", kind="static", mesh="hex8", cells_x=28, cells_y=28, cells_z=28,
             precision="fp64"),
        # The mixed-precision form with refinement, 40^3 cube (201 720 equations).
        dict(name="static_mixed_cube40", kind="static", mesh="hex8", cells_x=40, cells_y=40, cells_z=40,
             precision="mixed"),
        # A batch of independent hex8 and tet10 models of uneven size, factored in FP32 and solved
        # for many load cases with per-model refinement (a design study).
        dict(name="batch_fp32_8x64", kind="batch", models=8, first=4100, dofs_lo=2000, dofs_hi=12000, nrhs=64),
        # Shift-invert block solves: 16 vectors, the mixed factor of K - sigma M in hand.
        dict(name="shift_mixed_16vec", kind="shift", mesh="tet10", cells_x=13, cells_y=13, cells_z=13,
             precision="mixed", nrhs=16),
        # The stiffness matrix of a hex8 model with per-element moduli, assembled on the device.
        dict(name="assemble_hex8_k", kind="assemble", mesh="hex8", cells_x=40, cells_y=40, cells_z=40, what="K"),
        # K - sigma M of a tet10 model, the modal analysis's matrix.
        dict(name="assemble_tet10_shifted", kind="assemble", mesh="tet10", cells_x=14, cells_y=14, cells_z=14,
             what="shifted"),
        # The lowest modes of a tet10 block by the shifted block Lanczos method.
        dict(name="modes_tet10", kind="modes", mesh="tet10", cells_x=5, cells_y=7, cells_z=9, count=6),
        # LDL^T of an indefinite K - sigma M (a shift between modes) and one solve.
        dict(name="ldlt_tet10", kind="ldlt", mesh="tet10", cells_x=8, cells_y=8, cells_z=8, scalar="real"),
    ]


def _cells(rng, mesh, lo, hi):
    """Cells of a box of about lo..hi equations (log-uniform), sides within a factor of about 2."""
    per = 3.0 if mesh == "hex8" else 24.0
    n = math.exp(rng.uniform(math.log(lo), math.log(hi))) / per
    a = [rng.uniform(0.7, 1.4) for _ in range(3)]
    s = (n / (a[0] * a[1] * a[2])) ** (1.0 / 3.0)
    c = [max(2, round(s * v)) for v in a]
    while per * c[0] * c[1] * c[2] > hi:
        c[c.index(max(c))] -= 1
    return dict(mesh=mesh, cells_x=c[0], cells_y=c[1], cells_z=c[2])


def draw(rng):
    kind = rng.choice(["solve", "solve", "static", "static", "batch", "shift", "assemble", "modes", "ldlt"])
    mesh = rng.choice(["hex8", "tet10"])
    if kind == "solve":
        nrhs = rng.choice([1, 1, rng.randint(2, 8), rng.randint(9, 24)])
        return dict(kind=kind, precision=rng.choice(["fp64", "fp64", "fp32"]), nrhs=nrhs,
                    host=rng.random() < 0.3, **_cells(rng, mesh, 1500, 120000 if nrhs == 1 else 25000))
    if kind == "static":
        precision = rng.choice(["fp64", "mixed"])
        return dict(kind=kind, precision=precision,
                    **_cells(rng, mesh, 1500 if precision == "fp64" else 10000, 60000 if precision == "fp64" else 120000))
    if kind == "batch":
        return dict(kind=kind, models=rng.randint(2, 8), first=rng.randint(0, 10 ** 6), dofs_lo=2000,
                    dofs_hi=rng.randint(3000, 10000), nrhs=rng.randint(5, 64))
    if kind == "shift":
        return dict(kind=kind, precision=rng.choice(["mixed", "fp64"]), nrhs=rng.randint(4, 16),
                    **_cells(rng, "tet10", 3000, 50000))
    if kind == "assemble":
        if mesh == "hex8":
            return dict(kind=kind, what="K", **_cells(rng, mesh, 3000, 190000))
        return dict(kind=kind, what=rng.choice(["K", "M", "shifted"]), **_cells(rng, mesh, 2000, 60000))
    if kind == "modes":
        return dict(kind=kind, count=rng.randint(3, 6), **_cells(rng, "tet10", 2000, 6500))
    return dict(kind=kind, scalar=rng.choice(["real", "complex"]), **_cells(rng, "tet10", 1500, 9000))


# ------------------------------------------------------------------------------------------
# The meshes and matrices (host)

@functools.lru_cache(maxsize=6)
def _block(mesh, nx, ny, nz, jitter):
    """A box of unit-spaced (hex8) or 10 mm (tet10) cells, E = 210 GPa, z = 0 clamped."""
    h = 1.0 if mesh == "hex8" else 0.01
    size = (nx * h, ny * h, nz * h)
    return P.block(mesh, (nx, ny, nz), size, STEEL, POISSON, clamp_face=4, jitter=jitter, seed=11,
                   rho=DENSITY if mesh == "tet10" else 0.0)


@functools.lru_cache(maxsize=2)
def _models(count, first, lo, hi):
    return P.batch([P.random_model(first + q, lo, hi) for q in range(count)], nrhs=1)


def _problem(case):
    if case["kind"] == "batch":
        return _models(case["models"], case["first"], float(case["dofs_lo"]), float(case["dofs_hi"]))
    # modes of a symmetric block come in pairs and with free signs: its nodes are moved a little
    jitter = 0.1 if case["kind"] == "modes" else 0.0
    return _block(case["mesh"], case["cells_x"], case["cells_y"], case["cells_z"], jitter)


def _shift(case, p):
    """The spectral shift: (2 pi 50 Hz)^2 below the first mode, or for LDL^T a frequency at which
    some modes lie below it (mode frequencies go with 1 / the block's height)."""
    if case["kind"] == "ldlt":
        hz = 1250.0 / (0.01 * case["cells_z"])
        return (2 * math.pi * hz) ** 2
    return (2 * math.pi * 50.0) ** 2


def _values(case, p, seed):
    """The matrix's values by full rows for this seed, and its modulus scale(s)."""
    rng = np.random.default_rng([seed, 1])
    if case["kind"] == "batch":
        scale = rng.uniform(0.7, 1.3, case["models"])
        return p.kval * np.repeat(np.repeat(scale, np.diff(p.segments)), np.diff(p.ptr)), scale
    scale = rng.uniform(70e9, 210e9) / STEEL
    if case["kind"] in ("shift", "modes"):
        return scale * p.kval - _shift(case, p) * p.mval, scale
    if case["kind"] == "ldlt":
        scale = rng.uniform(0.95, 1.05)
        sigma = _shift(case, p)
        if case["scalar"] == "real":
            return scale * p.kval - sigma * p.mval, scale
        w = math.sqrt(sigma)
        return (scale * p.kval - sigma * p.mval) + 1j * w * (1e-6 * scale * p.kval + 10.0 * p.mval), scale
    return scale * p.kval, scale


def _loads(case, p, seed, nrhs):
    """Load cases: a uniform pressure on the top of a hex8 block and seeded body forces of its
    size, or seeded vectors (shift-invert, batches)."""
    rng = np.random.default_rng([seed, 2])
    f = rng.standard_normal((nrhs, p.n))
    if case["kind"] in ("solve", "static") and case["mesh"] == "hex8":
        fp = P.pressure_load(p)
        f = fp + f * (np.linalg.norm(fp) / math.sqrt(p.n))
    if case["kind"] == "ldlt" and case["scalar"] == "complex":
        f = f + 1j * rng.standard_normal((nrhs, p.n))
    return f


def _upper(p, vals):
    if np.iscomplexobj(vals):
        ptr, idx, re = p.upper(np.ascontiguousarray(vals.real))
        return ptr, idx, re + 1j * p.upper(np.ascontiguousarray(vals.imag))[2]
    return p.upper(vals)


def _young(case, p, seed):
    """Per-element moduli (a graded or sampled material)."""
    return np.random.default_rng([seed, 3]).uniform(70e9, 210e9, len(p.conn))


def prepare(case, seed):
    p = _problem(case)
    kind = case["kind"]
    s = dict(case=case, n=p.n)
    if kind == "assemble":
        uptr, uidx, _ = p.upper()
        s["assembly"] = AS.Assembly(p.kind, p.xyz, p.conn, _young(case, p, seed), POISSON, p.eq_dof, uptr, uidx,
                                    density=p.rho)
        s["shift"] = _shift(case, p) * (1.0 + (seed % 97) / 97.0)
        s["out"] = torch.empty(len(uidx), dtype=torch.float64, device=DEV)
        return s
    vals, _ = _values(case, p, seed)
    up = _upper(p, vals)
    sym = CH.Symbolic(CH.UpperColumns(p.n, up[0], up[1], up[2].real))
    if kind == "ldlt":
        s.update(symbolic=sym, values=up[2], b=_loads(case, p, seed, 1)[0])
        return s
    s["values"] = torch.from_numpy(up[2]).to(DEV)
    s["stream"] = torch.cuda.Stream(DEV)
    precision = case.get("precision", "fp32" if kind == "batch" else "fp64")
    torch.cuda.synchronize()
    s["factor"] = CH.Factor(sym, precision=precision, device_values=s["values"].data_ptr(),
                            stream=s["stream"].cuda_stream)
    if kind == "modes":
        s["mass"] = CH.Matrix(p.n, p.ptr, p.idx, p.mval)
        s["shift"] = _shift(case, p)
        return s
    nrhs = case.get("nrhs", 1)
    b = _loads(case, p, seed, nrhs)
    if case.get("host"):
        s["b"] = list(b)
        return s
    s["b"] = torch.from_numpy(b).to(DEV)
    s["x"] = torch.empty_like(s["b"])
    if kind in ("batch", "shift") or precision != "fp64" and kind == "static":
        s["matrix"] = CH.Matrix(p.n, p.ptr, p.idx, vals)
        if kind == "batch":
            s["matrix"].set_segments(p.segments)
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "assemble":
        s["assembly"].assemble_device(s["out"].data_ptr(), case["what"], s["shift"])
        return s["out"]
    if kind == "ldlt":
        make = CH.LdltFactor if case["scalar"] == "real" else CH.ZLdltFactor
        f = make(s["symbolic"], s["values"])
        x = f.solve(s["b"])
        return [x, f.two_by_two()] + ([list(f.inertia())] if case["scalar"] == "real" else [])
    f = s["factor"]
    if kind == "modes":
        f.refactor_device(s["values"].data_ptr())
        m = f.lanczos_device(s["mass"], s["shift"], case["count"], max_basis=300)
        return [m["values"], m["vectors"]]
    if kind in ("static", "batch"):
        f.refactor_device(s["values"].data_ptr())
    if case.get("host"):
        return f.solve(s["b"][0]) if len(s["b"]) == 1 else f.solve_many(s["b"])
    b, x = s["b"], s["x"]
    if "matrix" in s:
        if len(b) == 1:
            f.solve_refined_device(s["matrix"], b.data_ptr(), x.data_ptr(), target_berr=TARGET_BERR)
        else:
            f.solve_refined_many_device(s["matrix"], b.data_ptr(), x.data_ptr(), len(b), target_berr=TARGET_BERR)
        return x
    with torch.cuda.stream(s["stream"]):  # the factor's stream: the copy comes before the solve
        x.copy_(b)
    f.solve_device(x.data_ptr(), len(b))
    return x


@functools.lru_cache(maxsize=8)
def _info(key):
    case = dict(key)
    p = _problem(case)
    ptr, idx, _ = p.upper()
    return CH.Symbolic(CH.UpperColumns(p.n, ptr, idx, np.zeros(len(idx)))).info(), len(idx), p.nnz


def work(case):
    p = _problem(case)
    kind = case["kind"]
    if kind == "assemble":
        nnz = len(p.upper()[1])
        e, nn = p.conn.shape
        points = 8 if nn == 8 else 4
        flops = e * points * nn * (nn + 1) / 2 * 60.0 + (e * 64.0 * nn * nn * 3 if case["what"] != "K" else 0.0)
        return dict(bytes=8.0 * nnz + 24.0 * len(p.xyz) + 4.0 * e * nn + 8.0 * e, flops=flops)
    info, nnz, full = _info(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
    n, entries = p.n, info["entries"]
    nrhs = case.get("nrhs", 1)
    elem = 8.0 if case.get("precision", "fp32" if kind == "batch" else "fp64") == "fp64" else 4.0
    solve_b, solve_f = 16.0 * n * nrhs, 4.0 * entries * nrhs
    if kind in ("solve", "shift"):
        return dict(bytes=elem * entries + solve_b, flops=solve_f)
    if kind == "modes":
        return dict(bytes=8.0 * nnz + 8.0 * entries + 8.0 * n * case["count"],
                    flops=info["flops"] + 6 * case["count"] * (4.0 * entries + 2.0 * full))
    if kind == "ldlt":
        c = 2.0 if case["scalar"] == "complex" else 1.0
        return dict(bytes=c * (8.0 * nnz + 8.0 * entries + 16.0 * n), flops=c * c * info["flops"])
    return dict(bytes=8.0 * nnz + elem * entries + solve_b, flops=info["flops"] + solve_f)


# ------------------------------------------------------------------------------------------
# The same outputs in 64 bits, by plain torch

def _spmv(ptr, idx, val):
    """A function multiplying the matrix by full rows with an n x k block."""
    p, i, v = (torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for a in (ptr, idx, val))
    rows = torch.repeat_interleave(torch.arange(len(p) - 1, device=DEV), p[1:] - p[:-1])

    def mul(x):
        y = torch.zeros_like(x)
        for c in range(0, x.shape[1], 8):
            y[:, c:c + 8].index_add_(0, rows, v[:, None] * x[i, c:c + 8])
        return y

    return mul, v[i == rows]


def _spd_solve(ptr, idx, val, b):
    """Conjugate gradients with the diagonal as preconditioner on every column of b (n x k), then
    the same on the residual until it no longer shrinks."""
    mul, diag = _spmv(ptr, idx, val)
    x = torch.zeros_like(b)
    size = torch.linalg.norm(b, dim=0)
    for _ in range(4):
        r = b - mul(x)
        start = torch.linalg.norm(r, dim=0)
        if bool((start <= 1e-15 * size).all()):
            break
        d = torch.zeros_like(b)
        z = r / diag[:, None]
        q = z.clone()
        rz = (r * z).sum(0)
        for it in range(4000):
            aq = mul(q)
            den = (q * aq).sum(0)
            alpha = torch.where(den > 0, rz / den, torch.zeros_like(den))
            d += alpha * q
            r -= alpha * aq
            if it % 20 == 19 and bool((torch.linalg.norm(r, dim=0) <= 1e-9 * start).all()):
                break
            z = r / diag[:, None]
            rz2 = (r * z).sum(0)
            q = z + torch.where(rz > 0, rz2 / rz, torch.zeros_like(rz)) * q
            rz = rz2
        x += d
    return x


def _dense(p, vals):
    a = torch.zeros(p.n, p.n, dtype=torch.from_numpy(vals[:1]).dtype, device=DEV)
    rows = torch.from_numpy(np.repeat(np.arange(p.n), np.diff(p.ptr))).to(DEV)
    a[rows, torch.from_numpy(p.idx).to(DEV)] = torch.from_numpy(vals).to(DEV)
    return a


def _modes(case, p, scale):
    """The lowest modes above the shift: subspace iteration with the dense factor of K - sigma M."""
    sigma, count = _shift(case, p), case["count"]
    k, m = _dense(p, scale * p.kval), _dense(p, p.mval)
    chol = torch.linalg.cholesky(k - sigma * m)
    del k
    q = torch.from_numpy(np.random.default_rng(5).standard_normal((p.n, 4 * count + 16))).to(DEV)
    for _ in range(60):
        w = torch.cholesky_solve(m @ q, chol)
        for _ in range(2):  # M-orthonormal columns
            c = torch.linalg.cholesky((w.T @ (m @ w)).cpu()).to(DEV)
            w = torch.linalg.solve_triangular(c, w.T, upper=False).T
        mw = m @ w
        t = mw.T @ torch.cholesky_solve(mw, chol)
        theta, s = torch.linalg.eigh(0.5 * (t + t.T).cpu())
        q = w @ s.flip(1).to(DEV)
    vec = q[:, :count]
    at = vec.abs().argmax(0)
    vec = vec * torch.sign(vec[at, torch.arange(count, device=DEV)])
    return [(sigma + 1.0 / theta.flip(0)[:count]).numpy(), vec]


def _element_matrices(case, p, young):
    """Every element's stiffness (and mass per direction), elements x 3nn x 3nn (x nn x nn)."""
    x = torch.from_numpy(p.xyz[p.conn]).to(DEV)
    nn = p.conn.shape[1]
    if nn == 8:
        c = torch.tensor([[-1., -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1], [-1, -1, 1], [1, -1, 1], [1, 1, 1],
                          [-1, 1, 1]], dtype=torch.float64, device=DEV)
        points, weight = c / math.sqrt(3.0), 1.0

        def gradient(xi):
            f = 1.0 + xi * c
            return torch.stack([c[:, 0] * f[:, 1] * f[:, 2], c[:, 1] * f[:, 0] * f[:, 2],
                                c[:, 2] * f[:, 0] * f[:, 1]], 1) / 8.0
    else:
        a, b = (5.0 + 3.0 * math.sqrt(5.0)) / 20.0, (5.0 - math.sqrt(5.0)) / 20.0
        points = torch.full((4, 3), b, dtype=torch.float64, device=DEV)
        for q in range(3):
            points[q + 1, q] = a
        weight = 1.0 / 24.0
        dl = torch.tensor([[-1., -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1]], dtype=torch.float64, device=DEV)
        edges = [(0, 1), (1, 2), (2, 0), (0, 3), (1, 3), (2, 3)]

        def gradient(xi):
            l = torch.cat([(1.0 - xi.sum())[None], xi])
            corner = (4.0 * l - 1.0)[:, None] * dl
            return torch.cat([corner, torch.stack([4.0 * (dl[i] * l[j] + l[i] * dl[j]) for i, j in edges])])
    e = torch.from_numpy(young).to(DEV)
    lam = e * POISSON / ((1 + POISSON) * (1 - 2 * POISSON))
    mu = e / (2 * (1 + POISSON))
    ke = torch.zeros(len(e), nn, 3, nn, 3, dtype=torch.float64, device=DEV)
    eye = torch.eye(3, dtype=torch.float64, device=DEV)
    for xi in points:
        dn = gradient(xi)
        j = (dn.T[None, :, :, None] * x[:, None]).sum(2)  # J[a][b] = sum_i dN_i/dxi_a x_ib
        det = torch.linalg.det(j)
        g = (torch.linalg.inv(j)[:, None] * dn[None, :, None, :]).sum(3)  # dN_i/dx_b
        wd = weight * det
        gg = g[:, :, :, None, None] * g[:, None, None, :, :]  # g_ir g_jc
        dot = (g[:, :, None] * g[:, None]).sum(3)
        ke += (lam * wd)[:, None, None, None, None] * gg
        ke += (mu * wd)[:, None, None, None, None] * gg.permute(0, 1, 4, 3, 2)
        ke += (mu * wd)[:, None, None, None, None] * dot[:, :, None, :, None] * eye[None, None, :, None, :]
    me = None
    if nn == 10 and case["what"] != "K":
        # straight-edged tetrahedra: rho V times the integrals of products of quadratics
        poly = np.zeros((10, 10))  # shape functions over monomials l_i l_j (i <= j)
        mono = [(i, j) for i in range(4) for j in range(i, 4)]
        for i in range(4):  # l (2 l - 1) = l^2 - l sum_{j != i} l_j
            poly[i, mono.index((i, i))] = 1.0
            for q in range(4):
                if q != i:
                    poly[i, mono.index((min(i, q), max(i, q)))] = -1.0
        for q, (i, j) in enumerate([(0, 1), (1, 2), (2, 0), (0, 3), (1, 3), (2, 3)]):
            poly[4 + q, mono.index((min(i, j), max(i, j)))] = 4.0
        integ = np.zeros((10, 10))
        for r, (i, j) in enumerate(mono):
            for c, (k, l) in enumerate(mono):
                pw = [(i, j, k, l).count(t) for t in range(4)]
                integ[r, c] = math.prod(math.factorial(t) for t in pw) * 6.0 / math.factorial(7)
        ref = torch.from_numpy(poly @ integ @ poly.T).to(DEV)
        vol = torch.linalg.det(x[:, 1:4] - x[:, :1]) / 6.0
        me = DENSITY * vol[:, None, None] * ref
    return ke.reshape(len(e), 3 * nn, 3 * nn), me


def _assembled(case, p, seed):
    ke, me = _element_matrices(case, p, _young(case, p, seed))
    shift = _shift(case, p) * (1.0 + (seed % 97) / 97.0)
    if case["what"] != "K":
        full = torch.zeros_like(ke).reshape(len(ke), me.shape[1], 3, me.shape[1], 3)
        for c in range(3):
            full[:, :, c, :, c] = me
        full = full.reshape(ke.shape)
        ke = full if case["what"] == "M" else ke - shift * full
    uptr, uidx, _ = p.upper()
    eq = torch.full((3 * len(p.xyz),), -1, dtype=torch.int64, device=DEV)
    eq[torch.from_numpy(p.eq_dof).to(DEV)] = torch.arange(p.n, device=DEV)
    conn = torch.from_numpy(p.conn).to(DEV)
    dof = eq[(3 * conn[:, :, None] + torch.arange(3, device=DEV)).reshape(len(conn), -1)]
    r, c = dof[:, :, None].expand(ke.shape), dof[:, None, :].expand(ke.shape)
    keep = (r >= 0) & (c >= 0) & (r <= c)
    key = torch.from_numpy(np.repeat(np.arange(p.n), np.diff(uptr)) * p.n + uidx).to(DEV)
    out = torch.zeros(len(uidx), dtype=torch.float64, device=DEV)
    out.index_add_(0, torch.searchsorted(key, (c * p.n + r)[keep]), ke[keep])
    return out


def exact(case, seed):
    p = _problem(case)
    kind = case["kind"]
    if kind == "assemble":
        return _assembled(case, p, seed)
    vals, scale = _values(case, p, seed)
    if kind == "modes":
        return _modes(case, p, scale)
    if kind == "ldlt":
        b = torch.from_numpy(_loads(case, p, seed, 1)[0]).to(DEV)
        a = _dense(p, vals)
        lu, piv = torch.linalg.lu_factor(a)
        x = torch.linalg.lu_solve(lu, piv, b[:, None])
        for _ in range(3):
            x = x + torch.linalg.lu_solve(lu, piv, b[:, None] - a @ x)
        return [x[:, 0].cpu().numpy(), None] + ([[None, None]] if case["scalar"] == "real" else [])
    b = _loads(case, p, seed, case.get("nrhs", 1))
    x = _spd_solve(p.ptr, p.idx, vals, torch.from_numpy(b).to(DEV).T.contiguous()).T.contiguous()
    if case.get("host"):
        x = list(x.cpu().numpy())
        return x[0] if len(x) == 1 else x
    return x

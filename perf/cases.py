"""The work that users of tatva_amd have it do, as measurable cases.

Each case is one call (or one short chain of calls) through the package's
public entry points:

* ``map``       gradients at the quadrature points, the density there, and its
                integral: ``op.integrate(psi(op.grad(u)))`` written out
* ``gradient``  energy and residual of a state: ``E(u)`` and ``E.grad(u)``
* ``hvp``       the matrix-free product ``E.hvp(u, v)`` in FP32 or FP64
* ``jvp``       ``jvp(E_red.grad, (u,), (v,))`` on the free dofs of a lifter
* ``hessian``   ``sparse.linearized_jacfwd``: residual and colored Hessian (CSR)
* ``newton``    a whole ``solvers.Newton.solve`` (FP64 CSR or mixed precision)
* ``serve``     a burst of solve requests through ``serve.Server``

``prepare`` builds what a program keeps between calls (mesh on the device,
energy, lifter, colored pattern, solver, server) and the inputs of one call;
``run`` makes the call; ``exact`` is the same result from torch in 64 bits.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import tatva_amd as ta
from tatva_amd import energies, lifter, serve, solvers, sparse

DEV = "cuda"


def listed():
    return [
        # the smallest call: the 64 x 64 Poisson square of the README, where
        # launches and host work are all there is
        dict(name="poisson_tri3_gradient", kind="gradient", element="tri3", density="poisson",
             nx=64, ny=64, nz=0, jitter=0.0),
        # the 2-D colored Hessian of the reference's benchmark (200 x 200)
        dict(name="elastic_tri3_hessian", kind="hessian", element="tri3", density="elastic",
             nx=200, ny=200, nz=0, jitter=0.0),
        # a whole small solve: assembly, colored Hessian and PCG to convergence
        dict(name="poisson_tri3_newton", kind="newton", mode="csr", element="tri3",
             density="poisson", nx=64, ny=64, nz=0, jitter=0.0),
        # post-processing of a state (strain and energy density fields), a ragged box
        dict(name="neohooke_hex8_map", kind="map", element="hex8", density="neohooke",
             nx=64, ny=61, nz=67, jitter=0.0),
        # the FP64 residual of Newton and line searches on a distorted mesh
        dict(name="neohooke_hex8_gradient", kind="gradient", element="hex8", density="neohooke",
             nx=80, ny=80, nz=80, jitter=0.15),
        # the product inside the mixed-precision solve at the benchmark's size
        dict(name="neohooke_hex8_hvp_f32", kind="hvp", dtype="f32", element="hex8",
             density="neohooke", nx=160, ny=160, nz=160, jitter=0.0),
        # the same on tetrahedra with jittered nodes
        dict(name="neohooke_tet4_hvp_f32", kind="hvp", dtype="f32", element="tet4",
             density="neohooke", nx=72, ny=72, nz=72, jitter=0.2),
        # FP64 linearisation on the free dofs, two materials in one mesh
        dict(name="elastic_hex8_jvp", kind="jvp", element="hex8", density="elastic",
             materials=2, nx=48, ny=47, nz=49, jitter=0.0),
        # the FP64 path's matrix: residual and colored Hessian on the free dofs
        dict(name="elastic_hex8_hessian", kind="hessian", element="hex8", density="elastic",
             nx=64, ny=64, nz=64, jitter=0.0),
        # the FP64 Newton solve: Hessian and node-block PCG
        dict(name="elastic_hex8_newton", kind="newton", mode="csr", element="hex8",
             density="elastic", nx=48, ny=48, nz=48, jitter=0.0),
        # one load step of the mixed-precision Newton solve
        dict(name="neohooke_hex8_newton", kind="newton", mode="mixed", element="hex8",
             density="neohooke", nx=40, ny=40, nz=40, jitter=0.0),
        # a burst of solve requests of mixed sizes and materials
        dict(name="serve_burst", kind="serve", sizes="8 11 17 24 31 40"),
    ]


def draw(rng):
    """A case of the same ranges: sizes spread over the logarithm of the element
    count, boxes with sides of their own, every element and density."""
    kind = rng.choice(["map", "gradient", "hvp", "hvp", "jvp", "hessian", "hessian", "newton",
                       "newton", "serve"])
    if kind == "serve":
        return dict(kind=kind, sizes=" ".join(
            str(round(math.exp(rng.uniform(math.log(8), math.log(40))))) for _ in range(5)))
    element = rng.choice(["tri3", "tet4", "hex8", "hex8"])
    density = rng.choice(["elastic", "neohooke"])
    mode = rng.choice(["csr", "mixed"]) if kind == "newton" else None
    if element == "tri3" and (kind == "newton" or rng.random() < 0.5):
        density, mode = "poisson", ("csr" if kind == "newton" else None)
    # elements at most, by what a pass of the kind costs
    most = {"map": 3e5, "gradient": 5e5, "hvp": 1.2e6, "jvp": 4e5, "hessian": 1.2e5,
            "newton": 3e4}[kind]
    count = math.exp(rng.uniform(math.log(500.0), math.log(most)))
    d = 2 if element == "tri3" else 3
    side = (count / {"tri3": 2, "tet4": 6, "hex8": 1}[element]) ** (1.0 / d)
    n = [max(3, round(side * math.exp(rng.uniform(-0.25, 0.25)))) for _ in range(d)]
    case = dict(kind=kind, element=element, density=density, nx=n[0], ny=n[1],
                nz=n[2] if d == 3 else 0,
                jitter=rng.choice([0.0, 0.15]) if d == 3 else 0.0)
    if mode:
        case["mode"] = mode
    if kind == "hvp":
        case["dtype"] = rng.choice(["f32", "f32", "f64"])
    if kind in ("jvp", "gradient", "hvp") and density != "poisson":
        case["materials"] = rng.choice([1, 1, 2])
    return case


# ------------------------------------------------------------- the problem ----

ELEMENTS = {"tri3": ta.Tri3, "tet4": ta.Tetrahedron4, "hex8": ta.Hexahedron8}


def _mesh(case, seed):
    if case["element"] == "tri3":
        return ta.Mesh.unit_square(case["nx"], case["ny"])
    kind = "hexahedron" if case["element"] == "hex8" else "tetrahedron"
    return ta.Mesh.box((case["nx"], case["ny"], case["nz"]), type=kind, jitter=case["jitter"],
                       seed=seed)


def _inputs(case, seed):
    """Plain arrays of one problem, from the seed: mesh, material parameters,
    loads, constrained dofs and their values, state and tangent."""
    mesh = _mesh(case, seed)
    X = torch.as_tensor(mesh.coords, device=DEV)
    N, d = X.shape
    nc = 1 if case["density"] == "poisson" else d
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = np.random.default_rng(seed)
    h = 1.0 / max(case["nx"], case["ny"], case["nz"])
    # a smooth field with a little noise on the scale of an element
    k = torch.as_tensor(r.uniform(0.5, 2.0, (nc, d)), device=DEV)
    phase = torch.as_tensor(r.uniform(0.0, 2 * math.pi, nc), device=DEV)
    noise = torch.randn((N, nc), generator=g, device=DEV, dtype=torch.float64)
    u = 0.02 * torch.sin(math.pi * X @ k.T + phase) + 0.01 * h * noise
    v = torch.randn((N, nc), generator=g, device=DEV, dtype=torch.float64)
    E = mesh.n_elements
    if case["density"] == "poisson":
        params = (float(r.uniform(0.5, 1.5)),)
    elif case.get("materials", 1) == 2:
        soft = mesh.coords[mesh.elements].mean(axis=1)[:, 0] < 0.5
        a, b = r.uniform(0.3, 0.6, 2), r.uniform(1.0, 3.0, 2)
        params = (np.where(soft, a[0], b[0]), np.where(soft, a[1], b[1]))
    elif case["density"] == "elastic":
        params = serve.lame(float(r.lognormal(0.0, 0.5)), float(r.uniform(0.2, 0.4)))
    else:
        params = (float(r.uniform(0.8, 1.2)), float(r.uniform(5.0, 10.0)))
    x = mesh.coords[:, 0]
    x0, x1 = np.where(np.isclose(x, 0.0))[0], np.where(np.isclose(x, 1.0))[0]
    f = None
    if case["density"] == "poisson":
        c = mesh.coords
        fixed = np.where(np.isclose(c, 0.0).any(1) | np.isclose(c, 1.0).any(1))[0]
        values = np.zeros(fixed.size)
    else:
        fixed = (x0[:, None] * d + np.arange(d)).ravel()
        values = np.zeros(fixed.size)
        if case["density"] == "neohooke" and case["kind"] == "newton":
            # x = 1 is pulled out, starting from the homogeneous stretch
            s = float(r.uniform(0.02, 0.04))
            fixed, values = np.r_[fixed, x1 * d], np.r_[values, np.full(x1.size, s)]
            u = torch.zeros_like(u)
            u[:, 0] = s * X[:, 0]
        else:
            # a dead load on x = 1
            f = np.zeros(N * d)
            f[x1 * d] = float(r.uniform(0.5, 1.5)) * 1e-3 / max(1, x1.size)
    if case["kind"] == "newton" and case["density"] != "neohooke":
        u = torch.zeros_like(u)
    return dict(mesh=mesh, X=X, nc=nc, params=params, E=E, f=f, fixed=fixed, values=values,
                u=u.reshape(-1), v=v.reshape(-1))


def _requests(case, seed):
    r = np.random.default_rng(seed)
    out = []
    for i, n in enumerate(int(s) for s in case["sizes"].split()):
        nh = i % 2 == 1
        out.append(serve.SolveRequest(
            rid=i, n=n, material="neo_hookean" if nh else "linear_elastic",
            E=float(r.lognormal(0.0, 0.5)), nu=float(r.uniform(0.2, 0.45)),
            load_steps=2 if nh else 1, stretch=float(r.uniform(0.02, 0.03)),
            traction=float(r.uniform(0.5, 1.5)) * 1e-3))
    return out


def prepare(case, seed):
    if case["kind"] == "serve":
        return dict(kind="serve", server=serve.Server(keep_solutions=True, tol=1e-11),
                    requests=_requests(case, seed))
    P = _inputs(case, seed)
    op = ta.Operator(P["mesh"], ELEMENTS[case["element"]]())
    op.device_layout()  # the mesh goes to the device
    dens = {"poisson": energies.Poisson, "elastic": energies.LinearElasticity,
            "neohooke": energies.NeoHookean}[case["density"]](*P["params"])
    s = dict(kind=case["kind"], op=op, dens=dens, u=P["u"], v=P["v"])
    if case["kind"] == "map":
        s["u"] = P["u"].reshape(-1) if P["nc"] == 1 else P["u"].reshape(-1, P["nc"])
        return s
    E = s["E"] = op.energy(dens, external_force=P["f"])
    if case["kind"] == "hvp":
        dt = torch.float32 if case["dtype"] == "f32" else torch.float64
        s["u"], s["v"] = P["u"].to(dt), P["v"].to(dt)
    if case["kind"] in ("hvp", "gradient"):
        return s
    L = lifter.Lifter(E.size, lifter.Fixed(P["fixed"], P["values"]))
    red = s["red"] = E.reduced(L)
    if case["kind"] in ("jvp", "hessian"):
        free = torch.as_tensor(L.free_dofs, device=DEV)
        s["u"], s["v"] = P["u"][free], P["v"][free]
    if case["kind"] == "hessian":
        cm = sparse.ColoredMatrix.from_csr(L.adapt_sparsity(
            sparse.pattern_from_mesh(P["mesh"], P["nc"])))
        s["jac"] = sparse.linearized_jacfwd(red.grad, cm)
    if case["kind"] == "newton":
        tight = dict(tol=1e-10, lin_tol=1e-12) if case["mode"] == "csr" else dict(tol=1e-11)
        s["solver"] = solvers.Newton(E, L, mode=case["mode"], **tight)
    return s


def run(s):
    kind = s["kind"]
    if kind == "map":
        op, dens, u = s["op"], s["dens"], s["u"]
        g = op.grad(u)
        psi = dens(g, values=op.eval(u)) if dens.needs_values else dens(g)
        return {"grad": g, "psi": psi, "total": op.integrate(psi)}
    if kind == "gradient":
        return {"energy": s["E"](s["u"]), "residual": s["E"].grad(s["u"])}
    if kind == "hvp":
        return {"hv": s["E"].hvp(s["u"], s["v"])}
    if kind == "jvp":
        r, hv = ta.jvp(s["red"].grad, (s["u"],), (s["v"],))
        return {"residual": r, "hv": hv}
    if kind == "hessian":
        r, K = s["jac"](s["u"])
        return {"residual": r, "data": K.data}
    if kind == "newton":
        u = s["u"].clone()
        s["solver"].solve(u)
        return {"u": u}
    report = s["server"].run(s["requests"], realtime=False)
    return {"u": [r.u for r in report.results]}


# -------------------------------------------------------------------- work ----


def _sizes(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["element"] == "tri3":
        E, N, nne, d, Q = 2 * nx * ny, (nx + 1) * (ny + 1), 3, 2, 1
    else:
        E, N, d = nx * ny * nz, (nx + 1) * (ny + 1) * (nz + 1), 3
        nne, Q = (8, 8) if case["element"] == "hex8" else (4, 1)
        E *= 6 if case["element"] == "tet4" else 1
    return E, N, nne, d, Q, 1 if case["density"] == "poisson" else d


def _row_blocks(case):
    """Nodes coupled to a node, inside the mesh."""
    return {"tri3": 7, "tet4": 15, "hex8": 27}[case["element"]]


def work(case):
    """Bytes of inputs read once and outputs written once, and the operations of
    the element loop: geometry, gradients, the density and its derivatives."""
    if case["kind"] == "serve":
        total = {"bytes": 0.0, "flops": 0.0}
        for i, n in enumerate(int(s) for s in case["sizes"].split()):
            c = dict(kind="newton", mode="mixed", element="hex8", nx=n, ny=n, nz=n, jitter=0.0,
                     density="neohooke" if i % 2 else "elastic")
            w = work(c)
            for k in total:
                total[k] += w[k] * (2 if i % 2 else 1)
        return total
    E, N, nne, d, Q, nc = _sizes(case)
    mesh = 4.0 * nne * E + 8.0 * d * N
    vec = 8.0 * nc * N
    geometry = Q * (2 * nne * d * d + 14 * d + 2 * nne * d * d)
    field = Q * 2 * nne * nc * d          # gradients of one field, or B^T S
    density = Q * (6 * d * d + 30)
    kind = case["kind"]
    if kind == "map":
        return {"bytes": mesh + vec + 8.0 * E * Q * (nc * d + 1) + 8.0,
                "flops": E * (geometry + field + density)}
    gradient = {"bytes": mesh + 2 * vec + (vec if case["density"] == "elastic" else 0.0),
                "flops": E * (geometry + 2 * field + density)}
    if kind == "gradient":
        return gradient
    hvp_flops = E * (geometry + 3 * field + density + Q * 6 * d ** 3)
    if kind == "hvp":
        size = 0.5 if case["dtype"] == "f32" else 1.0
        return {"bytes": mesh + 3 * vec * size, "flops": hvp_flops}
    if kind == "jvp":
        return {"bytes": mesh + 4 * vec, "flops": gradient["flops"] + hvp_flops}
    nnz = float(N) * _row_blocks(case) * nc * nc
    hessian = {"bytes": mesh + 2 * vec + 12.0 * nnz,
               "flops": E * (geometry + field + density + Q * (nne * nc) ** 2 * 2 * d)}
    if kind == "hessian":
        return hessian
    n = max(case["nx"], case["ny"], case["nz"])
    if case["mode"] == "csr":
        steps = 1 if case["density"] != "neohooke" else 4
        its = steps * n * (2.2 if nc == 1 else 9.0)
        return {"bytes": steps * (hessian["bytes"] + gradient["bytes"])
                + its * (8.0 * nnz + 4.0 * nnz / (nc * nc) + 11 * vec),
                "flops": steps * (hessian["flops"] + gradient["flops"]) + its * (2 * nnz + 14 * N)}
    steps = 5
    its = steps * n * 5.0
    return {"bytes": steps * gradient["bytes"] + its * (mesh / 2 + 7 * vec),
            "flops": steps * gradient["flops"] + its * hvp_flops}


# ------------------------------------------------------------ 64-bit values ----


def _shape(element):
    """(N (Q, nne), dN/dxi (Q, nne, d), weights) of the default quadrature."""
    if element != "hex8":
        d = 2 if element == "tri3" else 3
        dn = torch.cat([-torch.ones(1, d), torch.eye(d)]).double().to(DEV)
        N = torch.full((1, d + 1), 1.0 / (d + 1), dtype=torch.float64, device=DEV)
        return N, dn[None], torch.tensor([1.0 / math.factorial(d)], dtype=torch.float64, device=DEV)
    s = torch.tensor([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1],
                      [-1, -1, 1], [1, -1, 1], [1, 1, 1], [-1, 1, 1]],
                     dtype=torch.float64, device=DEV)
    f = 1.0 + (s / math.sqrt(3.0))[:, None, :] * s[None]        # (Q, nne, 3)
    dn = torch.stack([s[None, :, i] * f[..., (i + 1) % 3] * f[..., (i + 2) % 3]
                      for i in range(3)], -1) / 8
    return f.prod(-1) / 8, dn, torch.ones(8, dtype=torch.float64, device=DEV)


class _Exact:
    """Energy, gradient and Hessian products by autograd, in chunks of elements."""

    def __init__(self, case, P, chunk=1 << 18):
        self.case, self.P = case, P
        self.conn = torch.as_tensor(P["mesh"].elements, device=DEV).long()
        self.N, self.dn, self.w = _shape(case["element"])
        self.f = None if P["f"] is None else torch.as_tensor(P["f"], device=DEV)
        self.params = [torch.as_tensor(p, device=DEV, dtype=torch.float64) for p in P["params"]]
        self.parts = [slice(i, min(i + chunk, P["E"])) for i in range(0, P["E"], chunk)]

    def geometry(self, part):
        J = torch.einsum("qak,eaj->eqkj", self.dn, self.P["X"][self.conn[part]])
        B = torch.einsum("eqjk,qak->eqaj", torch.linalg.inv(J), self.dn)
        return B, torch.linalg.det(J) * self.w

    def gather(self, u, part):
        return u.reshape(-1, self.P["nc"])[self.conn[part]]

    def psi(self, G, uq, part):
        p = [x if x.ndim == 0 else x[part][:, None] for x in self.params]
        if self.case["density"] == "poisson":
            return 0.5 * (G * G).sum((-1, -2)) - p[0] * uq[..., 0]
        if self.case["density"] == "elastic":
            e = 0.5 * (G + G.transpose(-1, -2))
            tr = e.diagonal(dim1=-2, dim2=-1).sum(-1)
            return p[0] * (e * e).sum((-1, -2)) + 0.5 * p[1] * tr * tr
        d = G.shape[-1]
        F = G + torch.eye(d, dtype=G.dtype, device=G.device)
        J = torch.linalg.det(F)
        return 0.5 * p[0] * ((F * F).sum((-1, -2)) - d - 2 * J.log()) + 0.5 * p[1] * J.log() ** 2

    def fields(self, ue, part):
        B, w = self.geometry(part)
        G = torch.einsum("eqaj,eac->eqcj", B, ue)
        return G, self.psi(G, torch.einsum("qa,eac->eqc", self.N, ue), part), w

    def linearize(self, u):
        """energy, gradient, and v -> H v holding one graph per chunk."""
        e, r, graphs = 0.0, torch.zeros_like(u), []
        for part in self.parts:
            ue = self.gather(u, part).clone().requires_grad_()
            _, psi, w = self.fields(ue, part)
            total = (psi * w).sum()
            g, = torch.autograd.grad(total, ue, create_graph=True)
            e = e + total.detach()
            self.add(r, g.detach(), part)
            graphs.append((part, ue, g))
        if self.f is not None:
            e, r = e - self.f @ u, r - self.f

        def product(v):
            out = torch.zeros_like(u)
            for part, ue, g in graphs:
                h, = torch.autograd.grad(g, ue, self.gather(v, part), retain_graph=True)
                self.add(out, h, part)
            return out
        return e, r, product

    def add(self, out, values, part):
        nc = self.P["nc"]
        out.view(-1, nc).index_add_(0, self.conn[part].reshape(-1), values.reshape(-1, nc))


def _free(P):
    mask = torch.ones(P["u"].numel(), dtype=torch.bool, device=DEV)
    mask[torch.as_tensor(P["fixed"], device=DEV)] = False
    return mask


def _lifted(P, u):
    """The full state: free entries of u, the constraint values elsewhere."""
    u = u.clone()
    u[torch.as_tensor(P["fixed"], device=DEV)] = torch.as_tensor(P["values"], device=DEV)
    return u


def _hessian_data(case, P, product, mask):
    """Values of the sorted CSR pattern of coupled free dofs: one product per
    color of the structured mesh's nodes (three per direction)."""
    nc, N = P["nc"], P["X"].shape[0]
    conn = torch.as_tensor(P["mesh"].elements, device=DEV).long()
    pairs = torch.unique((conn[:, :, None] * N + conn[:, None, :]).reshape(-1))
    c = torch.arange(nc, device=DEV)
    rows = ((pairs // N)[:, None, None] * nc + c[:, None]).expand(-1, nc, nc).reshape(-1)
    cols = ((pairs % N)[:, None, None] * nc + c[None, :]).expand(-1, nc, nc).reshape(-1)
    keep = mask[rows] & mask[cols]
    rows, cols = rows[keep], cols[keep]
    order = torch.argsort(rows * (N * nc) + cols)
    rows, cols = rows[order], cols[order]
    node = torch.arange(N, device=DEV)
    if case["element"] == "tri3":
        color = node // (case["ny"] + 1) % 3 * 3 + node % (case["ny"] + 1) % 3
    else:
        sx, sy = case["nx"] + 1, case["ny"] + 1
        color = (node % sx % 3 * 3 + node // sx % sy % 3) * 3 + node // (sx * sy) % 3
    color = (color[:, None] * nc + c).reshape(-1)
    of = color[cols]
    data = torch.empty(rows.numel(), dtype=torch.float64, device=DEV)
    for k in range(int(color.max()) + 1):
        y = product(((color == k) & mask).double())
        at = torch.nonzero(of == k).reshape(-1)
        data[at] = y[rows[at]]
    return data


def _newton(ref, P, mask):
    """Newton with conjugate gradients to the rounding of 64 bits."""
    u, first = _lifted(P, P["u"]), None
    for _ in range(14):
        _, r, product = ref.linearize(u)
        r = torch.where(mask, r, 0.0)
        rr = float(r @ r)
        first = rr if first is None else first
        if rr <= 1e-26 * first:
            break
        x, p = torch.zeros_like(r), -r
        res, gamma, stop = -r, rr, 1e-10 * rr
        while gamma > stop:
            Ap = torch.where(mask, product(p), 0.0)
            a = gamma / float(p @ Ap)
            x += a * p
            res = res - a * Ap
            new = float(res @ res)
            p = res + (new / gamma) * p
            gamma = new
        u = u + x
    return u


def exact(case, seed):
    if case["kind"] == "serve":
        return None
    P = _inputs(case, seed)
    ref = _Exact(case, P)
    kind = case["kind"]
    if kind == "map":
        G, psi, total = [], [], 0.0
        for part in ref.parts:
            g, p, w = ref.fields(ref.gather(P["u"], part), part)
            G.append(g)
            psi.append(p)
            total = total + (p * w).sum()
        G = torch.cat(G)
        return {"grad": G[..., 0, :] if P["nc"] == 1 else G, "psi": torch.cat(psi), "total": total}
    if kind == "hvp":
        dt = torch.float32 if case["dtype"] == "f32" else torch.float64
        u, v = P["u"].to(dt).double(), P["v"].to(dt).double()
        whole, hv = ref.parts, torch.zeros_like(u)
        for part in whole:  # one chunk's graph at a time
            ref.parts = [part]
            hv += ref.linearize(u)[2](v)
        return {"hv": hv}
    mask = _free(P)
    if kind == "gradient":
        e, r, _ = ref.linearize(P["u"])
        return {"energy": e, "residual": r}
    if kind == "newton":
        return {"u": _newton(ref, P, mask)}
    e, r, product = ref.linearize(_lifted(P, P["u"]))
    if kind == "jvp":
        return {"residual": r[mask], "hv": product(torch.where(mask, P["v"], 0.0))[mask]}
    return {"residual": r[mask], "data": _hessian_data(case, P, product, mask)}

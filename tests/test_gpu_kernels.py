"""GPU kernels at the sizes where their work splits: tile and lane remainders,
quadrature rules of other lengths, nodes shared by many elements, patterns with
many colors.  Each against the FP64 oracle; FP64 results to 1e-12 relative to
the largest entry (summation order and cofactor inverses, as the parity tests)."""

import numpy as np
import pytest
import scipy.sparse as sps

import tatva_amd as ta
from oracle import fem
from tatva_amd import energies, lifter, sparse

pytestmark = pytest.mark.gpu

RTOL = 1e-12
ORACLE_EL = {ta.Tri3: fem.Tri3, ta.Tetrahedron4: fem.Tet4, ta.Hexahedron8: fem.Hex8}


def to_np(t):
    return t.detach().cpu().numpy()


def rel_err(a, b):
    a, b = np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64)
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


def gauss(points_1d, dim=3):
    x, w = np.polynomial.legendre.leggauss(points_1d)
    g = np.meshgrid(*[x] * dim, indexing="ij")
    h = np.meshgrid(*[w] * dim, indexing="ij")
    return np.stack([a.ravel() for a in g], -1), np.prod([a.ravel() for a in h], axis=0)


def fan(kind, k):
    """k elements around one node or axis: triangles around a center, tetrahedra
    around a center (a triangulated sphere of k caps, two rings), hexahedra
    around a vertical axis (two layers)."""
    t = 2 * np.pi * np.arange(k) / k
    if kind == "tri3":
        X = np.vstack([[0.0, 0.0], np.c_[np.cos(t), np.sin(t)]])
        i = np.arange(k)
        return ta.Mesh(X, np.c_[np.zeros(k, int), 1 + i, 1 + (i + 1) % k])
    if kind == "tet4":
        ring = np.c_[np.cos(t), np.sin(t), np.zeros(k)]
        X = np.vstack([[0.0, 0.0, 0.0], [0.1, 0.0, 0.9], [0.0, -0.1, -1.1], ring])
        i = np.arange(k)
        a, b, o = 3 + i, 3 + (i + 1) % k, np.zeros(k, int)
        return ta.Mesh(X, np.vstack([np.c_[o, a, b, o + 1], np.c_[o, b, a, o + 2]]))
    # k quads (center, two spokes and the corner between them), extruded twice
    r = np.vstack([[0.0, 0.0], np.c_[np.cos(t), np.sin(t)],
                   1.3 * np.c_[np.cos(t + np.pi / k), np.sin(t + np.pi / k)]])
    n = r.shape[0]
    X = np.vstack([np.c_[r * s, np.full(n, z)] for z, s in ((0.0, 1.0), (0.7, 1.1), (1.5, 0.9))])
    i = np.arange(k)
    quad = np.c_[np.zeros(k, int), 1 + i, 1 + k + i, 1 + (i + 1) % k]
    return ta.Mesh(X, np.vstack([np.c_[quad + l * n, quad + (l + 1) * n] for l in (0, 1)]))


def hessian_pair(mesh, el, density, od, colors=None, fixed=None):
    """Colored Hessian data on the GPU, and the oracle's element stiffness summed
    into the same pattern."""
    nc = density.ncomp(el.dim)
    n = mesh.n_nodes * nc
    rng = np.random.default_rng(7)
    u = 0.02 * rng.standard_normal(n)
    E = ta.Operator(mesh, el).energy(density)
    S = sparse.pattern_from_mesh(mesh, nc)
    prob = fem.Problem(ORACLE_EL[type(el)](el.quad_points, el.quad_weights), mesh.coords,
                       mesh.elements, od)
    fixed = np.zeros(0, int) if fixed is None else fixed
    L = lifter.Lifter(n, lifter.Fixed(fixed, 0.0))
    u[fixed] = 0.0
    cm = sparse.ColoredMatrix.from_csr(L.adapt_sparsity(S),
                                       None if colors is None else colors(L.size_reduced))
    E_red = E.reduced(L) if fixed.size else E
    K = sparse.jacfwd(E_red.grad, cm)(u[L.free_dofs] if fixed.size else u)
    dofs = (mesh.elements[:, :, None] * nc + np.arange(nc)).reshape(mesh.n_elements, -1)
    Ke = prob.element_stiffness(u).reshape(mesh.n_elements, dofs.shape[1], dofs.shape[1])
    pair = L.dof_map[np.stack(np.broadcast_arrays(dofs[:, :, None], dofs[:, None, :]))]
    keep = (pair >= 0).all(axis=0)
    ref = sps.coo_matrix((Ke[keep], (pair[0][keep], pair[1][keep])), shape=cm.shape).tocsr()
    ref.sort_indices()
    assert np.array_equal(ref.indices, K.to_csr().indices)
    return to_np(K.data), ref.data


LE, NH, PO = (energies.LinearElasticity(0.7, 1.3), energies.NeoHookean(0.7, 1.3),
              energies.Poisson(1.5))
ORACLE = {LE: fem.LinearElasticity(0.7, 1.3), NH: fem.NeoHookean(0.7, 1.3), PO: fem.Poisson(1.5)}


@pytest.mark.parametrize("density", [LE, NH, PO], ids=["le", "nh", "poisson"])
@pytest.mark.parametrize("kind,k", [("tri3", 3), ("tri3", 16), ("tri3", 17), ("tri3", 40),
                                    ("tet4", 3), ("tet4", 16), ("tet4", 17), ("tet4", 40),
                                    ("hex8", 3), ("hex8", 4), ("hex8", 5), ("hex8", 9)])
def test_hessian_rows_of_a_node_in_many_elements(kind, k, density):
    """Nodes in fewer, exactly and more elements than a node's lanes hold at a
    time (16 triangles, 32 tetrahedra, 8 hexahedra)."""
    el = {"tri3": ta.Tri3, "tet4": ta.Tetrahedron4, "hex8": ta.Hexahedron8}[kind]()
    got, ref = hessian_pair(fan(kind, k), el, density, ORACLE[density])
    assert rel_err(got, ref) < RTOL


@pytest.mark.parametrize("density", [LE, NH, PO], ids=["le", "nh", "poisson"])
@pytest.mark.parametrize("jitter", [0.0, 0.15])
@pytest.mark.parametrize("points", [1, 2, 3])
def test_hessian_rows_hex8_quadrature_rules(points, jitter, density):
    """1, 8 and 27 points over eight lanes; parallelepipeds and general elements;
    rows and columns of constrained dofs left out."""
    qp, qw = gauss(points)
    mesh = ta.Mesh.box((4, 3, 5), jitter=jitter, seed=2)
    nc = density.ncomp(3)
    fixed = np.r_[0:4 * nc, [11 * nc, 30 * nc + nc - 1]]
    got, ref = hessian_pair(mesh, ta.Hexahedron8(qp, qw), density, ORACLE[density], fixed=fixed)
    assert rel_err(got, ref) < RTOL


@pytest.mark.parametrize("kind,shape", [("tri3", (29, 30)), ("tet4", (8, 8, 7)), ("hex8", (8, 8, 7))])
def test_hessian_rows_of_many_colors(kind, shape):
    """Almost 2048 colors: one wave's rows fill the LDS (Hex8) or do not fit and
    the rows come from the element stiffness (Tri3, Tet4)."""
    if kind == "tri3":
        mesh, el = ta.Mesh.unit_square(*shape), ta.Tri3()
    elif kind == "tet4":
        mesh, el = ta.Mesh.box(shape, type="tetrahedron", jitter=0.1, seed=3), ta.Tetrahedron4()
    else:
        mesh, el = ta.Mesh.box(shape, jitter=0.1, seed=3), ta.Hexahedron8()
    assert 1800 < mesh.n_nodes * el.dim <= 2048
    got, ref = hessian_pair(mesh, el, LE, ORACLE[LE], colors=np.arange)
    assert rel_err(got, ref) < RTOL


def hex_variant(form, shape=(5, 7, 9)):
    """Hex8 meshes that take each geometry variant of the tile kernels: boxes
    along the axes, the same boxes with their local axes turned (parallelepipeds
    whose Jacobian is a permutation), sheared boxes, and boxes of which one is
    distorted (the whole mesh is general)."""
    m = ta.Mesh.box(shape, lengths=(1.0, 0.7, 1.9), origin=(-0.3, 0.1, 2.0))
    if form == "turned":
        return ta.Mesh(m.coords, m.elements[:, [1, 2, 3, 0, 5, 6, 7, 4]])
    if form == "sheared":
        return m.set_coords(m.coords @ np.array([[1.0, 0.2, 0.0], [0.0, 1.0, 0.1], [0.3, 0.0, 1.0]]))
    X = m.coords.copy()
    if form == "general":
        X[X.shape[0] // 2] += 0.01
    return m.set_coords(X)


@pytest.mark.parametrize("density", [LE, NH, PO], ids=["le", "nh", "poisson"])
@pytest.mark.parametrize("form", ["box", "turned", "sheared", "general"])
def test_hex8_geometry_variants(form, density):
    """Residual and product (FP64 to 1e-12; FP32 to 2e-6 of the largest entry: some
    tens of roundings of 6e-8) of every Hex8 geometry variant against the oracle."""
    import torch

    mesh = hex_variant(form)
    E = ta.Operator(mesh, ta.Hexahedron8()).energy(density)
    if form != "sheared":  # (rounding may leave a sheared box's bilinear modes nonzero)
        assert E.op.device_layout()["hex_affine"] == (form != "general")
    prob = fem.Problem(fem.Hex8(), mesh.coords, mesh.elements, ORACLE[density])
    rng = np.random.default_rng(5)
    u, v = 0.005 * rng.standard_normal(E.size), rng.standard_normal(E.size)
    assert rel_err(to_np(E.grad(u)), prob.residual(u)) < RTOL
    assert rel_err(to_np(E.hvp(u, v)), prob.hvp(u, v)) < RTOL
    u32, v32 = (torch.as_tensor(a, dtype=torch.float32, device="cuda") for a in (u, v))
    ref = prob.hvp(to_np(u32).astype(float), to_np(v32).astype(float))
    assert rel_err(to_np(E.hvp(u32, v32)), ref) < 2e-6


@pytest.mark.parametrize("full", [True, False])
@pytest.mark.parametrize("shape,density", [((6, 5, 4), LE), ((9, 7, 5), PO), ((82, 81, 80), PO),
                                           ((82, 81, 80), LE)],
                         ids=["le-small", "poisson-small", "poisson-folded", "le-folded"])
def test_matfree_pcg_step_by_nodes(shape, density, full):
    """Hex8 FP32 PCG whose step gathers the product by nodes: one and three
    components, full-length and reduced vectors, few and more than 2048 tiles
    (their shares folded first), deferred updates on and off (the same bits).
    Stopped at a recurrence residual of 1e-4; the true FP64 residual may differ
    from it by FP32 rounding over the iterations (some 1e2 of 6e-8 relative to
    b, so 2e-4 bounds the sum)."""
    import torch

    from tatva_amd import solvers

    mesh = ta.Mesh.box(shape)
    E = ta.Operator(mesh, ta.Hexahedron8()).energy(density)
    x0 = np.where(mesh.coords[:, 0] == 0.0)[0]
    nc = density.ncomp(3)
    L = lifter.Lifter(E.size, lifter.Fixed((x0[:, None] * nc + np.arange(nc)).ravel(), 0.0))
    red = E.reduced(L)
    u = torch.zeros(E.size, dtype=torch.float32, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(3)
    b = torch.randn(red.size, dtype=torch.float32, device="cuda", generator=g)
    out = []
    solvers.set_full_vectors(full)
    try:
        for defer in (True, False):
            solvers.set_deferred_update(defer)
            x, info = solvers.pcg_matfree(red, u, b, tol=1e-4)
            assert info.converged
            out.append((info.iterations, x))
    finally:
        solvers.set_deferred_update(True)   # the defaults
        solvers.set_full_vectors(True)
    assert out[0][0] == out[1][0] and torch.equal(out[0][1], out[1][1])
    r = b.double() - red.hvp_full_state(u.double(), out[0][1].double())
    assert float(r.norm() / b.double().norm()) < 2e-4


@pytest.mark.parametrize("nc", [1, 2, 3, 4])
@pytest.mark.parametrize("kind,points", [("tri3", 1), ("tri3", 3), ("tet4", 1), ("hex8", 1),
                                         ("hex8", 2), ("hex8", 3)])
@pytest.mark.parametrize("cells", [1, 2, 11])
def test_point_fields(cells, kind, points, nc):
    """Values and gradients at the points: elements that do not fill a wave and that
    spill into the next block, 1, 8 and 27 points over eight lanes, the components
    that are template parameters and one more."""
    rule = (None, None)
    if kind == "tri3":
        mesh, el = ta.Mesh.unit_square(cells, 3), ta.Tri3
        if points == 3:
            rule = np.array([[1 / 6, 1 / 6], [2 / 3, 1 / 6], [1 / 6, 2 / 3]]), np.full(3, 1 / 6)
    elif kind == "tet4":
        mesh, el = ta.Mesh.box((cells, 3, 5), type="tetrahedron", jitter=0.1), ta.Tetrahedron4
    else:
        mesh, el, rule = ta.Mesh.box((cells, 3, 5), jitter=0.1), ta.Hexahedron8, gauss(points)
    el = el(*rule)
    op = ta.Operator(mesh, el)
    oel = ORACLE_EL[type(el)](el.quad_points, el.quad_weights)
    u = np.random.default_rng(1).standard_normal((mesh.n_nodes, nc))
    assert rel_err(to_np(op.eval(u)), fem.op_eval(oel, mesh.coords, mesh.elements, u)) < RTOL
    assert rel_err(to_np(op.grad(u)), fem.op_grad(oel, mesh.coords, mesh.elements, u)) < RTOL


@pytest.mark.parametrize("density", [LE, NH, PO], ids=["le", "nh", "poisson"])
@pytest.mark.parametrize("points", [1, 2, 3])
@pytest.mark.parametrize("shape,jitter", [((1, 1, 1), 0.0), ((8, 8, 4), 0.0), ((257, 1, 1), 0.1),
                                          ((9, 7, 5), 0.1)])
def test_hex8_energy_by_tiles(shape, jitter, points, density):
    """One element, exactly a tile (256), one element more and a part-filled last
    tile; affine and general elements, other rules, the Poisson source.  Neo-Hookean
    energies are differences of terms of mu/2 (I1, 3, 2 ln J) over the unit volume, so
    rounding is relative to those; gradients stay near 0.1, short of inverted elements."""
    el = ta.Hexahedron8(*gauss(points))
    mesh = ta.Mesh.box(shape, jitter=jitter, seed=4)
    prob = fem.Problem(fem.Hex8(el.quad_points, el.quad_weights), mesh.coords, mesh.elements,
                       ORACLE[density])
    E = ta.Operator(mesh, el).energy(density)
    u = 0.05 / max(shape) * np.random.default_rng(2).uniform(-1, 1, E.size)
    ref = prob.energy(u)
    assert abs(float(E(u)) - ref) < RTOL * (abs(ref) + 1.5 * 0.7)


@pytest.mark.parametrize("density", [LE, NH, PO], ids=["le", "nh", "poisson"])
@pytest.mark.parametrize("form", ["box", "turned", "sheared", "general", "tet4"])
def test_stiffness_diagonal(form, density):
    """The closed forms against the oracle: FP64 to 1e-12, FP32 to 2e-6 of the largest
    entry (some tens of roundings of 6e-8, as the product)."""
    import torch

    if form == "tet4":
        mesh, el = ta.Mesh.box((5, 4, 7), type="tetrahedron", jitter=0.1), ta.Tetrahedron4
    else:
        mesh, el = hex_variant(form), ta.Hexahedron8
    E = ta.Operator(mesh, el()).energy(density)
    prob = fem.Problem(ORACLE_EL[el](), mesh.coords, mesh.elements, ORACLE[density])
    u = 0.005 * np.random.default_rng(5).standard_normal(E.size)
    assert rel_err(to_np(E.hessian_diag(u)), prob.hessian_diag(u)) < RTOL
    u32 = torch.as_tensor(u, dtype=torch.float32, device="cuda")
    ref = prob.hessian_diag(to_np(u32).astype(float))
    assert rel_err(to_np(E.hessian_diag(u32, dtype=torch.float32)), ref) < 2e-6


@pytest.mark.parametrize("longer", [False, True], ids=["short-rows", "a-longer-row"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1025, 4033, 4096, 4097])
def test_small_csr_pcg(n, longer):
    """Systems solved in one workgroup (at most 4096 rows of 8 entries on average), a
    row longer than the registers hold, and the first size past the limit; stopped by
    the tolerance (on a recurrence residual of 1e-12 of b; FP64 rounding over a few
    hundred iterations of a matrix of condition 1e3 stays far below 1e-9) and, more
    launches than one, by the iteration limit."""
    from tatva_amd import solvers

    rng = np.random.default_rng(n)
    A = sps.lil_matrix((n, n))
    for value, off in ((-1.0, 1), (-0.5, 2), (-0.25, 60)):
        if off < n:
            A += sps.diags([value], [off], shape=(n, n))
    A = A.tolil()
    if longer and n > 40:
        A[7, 12:38:2] = -0.03
    A = (A + A.T).tocsr()
    A = (A + sps.diags(np.asarray(-A.sum(axis=1)).ravel() + 0.003)).tocsr()
    A.sort_indices()
    K = sparse.ColoredMatrix.from_csr(A)
    b = rng.standard_normal(n)
    x, info = solvers.pcg(K, b, tol=1e-12)
    assert info.converged
    assert np.linalg.norm(b - A @ to_np(x)) < 1e-9 * np.linalg.norm(b)
    x0 = rng.standard_normal(n)
    x, info = solvers.pcg(K, A @ x0, x0=x0, tol=1e-12)
    assert info.iterations <= 1 and rel_err(to_np(x), x0) < 1e-9
    if n > 1000:
        x, info = solvers.pcg(K, b, tol=0.0, maxiter=300)
        assert not info.converged and info.iterations == 300
        assert np.isfinite(to_np(x)).all()


@pytest.mark.parametrize("case", ["none", "fixed", "values", "all", "periodic"])
def test_lift_in_one_pass_and_once_per_jvp(case):
    """lift_from_zeros against its definition (exact), with no, some and only
    constrained dofs; jvp and linearized_jacfwd, which lift once, against the separate
    calls (the same kernels on the same state: exact)."""
    mesh = ta.Mesh.unit_square(4, 3)
    n, rng = mesh.n_nodes, np.random.default_rng(0)
    left, right = (np.where(mesh.coords[:, 0] == x)[0] for x in (0.0, 1.0))
    ref = np.zeros(n)
    cons = {"none": [], "fixed": [lifter.Fixed(left, 0.5)],
            "values": [lifter.Fixed(left, np.arange(left.size) + 1.0)],
            "all": [lifter.Fixed(np.arange(n), 2.0)],
            "periodic": [lifter.Periodic(right, left)]}[case]
    L = lifter.Lifter(n, *cons)
    u = rng.standard_normal(L.size_reduced)
    ref[L.free_dofs] = u
    for c in cons:
        ref[c.dofs] = ref[left] if case == "periodic" else c.values
    assert np.array_equal(to_np(L.lift_from_zeros(u)), ref)
    if case in ("all", "periodic"):
        return
    red = ta.Operator(mesh, ta.Tri3()).energy(PO).reduced(L)
    v = rng.standard_normal(red.size)
    r, hv = ta.jvp(red.grad, (u,), (v,))
    assert np.array_equal(to_np(r), to_np(red.residual(u)))
    assert np.array_equal(to_np(hv), to_np(red.hvp(u, v)))
    cm = sparse.ColoredMatrix.from_csr(L.adapt_sparsity(sparse.pattern_from_mesh(mesh, 1)))
    r, K = sparse.linearized_jacfwd(red.grad, cm)(u)
    assert np.array_equal(to_np(r), to_np(red.residual(u)))
    assert np.array_equal(to_np(K.data), to_np(sparse.jacfwd(red.grad, cm)(u).data))


@pytest.mark.parametrize("points", [1, 2, 3])
@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 5, 9)])
def test_hex8_integrals(shape, points):
    """1, 8 and 27 points in chunks of eight: fields at the points and at the nodes,
    one component and three; sums of values of one sign, so relative to the result."""
    el = ta.Hexahedron8(*gauss(points))
    mesh = ta.Mesh.box(shape, jitter=0.1, seed=6)
    oel = fem.Hex8(el.quad_points, el.quad_weights)
    op = ta.Operator(mesh, el)
    rng = np.random.default_rng(3)
    for field in (rng.uniform(1, 2, (mesh.n_elements, points**3)),
                  rng.uniform(1, 2, (mesh.n_elements, points**3, 3)),
                  rng.uniform(1, 2, mesh.n_nodes), rng.uniform(1, 2, (mesh.n_nodes, 3))):
        if field.shape[0] == mesh.n_nodes and mesh.n_nodes == mesh.n_elements:
            continue
        ref = fem.integrate(oel, mesh.coords, mesh.elements, field)
        assert rel_err(to_np(op.integrate(field)), ref) < RTOL


@pytest.mark.parametrize("density", [LE, PO], ids=["le", "poisson"])
@pytest.mark.parametrize("form", ["box", "turned", "general"])
def test_hessian_rows_after_lds_of_nan(form, density):
    """A node's rows are zeroed in LDS by other lanes than those that add to them: on
    every geometry variant, right after kernels that leave NaN in the LDS, the rows
    equal the oracle's, and those of a second assembly bit for bit."""
    import torch

    mesh = hex_variant(form, (11, 9, 8))
    op = ta.Operator(mesh, ta.Hexahedron8())
    E = op.energy(density)
    cm = sparse.ColoredMatrix.from_csr(sparse.pattern_from_mesh(mesh, E.ncomp))
    J = sparse.jacfwd(E.grad, cm)
    nan = torch.full((E.size,), float("nan"), dtype=torch.float64, device="cuda")
    u = torch.zeros(E.size, dtype=torch.float64, device="cuda")
    data = []
    for _ in range(2):
        E.residual(nan)
        op.grad(nan.reshape(mesh.n_nodes, -1))
        data.append(to_np(J(u).data))
    assert np.array_equal(data[0], data[1])
    ref = hessian_pair(mesh, ta.Hexahedron8(), density, ORACLE[density])[1]
    assert rel_err(data[0], ref) < RTOL


def test_boxes_are_told_by_their_coordinates():
    """A Hex8 of equal edges whose corner line is one last place off has no linear or
    bilinear mode that is not rounded to zero, and is no box: two of its nodes across
    the body do not give its edge lengths.  One element, the corner line along x at
    y = z = 1 shifted; and meshes that are boxes, turned, sheared and general."""
    def hex_box(mesh):
        return ta.Operator(mesh, ta.Hexahedron8()).device_layout()["hex_box"]

    # lo + hi is an odd number of last places, a tie in the coarser sum: one place less
    # at both rounds to the same
    place = np.spacing(0.875)
    m = ta.Mesh.box((1, 1, 1), lengths=(0.0625, 1.0, 1.0), origin=(0.875, 0.0, 0.0))
    X = m.coords.copy()
    X[X[:, 0] > 0.9, 0] += place
    assert hex_box(m.set_coords(X)) == 1
    X[(X[:, 1] == 1.0) & (X[:, 2] == 1.0), 0] -= place
    v = X[:, 0][m.elements[0]][[0, 1, 3, 2, 4, 5, 7, 6]].reshape(2, 2, 2)  # z, y, x
    for axis in (2, 1, 0):
        v = np.stack([v.take(1, axis) + v.take(0, axis), v.take(1, axis) - v.take(0, axis)], axis)
    assert np.count_nonzero(v) == 2  # the sum and the x mode
    assert hex_box(m.set_coords(X)) == 0
    assert [hex_box(hex_variant(f)) for f in ("box", "turned", "sheared", "general")] == [1, 0, 0, 0]


@pytest.mark.parametrize("density", [LE, NH, PO], ids=["le", "nh", "poisson"])
@pytest.mark.parametrize("joined,elements", [(1, 255), (1, 256), (1, 700), (2, 512)])
def test_hex8_energy_of_separate_bodies(joined, elements, density):
    """Bodies of one or two elements: a tile of 256 elements has up to 2048 nodes, more
    than its LDS holds (1365 of three components).  Tolerance as test_hex8_energy_by_tiles."""
    body = ta.Mesh.box((joined, 1, 1), jitter=0.1, seed=7)
    k = elements // joined
    X = (body.coords + 3.0 * np.arange(k)[:, None, None] * [0, 0, 1]).reshape(-1, 3)
    conn = (body.elements + body.n_nodes * np.arange(k)[:, None, None]).reshape(-1, 8)
    mesh = ta.Mesh(X, conn)
    E = ta.Operator(mesh, ta.Hexahedron8()).energy(density)
    u = 0.02 * np.random.default_rng(3).uniform(-1, 1, E.size)
    ref = fem.Problem(fem.Hex8(), mesh.coords, mesh.elements, ORACLE[density]).energy(u)
    assert abs(float(E(u)) - ref) < RTOL * (abs(ref) + 1.5 * 0.7 * k)


@pytest.mark.parametrize("kind", ["hex8", "hex8-general", "tet4", "tri3"])
@pytest.mark.parametrize("density", [LE, NH, PO], ids=["le", "nh", "poisson"])
def test_hessian_takes_no_memory_that_it_does_not_use(kind, density):
    """No element-stiffness buffer where the rows come from the mesh; the stiffness of
    every element where the colors are too many (refused with a byte less) and in a
    Periodic call of the same assembler."""
    import ctypes

    import torch

    from tatva_amd import _native as nat

    if kind == "tri3":
        mesh, el = ta.Mesh.unit_square(9, 8), ta.Tri3()
    elif kind == "tet4":
        mesh, el = ta.Mesh.box((5, 4, 3), type="tetrahedron"), ta.Tetrahedron4()
    else:
        mesh, el = ta.Mesh.box((5, 4, 3), jitter=0.1 if kind == "hex8-general" else 0.0), ta.Hexahedron8()
    op = ta.Operator(mesh, el)
    E = op.energy(density)
    L, h, desc = nat.lib(), op.handle, E._desc
    full = L.tatva_colored_hessian_workspace(h, E.ncomp)
    assert full == mesh.n_elements * (mesh.elements.shape[1] * E.ncomp) ** 2 * 8
    needs = [L.tatva_colored_hessian_need(h, ctypes.byref(desc), c) for c in (1, 150, 2048)]
    assert needs[:2] == [0, 0] and needs[2] in (0, full)
    assert L.tatva_colored_hessian_need(h, ctypes.byref(desc), 0) == -1
    assert L.tatva_colored_hessian_need(h, ctypes.byref(desc), 2049) == -1

    cm = sparse.ColoredMatrix.from_csr(sparse.pattern_from_mesh(mesh, E.ncomp))
    u = torch.zeros(E.size, dtype=torch.float64, device="cuda")
    J = sparse.jacfwd(E.grad, cm)
    K = J(u)
    assert J.assembler.workspace(False).numel() == 0
    n_colors = 2048
    data = torch.empty(cm.nnz, dtype=torch.float64, device="cuda")
    ws = torch.empty(max(full, 1), dtype=torch.uint8, device="cuda")

    def call(nbytes):
        return L.tatva_colored_hessian(h, ctypes.byref(desc), u.data_ptr(), None, None, E.size,
                                       cm.colors.data_ptr(), n_colors, cm.indptr.data_ptr(),
                                       cm.indices.data_ptr(), cm.nnz, data.data_ptr(),
                                       ws.data_ptr() if nbytes else None, nbytes, nat.stream())

    assert call(needs[2]) == nat.OK
    assert rel_err(to_np(data), to_np(K.data)) < RTOL
    if needs[2]:
        assert call(needs[2] - 1) != nat.OK and call(0) != nat.OK
    assert J.assembler.workspace().numel() == full


@pytest.mark.parametrize("nc", [1, 2, 3])
@pytest.mark.parametrize("points", [1, 2, 3, 4, 5, 6, 7, 9])
def test_point_fields_of_rules_of_few_points(points, nc):
    """Hex8 rules on both sides of every line between the two kernels of values and
    gradients."""
    qp, qw = gauss(3)
    mesh, el = ta.Mesh.box((5, 7, 3), jitter=0.1), ta.Hexahedron8(qp[:points], qw[:points])
    op, oel = ta.Operator(mesh, el), fem.Hex8(el.quad_points, el.quad_weights)
    u = np.random.default_rng(1).standard_normal((mesh.n_nodes, nc))
    assert rel_err(to_np(op.eval(u)), fem.op_eval(oel, mesh.coords, mesh.elements, u)) < RTOL
    assert rel_err(to_np(op.grad(u)), fem.op_grad(oel, mesh.coords, mesh.elements, u)) < RTOL


def median_ms(call, runs=5, calls=20):
    import torch

    call()
    times = []
    for _ in range(runs):
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        start.record()
        for _ in range(calls):
            call()
        end.record()
        end.synchronize()
        times.append(start.elapsed_time(end))
    return np.median(times)


def test_gradients_at_one_point_cost_less_than_at_eight():
    """One point an element (an eighth of the output) took 0.59 of the time of eight on
    96^3 Hex8 when eight lanes shared an element whatever its rule; a thread an element
    takes 0.19, so half way is the limit.  Medians of five runs of twenty."""
    import torch

    mesh = ta.Mesh.box((96, 96, 96))
    u = torch.zeros(mesh.n_nodes, 3, dtype=torch.float64, device="cuda")
    times = []
    for points in (1, 2):
        op = ta.Operator(mesh, ta.Hexahedron8(*gauss(points)))
        times.append(median_ms(lambda op=op: op.grad(u)))
        op.close()
    assert times[0] < 0.39 * times[1]


def system_with_long_rows(n, entries, rows):
    """A diagonally dominant tridiagonal system with `entries` more in each of some rows
    (and columns)."""
    A = sps.diags([-1.0, 2.01, -1.0], [-1, 0, 1], shape=(n, n)).tolil()
    for row in rows:
        for col in row + 5 + np.arange(entries):
            A[row, col % n] = A[col % n, row] = -0.001
        A[row, row] += 0.001 * entries
    A = A.tocsr()
    A.sort_indices()
    return A


@pytest.mark.parametrize("entries,rows", [(28, [3]), (29, [3]), (300, [3]), (16, [3, 515]),
                                          (17, [3, 515]), (40, range(3, 4096, 512))],
                         ids=["24", "25", "296", "24-in-two", "26-in-two", "288-in-eight"])
def test_small_csr_pcg_of_long_rows(entries, rows):
    """At most, and more than, 24 entries past the registers in one wave of the
    one-workgroup solve (rows of entries + 3, 7 in registers); tolerances as
    test_small_csr_pcg."""
    from tatva_amd import solvers

    A = system_with_long_rows(4096, entries, rows)
    b = np.random.default_rng(1).standard_normal(4096)
    x, info = solvers.pcg(sparse.ColoredMatrix.from_csr(A), b, tol=1e-12)
    assert info.converged
    assert np.linalg.norm(b - A @ to_np(x)) < 1e-9 * np.linalg.norm(b)


def test_small_csr_pcg_of_long_rows_is_no_slower_than_a_larger_one():
    """Eight rows of 43 entries that one wave would read one after another: 128 iterations
    of 4096 rows took 5.6 times those of 4097 (which never run in one workgroup); the
    same kernels now, so half as much again is the limit.  Medians of five."""
    import time

    import torch

    from tatva_amd import solvers

    times = []
    for n in (4096, 4097):
        K = sparse.ColoredMatrix.from_csr(system_with_long_rows(n, 40, range(3, 4096, 512)))
        b, ws = torch.ones(n, dtype=torch.float64, device="cuda"), solvers._Workspace()
        runs = []
        for maxiter in (16, 144) * 6:
            start = time.perf_counter()
            solvers.pcg(K, b, tol=0.0, maxiter=maxiter, workspace=ws)
            torch.cuda.synchronize()
            runs.append(time.perf_counter() - start)
        times.append(np.median(runs[3::2]) - np.median(runs[2::2]))
    assert times[0] < 1.5 * times[1]


@pytest.mark.parametrize("density", [LE, NH, PO], ids=["le", "nh", "poisson"])
@pytest.mark.parametrize("k", [3, 4, 9])
def test_hessian_rows_at_one_point(k, density):
    """General Hex8 elements of a one-point rule, whose lanes all take that point: nodes
    in fewer, as many and more elements than are held at a time."""
    got, ref = hessian_pair(fan("hex8", k), ta.Hexahedron8(*gauss(1)), density, ORACLE[density])
    assert rel_err(got, ref) < RTOL


def test_hessian_rows_at_one_point_cost_less_than_at_eight():
    """32^3 Neo-Hookean: 212 us for one point and for eight when the lanes without a point
    computed theirs for a weight of zero; 92 and 210 now, so 0.7 is between."""
    import torch

    mesh = ta.Mesh.box((32, 32, 32), jitter=0.1)
    times = []
    for points in (1, 2):
        E = ta.Operator(mesh, ta.Hexahedron8(*gauss(points))).energy(NH)
        u = torch.zeros(E.size, dtype=torch.float64, device="cuda")
        J = sparse.jacfwd(E.grad, sparse.ColoredMatrix.from_csr(sparse.pattern_from_mesh(mesh, 3)))
        times.append(median_ms(lambda J=J, u=u: J(u)))
    assert times[0] < 0.7 * times[1]


def parallelepipeds(shape):
    """Hex8 parallelepipeds that are no boxes: node numbers over 8 times a matrix of
    multiples of 1/8, so that every sum of coordinates is exact."""
    m = ta.Mesh.box(shape)
    X = np.round(m.coords * shape) / 8.0
    m = m.set_coords(X @ np.array([[1.0, 0.25, 0.0], [0.5, 1.0, 0.125], [0.0, -0.25, 1.0]]))
    lay = ta.Operator(m, ta.Hexahedron8()).device_layout()
    assert (lay["hex_affine"], lay["hex_box"]) == (1, 0)
    return m


@pytest.mark.parametrize("density", [LE, NH, PO], ids=["le", "nh", "poisson"])
@pytest.mark.parametrize("points", [1, 2, 3])
def test_parallelepipeds(points, density):
    """Energy, residual, product, diagonal and Hessian rows (with and without constrained
    dofs) against the oracle; tolerances as the tests of each above."""
    import torch

    mesh, el = parallelepipeds((5, 7, 9)), ta.Hexahedron8(*gauss(points))
    E = ta.Operator(mesh, el).energy(density)
    prob = fem.Problem(fem.Hex8(el.quad_points, el.quad_weights), mesh.coords, mesh.elements,
                       ORACLE[density])
    rng = np.random.default_rng(5)
    u, v = 0.005 * rng.standard_normal(E.size), rng.standard_normal(E.size)
    volume = 0.90625 * 315 / 512
    assert abs(float(E(u)) - prob.energy(u)) < RTOL * (abs(prob.energy(u)) + 1.5 * 0.7 * volume)
    assert rel_err(to_np(E.grad(u)), prob.residual(u)) < RTOL
    assert rel_err(to_np(E.hvp(u, v)), prob.hvp(u, v)) < RTOL
    assert rel_err(to_np(E.hessian_diag(u)), prob.hessian_diag(u)) < RTOL
    u32, v32 = (torch.as_tensor(a, dtype=torch.float32, device="cuda") for a in (u, v))
    u_, v_ = to_np(u32).astype(float), to_np(v32).astype(float)
    assert rel_err(to_np(E.hvp(u32, v32)), prob.hvp(u_, v_)) < 2e-6
    assert rel_err(to_np(E.hessian_diag(u32, dtype=torch.float32)), prob.hessian_diag(u_)) < 2e-6
    nc = E.ncomp
    for fixed in (None, np.r_[0:4 * nc, [11 * nc, 30 * nc + nc - 1]]):
        got, ref = hessian_pair(parallelepipeds((4, 3, 5)), el, density, ORACLE[density], fixed=fixed)
        assert rel_err(got, ref) < RTOL


@pytest.mark.parametrize("density", [LE, NH, PO], ids=["le", "nh", "poisson"])
def test_parallelepipeds_matfree_pcg(density):
    """The FP32 PCG reads the geometry of parallelepipeds (44 bytes an element) or computes
    it: the same bits, also where the linearisation is written through it.  Residual as
    test_matfree_pcg_step_by_nodes."""
    import torch

    from tatva_amd import solvers

    mesh = parallelepipeds((9, 7, 10))
    E = ta.Operator(mesh, ta.Hexahedron8()).energy(density)
    nc = E.ncomp
    low = np.where(mesh.coords[:, 2] <= mesh.coords[:, 1] * 0.125)[0]
    L = lifter.Lifter(E.size, lifter.Fixed((low[:, None] * nc + np.arange(nc)).ravel(), 0.0))
    red = E.reduced(L)
    g = torch.Generator(device="cuda").manual_seed(3)
    u = 1e-3 * torch.randn(E.size, dtype=torch.float32, device="cuda", generator=g)
    b = torch.randn(red.size, dtype=torch.float32, device="cuda", generator=g)
    try:
        for lin in ("never", "always"):
            solvers.set_linearization_cache(lin)
            out = []
            for geo in (True, False):
                solvers.set_geometry_cache(geo)
                x, info = solvers.pcg_matfree(red, u, b, tol=1e-4)
                assert info.converged
                out.append((info.iterations, x))
            assert out[0][0] == out[1][0] and torch.equal(out[0][1], out[1][1])
            r = b.double() - red.hvp_full_state(u.double(), out[0][1].double())
            assert float(r.norm() / b.double().norm()) < 2e-4
    finally:
        solvers.set_geometry_cache(True)   # the defaults
        solvers.set_linearization_cache("never")


def batch_solve(problems, tol=1e-4):
    """x of H(u) x = b of each (reduced energy, u, b) as slots of one batch, and its
    iterations."""
    import ctypes

    import torch

    from tatva_amd import _native as nat

    L, s, B = nat.lib(), nat.stream(), ctypes.c_void_p()
    nat.check(L.tatva_batch_create(0, len(problems), ctypes.byref(B)))
    keep, xs = [], []
    for k, (red, u, b) in enumerate(problems):
        E, dmap, n = red.energy, red.lifter.dof_map_device(), red.size
        diag = E.hessian_diag(u, dof_map=dmap, n_out=n, dtype=torch.float32)
        x = torch.zeros_like(b)
        nbytes = L.tatva_batch_slot_workspace(E.op.handle, E.ncomp, n)
        ws = torch.empty(int(nbytes), dtype=torch.uint8, device="cuda")
        nat.check(L.tatva_batch_start(B, k, E.op.handle, ctypes.byref(E._desc), nat.dptr(u),
                                      nat.dptr(dmap), n, nat.dptr(diag), nat.dptr(b), nat.dptr(x),
                                      tol, 2000, nat.dptr(ws), ws.numel(), s))
        keep.append((diag, ws))
        xs.append(x)
    stats, running = (nat.PcgStats * len(problems))(), ctypes.c_int32(1)
    for _ in range(300):
        nat.check(L.tatva_batch_iterate(B, 8, s))
        nat.check(L.tatva_batch_poll(B, stats, ctypes.byref(running), s))
        if running.value == 0:
            break
    assert running.value == 0
    assert all(st.reserved != 0 and st.status == 0 for st in stats)
    for k in range(len(problems)):
        nat.check(L.tatva_batch_release(B, k))
    nat.check(L.tatva_batch_destroy(B))
    return xs, [st.iterations for st in stats]


def clamped(mesh, density, end):
    """(reduced energy, state, right-hand side) with the nodes ``end`` fixed."""
    import torch

    E = ta.Operator(mesh, ta.Hexahedron8()).energy(density)
    nc = E.ncomp
    L = lifter.Lifter(E.size, lifter.Fixed((end[:, None] * nc + np.arange(nc)).ravel(), 0.0))
    g = torch.Generator(device="cuda").manual_seed(E.size)
    u = 1e-4 * torch.randn(E.size, dtype=torch.float32, device="cuda", generator=g)
    red = E.reduced(L)
    return red, u, torch.randn(red.size, dtype=torch.float32, device="cuda", generator=g)


def test_batch_class_of_mixed_densities_and_geometries():
    """Hex8 slots of every density on boxes, parallelepipeds and general elements, three
    launch classes of three densities each: every slot as alone, bit for bit, and its
    residual as test_matfree_pcg_step_by_nodes."""
    import torch

    problems = [clamped(mesh, density, np.where(ta.Mesh.box(shape).coords[:, 2] == 0.0)[0])
                for shape, mesh in (((6, 5, 7), ta.Mesh.box((6, 5, 7))),
                                    ((6, 5, 7), parallelepipeds((6, 5, 7))),
                                    ((9, 6, 8), ta.Mesh.box((9, 6, 8), jitter=0.1)))
                for density in (PO, LE, NH)]
    together, its = batch_solve(problems)
    for (red, u, b), x, it in zip(problems, together, its):
        (alone,), (it_alone,) = batch_solve([(red, u, b)])
        assert it == it_alone and torch.equal(x, alone)
        r = b.double() - red.hvp_full_state(u.double(), x.double())
        assert float(r.norm() / b.double().norm()) < 2e-4


@pytest.mark.parametrize("density", [LE, NH, PO], ids=["le", "nh", "poisson"])
def test_matfree_pcg_dot_of_tiles_of_many_nodes(density):
    """Tiles of more than 512 local nodes (a beam one element thick: 1028), whose dot reads
    v again past the first two of a thread: iterations within 10 % of the FP64 PCG's (a
    wrong dot is a wrong step length) and the residual as test_matfree_pcg_step_by_nodes,
    single and batched."""
    from tatva_amd import solvers

    mesh = ta.Mesh.box((515, 1, 1), lengths=(515.0, 1.0, 1.0))
    red, u, b = clamped(mesh, density, np.where(mesh.coords[:, 2] == 0.0)[0])
    lay = red.op.device_layout()
    assert lay["max_local"] > 1024 and lay["n_tiles"] >= 2
    cm = sparse.ColoredMatrix.from_csr(
        red.lifter.adapt_sparsity(sparse.pattern_from_mesh(mesh, red.ncomp)))
    data = sparse._HessianAssembler(red.grad, cm).assemble_full_state(u.double(), red.lifter)
    H = sps.csr_matrix((to_np(data), to_np(cm.indices), to_np(cm.indptr)), shape=cm.shape)
    b64 = to_np(b).astype(float)
    want = fem.pcg(H, b64, tol=1e-4)[1]
    single, info = solvers.pcg_matfree(red, u, b, tol=1e-4)
    assert info.converged
    (batched,), (its,) = batch_solve([(red, u, b)])
    for x, it in ((single, info.iterations), (batched, its)):
        assert abs(it - want) <= max(2, 0.1 * want)
        assert np.linalg.norm(b64 - H @ to_np(x).astype(float)) < 2e-4 * np.linalg.norm(b64)


def shape_gradients(mesh, el):
    """dN_a/dx_j at the points, (element, point, j, a), in 80-bit arithmetic."""
    X = mesh.coords[mesh.elements].astype(np.longdouble)
    s, q = el._reference_nodes().astype(np.longdouble), el.quad_points.astype(np.longdouble)
    f = 1 + s[None] * q[:, None]  # (point, node, axis)
    dN = np.stack([s[:, k] / 8 * np.prod(np.delete(f, k, axis=2), axis=2) for k in range(3)], axis=2)
    J = np.einsum("qak,eaj->eqkj", dN, X)
    inv = np.empty_like(J)  # cofactors
    for i in range(3):
        for j in range(3):
            a, b, c, d = (i + 1) % 3, (i + 2) % 3, (j + 1) % 3, (j + 2) % 3
            inv[..., j, i] = J[..., a, c] * J[..., b, d] - J[..., a, d] * J[..., b, c]
    det = np.einsum("...k,...k->...", J[..., 0, :], inv[..., :, 0])
    return np.einsum("eqjk,qak->eqja", inv / det[..., None, None], dN)


def test_point_gradients_do_not_lose_the_coordinates_places():
    """Gradients on small elements far from the origin (edges 1/64 at 100, 50, -70) against
    80-bit arithmetic: the differences of an element's coordinates are exact, so J and the
    natural gradients carry the rounding of some eight operations each and the inverse a
    few more; 20 last places relative to the largest gradient bound them, where sums of the
    coordinates themselves would leave 100 / (1/64) = 6400."""
    mesh = ta.Mesh.box((6, 5, 7), lengths=(6 / 64, 5 / 64, 7 / 64), origin=(100.0, 50.0, -70.0),
                       jitter=0.1, seed=3)
    op = ta.Operator(mesh, ta.Hexahedron8())
    u = np.random.default_rng(1).uniform(1.0, 2.0, (mesh.n_nodes, 3))
    ref = np.einsum("eqja,eac->eqcj", shape_gradients(mesh, op.element), u[mesh.elements].astype(np.longdouble))
    err = np.max(np.abs(to_np(op.grad(u)).astype(np.longdouble) - ref))
    assert err < 20 * np.finfo(float).eps * np.max(np.abs(ref))


@pytest.mark.parametrize("nc", [1, 2, 3])
@pytest.mark.parametrize("points", [2, 3])
@pytest.mark.parametrize("jitter", [0.0, 0.1])
def test_point_gradients_of_infinite_values(jitter, points, nc):
    """A node's infinite value makes the gradients around it infinite, with the signs of
    its shape gradients (NaN where two disagree or the value is NaN), and no others."""
    mesh, el = ta.Mesh.box((4, 3, 5), jitter=jitter, seed=5), ta.Hexahedron8(*gauss(points))
    u = np.random.default_rng(0).standard_normal((mesh.n_nodes, nc))
    u[37, 0], u[38, nc - 1], u[60, 0], u[0, nc - 1], u[11, 0] = np.inf, np.inf, -np.inf, -np.inf, np.nan
    got = to_np(ta.Operator(mesh, el).grad(u))
    B = shape_gradients(mesh, el).astype(float)
    with np.errstate(invalid="ignore"):
        ref = (B[:, :, None] * np.moveaxis(u[mesh.elements], 1, 2)[:, None, :, None]).sum(axis=-1)
    assert np.isinf(ref).any() and np.isnan(ref).any()
    for of in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(of(got), of(ref))
    finite = np.isfinite(ref)
    assert rel_err(got[finite], ref[finite]) < RTOL

"""The multigrid preconditioner of the linear solves (taken by the automatic
choice on large systems): solutions against scipy's splu, and the systems it
has to leave to Jacobi.

Tolerance: both solves end at a relative residual of 1e-12 or below, so they
differ by at most a few 1e-12 times the condition number in the norm of
x: 1e-12 * 1e4 for the regular systems here (the largest condition number is
that of the Jacobi-scaled 16,000-row ones); the true residual is held to 1e-11,
ten times the recurrence's, for what rounding adds to it."""

import numpy as np
import pytest
from scipy import sparse
from scipy.sparse.linalg import splu

from lapy_amd import Solver, TetMesh, TriaMesh, _lib, meshgen

pytestmark = pytest.mark.gpu


def _cap(level, keep):
    """Open surface with an odd number of vertices."""
    v, t = meshgen.perturbed_sphere(level, np.random.default_rng(4), axes=(1.3, 0.8, 1.0), sigma=0.02)
    t = t[(v[:, 2] > np.quantile(v[:, 2], 1 - keep))[t].all(axis=1)]
    used, t = np.unique(t, return_inverse=True)
    return v[used], t.reshape(-1, 3)


def _systems():
    v, t = _cap(5, 0.43)  # 4,3xx rows: just above the smallest system that takes the cycle
    yield "cap", Solver(TriaMesh(v, t), lump=True), 20
    yield "closed", Solver(TriaMesh(*meshgen.perturbed_sphere(5, np.random.default_rng(3), sigma=0.05)), lump=True), 1
    yield "tets", Solver(TetMesh(*meshgen.tet_cube(25, jitter=0.15)), lump=True), 40


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 9])  # partials in the cycle up to 4 columns, their own launch beyond
def test_dirichlet_systems_against_splu(m):
    ctx = _lib.default_context()
    rng = np.random.default_rng(m)
    for name, fem, nd in _systems():
        a = sparse.csr_matrix(fem.stiffness)
        n = a.shape[0]
        dmask = np.zeros(n, np.uint8)
        dmask[rng.choice(n, nd, replace=False)] = 1
        free = np.flatnonzero(dmask == 0)
        b = rng.standard_normal((n, m))
        x, st = _lib.pcg(ctx, fem.device_matrices()[0], None, 0.0, 1.0, b, dmask=dmask, rtol=1e-12)
        _, st_j = _lib.pcg(ctx, fem.device_matrices()[0], None, 0.0, 1.0, b[:, 0], dmask=dmask, rtol=1e-12,
                           poly_degree=1)
        print(name, n, "columns", m, "iterations", st.iterations, "jacobi", st_j.iterations, flush=True)
        assert st.fallback_used == 0 and 4 * st.iterations < st_j.iterations  # the cycle ran
        af = a[free][:, free]
        xo = splu(sparse.csc_matrix(af)).solve(b[free])
        for c in range(m):
            assert np.linalg.norm(b[free, c] - af @ x[free, c]) <= 1e-11 * np.linalg.norm(b[free, c])
            assert np.linalg.norm(x[free, c] - xo[:, c]) <= 1e-8 * np.linalg.norm(xo[:, c])
        assert np.all(x[dmask == 1] == 0.0)


def test_singular_and_mass_systems():
    ctx = _lib.default_context()
    rng = np.random.default_rng(2)
    for name, fem, _ in _systems():
        a, b = fem.device_matrices()
        A, B = sparse.csr_matrix(fem.stiffness), sparse.csr_matrix(fem.mass)
        n = A.shape[0]
        f = rng.standard_normal((n, 2))
        x, st = _lib.pcg(ctx, a, None, 0.0, 1.0, f, rtol=1e-12)  # constants: the null space
        p = f - f.mean(axis=0)
        assert st.fallback_used == 0 and st.iterations < 120
        for c in range(2):
            assert abs(x[:, c].mean()) <= 1e-12 * np.abs(x[:, c]).max()
            assert np.linalg.norm(p[:, c] - A @ x[:, c]) <= 1e-11 * np.linalg.norm(p[:, c])
        t = 1.0  # a long time step: mass + t stiffness, ill-conditioned
        h, st = _lib.pcg(ctx, a, b, 1.0, t, f, rtol=1e-12)
        k = sparse.csc_matrix(B + t * A)
        ho = splu(k).solve(f)
        print(name, "mass system iterations", st.iterations, flush=True)
        for c in range(2):
            assert np.linalg.norm(f[:, c] - k @ h[:, c]) <= 1e-11 * np.linalg.norm(f[:, c])
            assert np.linalg.norm(h[:, c] - ho[:, c]) <= 1e-8 * np.linalg.norm(ho[:, c])


def test_repeated_solves_are_bit_identical():
    """Hierarchy, cycle and reductions are summed in fixed orders."""
    ctx = _lib.default_context()
    _, fem, _ = next(_systems())
    b = np.random.default_rng(1).standard_normal(fem.device_matrices()[0].n)
    x = [_lib.pcg(ctx, fem.device_matrices()[0], None, 0.0, 1.0, b, rtol=1e-12)[0] for _ in range(2)]
    assert np.array_equal(x[0], x[1])


def test_systems_left_to_jacobi():
    """A negative definite matrix, a diagonal one and one whose rows couple to
    nothing strongly: solved as before, without the cycle."""
    ctx = _lib.default_context()
    n = 6000
    rng = np.random.default_rng(5)
    lap = sparse.diags([-np.ones(n - 1), 2.0 * np.ones(n) + 0.5, -np.ones(n - 1)], [-1, 0, 1], format="csr")
    weak = sparse.diags([-1e-3 * np.ones(n - 1), np.ones(n), -1e-3 * np.ones(n - 1)], [-1, 0, 1], format="csr")
    b = rng.standard_normal(n)
    for m in (-lap, sparse.csr_matrix(sparse.diags(rng.uniform(1, 2, n))), weak):
        a = _lib.DeviceCSR.from_scipy(ctx, m)
        x, st = _lib.pcg(ctx, a, None, 0.0, 1.0, b, rtol=1e-12)
        assert np.linalg.norm(b - m @ x) <= 1e-11 * np.linalg.norm(b)
        xj, st_j = _lib.pcg(ctx, a, None, 0.0, 1.0, b, rtol=1e-12, poly_degree=1)
        assert (st.iterations, st.fallback_used) == (st_j.iterations, 0) and np.array_equal(x, xj)


def test_rows_with_many_entries():
    """A graph Laplacian with rows of 3 to ~300 entries, not from a mesh: CSR
    products, long rows in every setup kernel, hash tables of both sizes (a hub
    couples most of the ~700 aggregates, weakly)."""
    ctx = _lib.default_context()
    n = 5003
    rng = np.random.default_rng(6)
    i = np.repeat(np.arange(n), 3)
    j = (i + np.rint(rng.normal(0, 3, len(i))).astype(int)) % n
    hub = rng.choice(n, 8, replace=False)
    i = np.concatenate([i, np.repeat(hub, 300)])
    j = np.concatenate([j, rng.integers(0, n, 8 * 300)])
    wt = np.where(np.arange(len(i)) < 3 * n, rng.uniform(0.5, 1.5, len(i)), 0.01)
    keep = i != j
    w = sparse.coo_matrix((wt[keep], (i[keep], j[keep])), shape=(n, n)).tocsr()
    w = w + w.T
    a = sparse.csr_matrix(sparse.diags(np.asarray(w.sum(axis=1)).ravel() + 1e-3) - w)
    b = rng.standard_normal(n)
    d = _lib.DeviceCSR.from_scipy(ctx, a)
    x, st = _lib.pcg(ctx, d, None, 0.0, 1.0, b, rtol=1e-12)
    _, st_j = _lib.pcg(ctx, d, None, 0.0, 1.0, b, rtol=1e-12, poly_degree=1)
    print("iterations", st.iterations, "jacobi", st_j.iterations, "longest row", np.diff(a.indptr).max())
    assert st.fallback_used == 0 and 4 * st.iterations < st_j.iterations  # the cycle ran
    assert np.linalg.norm(b - a @ x) <= 1e-11 * np.linalg.norm(b)


@pytest.mark.parametrize("spokes", [1000, 1024, 1025, 1500])  # entries of the longest row of P^T: about one a spoke
def test_long_coarse_rows(spokes):
    ctx = _lib.default_context()
    n = 6001
    i = np.arange(n - 1)
    r, c = np.r_[i, np.full(spokes, n - 1)], np.r_[(i + 1) % (n - 1), np.arange(spokes)]
    w = sparse.coo_matrix((np.r_[np.ones(n - 1), np.full(spokes, 0.01)], (r, c)), shape=(n, n)).tocsr()
    w = w + w.T
    a = sparse.csr_matrix(sparse.diags(np.asarray(w.sum(axis=1)).ravel() + 1e-4) - w)
    b = np.random.default_rng(spokes).standard_normal(n)
    x, st = _lib.pcg(ctx, _lib.DeviceCSR.from_scipy(ctx, a), None, 0.0, 1.0, b, rtol=1e-12)
    assert st.fallback_used == 0 and st.iterations < 120
    assert np.linalg.norm(b - a @ x) <= 1e-11 * np.linalg.norm(b)


def _meridians(nu, nv):
    """A sphere of nu meridians: two vertices with nu neighbours."""
    th, ph = np.linspace(0.0, np.pi, nv + 1)[1:-1], 2 * np.pi * np.arange(nu) / nu
    ring = np.stack([np.outer(np.sin(th), np.cos(ph)), np.outer(np.sin(th), np.sin(ph)),
                     np.outer(np.cos(th), np.ones(nu))], axis=-1).reshape(-1, 3)
    v = np.r_[[[0.0, 0.0, 1.0]], ring, [[0.0, 0.0, -1.0]]]
    j = np.arange(nu)
    at = lambda r, q: 1 + r * nu + q % nu  # noqa: E731
    t = [np.c_[np.zeros(nu, int), at(0, j), at(0, j + 1)]]
    for r in range(nv - 2):
        t += [np.c_[at(r, j), at(r + 1, j), at(r + 1, j + 1)], np.c_[at(r, j), at(r + 1, j + 1), at(r, j + 1)]]
    t.append(np.c_[at(nv - 2, j), np.full(nu, len(v) - 1), at(nv - 2, j + 1)])
    return v, np.concatenate(t)


@pytest.mark.parametrize("nu", [126, 127, 128, 300])  # rows of nu + 1 entries: either side of the limit of 128
def test_poles_with_many_neighbours(nu):
    ctx = _lib.default_context()
    fem = Solver(TriaMesh(*_meridians(nu, 50)), lump=True)
    a = sparse.csr_matrix(fem.stiffness)
    assert np.diff(a.indptr).max() == nu + 1
    b = np.random.default_rng(nu).standard_normal(a.shape[0])
    b -= b.mean()
    x, st = _lib.pcg(ctx, fem.device_matrices()[0], None, 0.0, 1.0, b, rtol=1e-12)
    assert st.fallback_used == 0 and st.iterations < 60
    assert np.linalg.norm(b - a @ x) <= 1e-11 * np.linalg.norm(b)


def test_rejected_hierarchy_costs_little():
    """Poles of 1,000 neighbours couple more columns than the products' hash
    tables hold, so the solve is Jacobi's after all: the set-up's try may not
    cost half as much again (one thread forming a pole's row of P made it 2.4
    times the call; 1.05 now)."""
    ctx = _lib.default_context()
    fem = Solver(TriaMesh(*_meridians(1000, 24)), lump=True)
    n = fem.stiffness.shape[0]
    b = np.random.default_rng(1).standard_normal(n)
    b -= b.mean()
    best = {}
    for degree in (1, 0, 1, 0, 1, 0):
        _, st = _lib.pcg(ctx, fem.device_matrices()[0], None, 0.0, 1.0, b, rtol=1e-12, poly_degree=degree)
        best[degree] = min(best.get(degree, np.inf), st.t_total_us)
    print("n", n, "Jacobi us", best[1], "automatic us", best[0], "iterations", st.iterations)
    assert st.iterations > 200 and best[0] < 1.5 * best[1]


def _eig_problem(name, unit=1.0):
    if name == "tail":  # 642 rows: every level in the one-launch tail
        v, t = meshgen.perturbed_sphere(3, np.random.default_rng(1), axes=(1.3, 0.8, 1.0), sigma=0.02)
    elif name == "one level":  # 2,562 rows: the finest level launched, lumped mass
        v, t = meshgen.perturbed_sphere(4, np.random.default_rng(2), axes=(1.3, 0.8, 1.0), sigma=0.05)
    elif name == "cap":  # odd rows, the locality order, 8 slots a row
        v, t = _cap(5, 0.43)
    else:
        v, t = meshgen.tet_cube(17, jitter=0.15)  # 5,832 rows of ~15 entries
        return Solver(TetMesh(unit * v, t))
    return Solver(TriaMesh(unit * v, t), lump=name == "one level")


@pytest.mark.parametrize("name,k,block", [("tail", 5, 0), ("tail", 10, 13), ("one level", 9, 18), ("one level", 33, 0),
                                          ("cap", 3, 7), ("cap", 40, 66), ("tets", 12, 0)])
def test_eigenpairs_with_the_block_cycle(name, k, block):
    """Widths that are no multiples of the four columns a lane holds, one
    lane to more than 16 lanes a row, each kind of finest level.  Held to the
    solver's own bar: residuals of 1e-9 (ten times that for the host's
    rounding), eigenvalues within 1e-10 of scipy's (their error is the
    residual's square), B-orthonormal to 1e-9."""
    from oracle import fem as ofem

    fem = _eig_problem(name)
    lam, x = fem.eigs(k=k, block=block)
    st = fem.last_stats
    print(name, x.shape, "block", block, "iterations", st.iterations)
    assert st.fallback_used == 0 and st.iterations <= 60
    a, b = fem.stiffness, fem.mass
    bx = b @ x
    res = np.linalg.norm(a @ x - bx * lam, axis=0) / np.linalg.norm(bx, axis=0)
    assert np.all(res <= 1e-8 * np.maximum(np.abs(lam), 1e-2 * lam[-1]))
    assert np.abs(x.T @ bx - np.eye(k)).max() <= 1e-9
    lo = ofem.eigs(a, b, k=k)[0]
    assert np.all(np.abs(lam - lo) <= 1e-10 * lo[-1])


def _bad_element(name):
    """A regular mesh with one bad element: the vertex moved."""
    if name == "sliver":  # to 0.08 of its height over an edge
        v, t = meshgen.icosphere(6)
        tri = t[(t == 20000).any(axis=1)][0]
        mid = v[tri[tri != 20000]].mean(axis=0)
        v[20000] = mid + 0.08 * (v[20000] - mid)
        return Solver(TriaMesh(v, t))
    v, t = meshgen.tet_cube(24)
    v[25**3 // 2] += 0.48 / 24 * np.array([1.0, -1.0, 0.0])  # almost into a face
    return Solver(TetMesh(v, t))


@pytest.mark.parametrize("name", ["sliver", "flat tet"])
def test_cycle_is_positive_definite_on_bad_elements(name):
    """On the top eigenvector x of D^-1 K, which one element's mode is here,
    the smoother's error polynomial is largest.  0 < x K M K x <= x K x says
    that M is positive and does not overshoot there; 1e-8 allows for the
    rounding of x."""
    from scipy.sparse.linalg import eigsh

    fem = _bad_element(name)
    k = sparse.csr_matrix(fem.stiffness)
    k = k + sparse.diags(1e-6 * k.diagonal())  # regular
    s = sparse.diags(1.0 / np.sqrt(k.diagonal()))
    lam, x = eigsh(s @ k @ s, k=1, which="LA", tol=1e-6)
    kx = k @ (s @ x)
    ctx = _lib.default_context()
    z = _lib.cycle_apply(ctx, _lib.DeviceCSR.from_scipy(ctx, k), kx)
    part = float(kx[:, 0] @ z[:, 0]) / float((s @ x)[:, 0] @ kx[:, 0])
    print(name, "top eigenvalue", lam[0], "x K M K x / x K x", part)
    assert 0.0 < part <= 1.0 + 1e-8


@pytest.mark.parametrize("name", ["tail", "rough surface", "rough tets", "flat tets"])
def test_cycle_spectrum(name):
    """M symmetric and M K's eigenvalues in (0, 1], from the whole matrices:
    as far as rounding goes, which the condition number (1e7 at most) raises
    to about 1e-9."""
    from scipy.linalg import cholesky, eigvalsh

    if name == "tail":
        fem = _eig_problem("tail")
    elif name == "rough surface":
        fem = Solver(TriaMesh(*meshgen.perturbed_sphere(4, np.random.default_rng(5), sigma=0.06)))
    elif name == "rough tets":
        fem = Solver(TetMesh(*meshgen.tet_cube(12, jitter=0.2)))
    else:
        fem = Solver(TetMesh(*meshgen.tet_cube(11, jitter=0.28)))
    k = sparse.csr_matrix(fem.stiffness)
    k = k + sparse.diags(1e-5 * k.diagonal())
    n = k.shape[0]
    ctx = _lib.default_context()
    m = _lib.cycle_apply(ctx, _lib.DeviceCSR.from_scipy(ctx, k), np.eye(n))
    assert np.abs(m - m.T).max() <= 1e-9 * np.abs(m).max()
    c = cholesky(k.toarray(), lower=True)
    w = eigvalsh(c.T @ (0.5 * (m + m.T)) @ c)
    print(name, n, "M K in", w[0], w[-1])
    assert w[0] > 0.02 and w[-1] <= 1.0 + 1e-8


@pytest.mark.parametrize("unit", [1.0, 1e-2, 1e-3])
@pytest.mark.parametrize("name,k", [("tets", 20), ("tets", 77), ("cap", 50), ("tail", 10)])
def test_mixed_precision_keeps_the_cycle(name, k, unit):
    """FP32 blocks whose first preconditioned columns are the same to 1e-4 or
    less (near-null components): orthonormalised in two steps instead of
    refused, so that the solve takes the FP64 one's iterations, a few more for
    the hand-over."""
    fem = _eig_problem(name, unit)
    lam, _ = fem.eigs(k=k)
    its = fem.last_stats.iterations
    mixed, _ = fem.eigs(k=k, precision="mixed")
    st = fem.last_stats
    print(name, k, unit, "iterations", its, "mixed", st.iterations)
    assert st.fallback_used == 0 and st.iterations <= its + 8
    assert np.all(np.abs(mixed - lam) <= 1e-10 * lam[-1])


@pytest.mark.parametrize("cells,seed,unit", [(10, 2, 1e-2), (11, 3, 1e-2), (11, 3, 1e-3)])
def test_mixed_precision_basis_stays_orthonormal(cells, seed, unit):
    """Short directions of the first blocks, made long, carry parts of X: with
    those left in, the FP32 phase ended in a block that the FP64 phase refused."""
    v, t = meshgen.tet_cube(cells, jitter=0.2, seed=seed)
    fem = Solver(TetMesh(unit * v, t))
    lam, _ = fem.eigs(k=50)
    its = fem.last_stats.iterations
    mixed, _ = fem.eigs(k=50, precision="mixed")
    st = fem.last_stats
    print(cells, seed, unit, "iterations", its, "mixed", st.iterations, "FP32", st.iterations_fp32)
    assert st.fallback_used == 0 and st.iterations <= its + 8
    assert np.all(np.abs(mixed - lam) <= 1e-10 * lam[-1])


def _two_spheres():
    v, t = meshgen.perturbed_sphere(4, np.random.default_rng(2), axes=(1.3, 0.8, 1.0), sigma=0.02)
    return np.r_[v, v + 3.0], np.r_[t, t + len(v)]  # a constant of its own on each part


@pytest.mark.parametrize("unit,sigma", [(1e-2, -0.01), (1e-3, -0.01), (1e-4, -0.01), (1.0, 0.0), (1.0, -1e-12)])
@pytest.mark.parametrize("name", ["sphere", "two spheres"])
def test_eigenpairs_in_small_units(name, unit, sigma):
    """The shift sigma far below the spectrum, so that A - sigma B is singular
    to rounding: eigenvalues and iterations are those of the same mesh in
    ordinary units."""
    v, t = meshgen.perturbed_sphere(5, np.random.default_rng(2), axes=(1.3, 0.8, 1.0), sigma=0.02) \
        if name == "sphere" else _two_spheres()
    fem = Solver(TriaMesh(v, t))
    lam, _ = fem.eigs(k=10)
    its = fem.last_stats.iterations
    fem = Solver(TriaMesh(v * unit, t))
    small, _ = fem.eigs(k=10, sigma=sigma)
    st = fem.last_stats
    print(name, unit, sigma, "iterations", its, st.iterations)
    assert st.fallback_used == 0 and st.iterations <= its + 3
    assert np.all(np.abs(small * unit**2 - lam) <= 1e-10 * lam[-1])


@pytest.mark.parametrize("shape", [{"poly_ratio": 50.0}, {"poly_storage": _lib.LH_STORE_F32},
                                   {"poly_storage": _lib.LH_STORE_F16}])
def test_shaped_polynomial_runs(shape):
    """An interval or storage for the automatic polynomial is an explicit choice
    of it: bit for bit the solve with its degree spelled out."""
    ctx = _lib.default_context()
    a, b = Solver(TriaMesh(*meshgen.perturbed_sphere(5, np.random.default_rng(2), sigma=0.02))).device_matrices()
    lam, x, st = _lib.eigs(ctx, a, b, 10, -0.01, **shape)
    lam16, x16, st16 = _lib.eigs(ctx, a, b, 10, -0.01, poly_degree=16, **shape)  # round(sqrt(10,242) / 6.3)
    assert (st.iterations, st.spmm_calls, st.fallback_used) == (st16.iterations, st16.spmm_calls, 0)
    assert np.array_equal(lam, lam16) and np.array_equal(x, x16)


def test_cycle_that_overflows_gives_way():
    """A and B near the largest FP32 number: the finest level fits, the coarse
    matrices of a volume, whose entries grow with the spacing, do not.  The
    solve goes on without the cycle (block of 18: FP32 work blocks; FP16 ones
    underflow here, as they did before there was a cycle)."""
    fem = Solver(TetMesh(*meshgen.tet_cube(17, jitter=0.1)), lump=True)
    lam, _ = fem.eigs(k=10)
    scale = 2.0**127 / np.abs(fem.stiffness).max()
    fem.stiffness, fem.mass = fem.stiffness * scale, fem.mass * scale
    big, x = fem.eigs(k=10, block=18)
    print("iterations", fem.last_stats.iterations)
    assert fem.last_stats.fallback_used == 1
    assert np.all(np.abs(big - lam) <= 1e-10 * lam[-1])


# partials of r.z from the cycle (up to four columns) and from a launch of
# their own: both go back to Jacobi's after the limit
@pytest.mark.parametrize("m", [1, 3, 4, 6])
@pytest.mark.parametrize("singular", [False, True])
def test_linear_solves_past_the_cycles_limit(m, singular, cycle_limits):
    ctx = _lib.default_context()
    _, fem, _ = next(_systems())
    a = sparse.csr_matrix(fem.stiffness)
    n = a.shape[0]
    rng = np.random.default_rng(m)
    dmask = np.zeros(n, np.uint8)
    if not singular:
        dmask[rng.choice(n, 20, replace=False)] = 1
    free = np.flatnonzero(dmask == 0)
    b = rng.standard_normal((n, m))
    if singular:
        b -= b.mean(axis=0)
    dm = None if singular else dmask
    _, full = _lib.pcg(ctx, fem.device_matrices()[0], None, 0.0, 1.0, b, dmask=dm, rtol=1e-12)
    cycle_limits(cg=8)
    x, st = _lib.pcg(ctx, fem.device_matrices()[0], None, 0.0, 1.0, b, dmask=dm, rtol=1e-12)
    print("columns", m, "iterations", full.iterations, "with the limit", st.iterations)
    assert full.fallback_used == 0 and st.fallback_used == 1 and st.iterations > 100
    for c in range(m):
        assert np.linalg.norm(b[free, c] - a[free][:, free] @ x[free, c]) <= 1e-11 * np.linalg.norm(b[free, c])


@pytest.mark.parametrize("limit", [1, 5])
def test_eigensolve_past_the_cycles_limit(limit, cycle_limits):
    fem = _eig_problem("cap")
    lam, _ = fem.eigs(k=12)
    cycle_limits(eig=limit)
    late, _ = fem.eigs(k=12)
    assert fem.last_stats.fallback_used == 1 and fem.last_stats.iterations > limit
    assert np.all(np.abs(late - lam) <= 1e-10 * lam[-1])


@pytest.mark.parametrize("jitter", [0.2, 0.25, 0.28])  # of the spacing: elements from bad to almost flat
def test_eigenpairs_on_flat_tets(jitter):
    """The block cycle that rough elements get: about the iterations that the
    Chebyshev polynomial takes (21 to 27), held to the solver's own bar."""
    fem = Solver(TetMesh(*meshgen.tet_cube(25, jitter=jitter)))
    lam, x = fem.eigs(k=10)
    st = fem.last_stats
    poly, _ = fem.eigs(k=10, poly_degree=21)
    print(jitter, "iterations", st.iterations, "polynomial", fem.last_stats.iterations)
    assert st.fallback_used == 0 and st.iterations <= 27
    bx = fem.mass @ x
    res = np.linalg.norm(fem.stiffness @ x - bx * lam, axis=0) / np.linalg.norm(bx, axis=0)
    assert np.all(res <= 1e-8 * np.maximum(np.abs(lam), 1e-2 * lam[-1]))
    assert np.all(np.abs(poly - lam) <= 1e-10 * lam[-1])


def test_eigenpairs_of_a_noisy_cap():
    """A cap of an icosphere with 1 % noise in float32, whose worst sliver the power
    steps miss: with the smoother that amplified its mode the residuals of
    this mesh stopped falling and the solve ended in the Cholesky-QR."""
    rng = np.random.default_rng([1, 20260])
    v, t = meshgen.icosphere(6)
    height = v @ np.array([0.48, 0.6, 0.64])
    t = t[(height > np.quantile(height, 1.0 - 0.713))[t].all(axis=1)]
    used, t = np.unique(t, return_inverse=True)
    v, t = v[used], t.reshape(-1, 3)
    v = v * (1.0 + 0.01 * rng.standard_normal(len(v)))[:, None] * rng.uniform(0.5, 2.0, size=3)
    fem = Solver(TriaMesh(v.astype(np.float32), t), lump=True)
    lam, x = fem.eigs(k=50)
    st = fem.last_stats
    print(len(v), "iterations", st.iterations)
    assert st.fallback_used == 0 and st.iterations <= 30
    bx = fem.mass @ x
    res = np.linalg.norm(fem.stiffness @ x - bx * lam, axis=0) / np.linalg.norm(bx, axis=0)
    assert np.all(res <= 1e-8 * np.maximum(np.abs(lam), 1e-2 * lam[-1]))


@pytest.fixture
def cycle_limits():
    ctx = _lib.default_context()
    yield ctx.set_cycle_limits
    ctx.set_cycle_limits()


# limit 3: the FP32 phase drops the cycle and the FP64 one starts without it;
# 11: the FP64 phase drops it; tol 1e-15, which nothing reaches: the default
# limit of 80 iterations, results of the last one
@pytest.mark.parametrize("limit,tol,max_iter", [(3, 0.0, 0), (11, 1e-13, 200), (0, 1e-15, 110)])
@pytest.mark.parametrize("name", ["tail", "cap"])  # 642 rows: degree 4; 4,403: 11
def test_mixed_solves_past_the_cycles_limit(name, limit, tol, max_iter, cycle_limits):
    fem = _eig_problem(name)
    a, b = fem.device_matrices()
    lam, _ = fem.eigs(k=12)
    cycle_limits(eig=limit)
    mixed, x, st = _lib.eigs(_lib.default_context(), a, b, 12, -0.01, precision=_lib.LH_PREC_MIXED, tol=tol,
                             max_iter=max_iter, allow_noconv=True)
    fp64 = st.iterations - st.iterations_fp32
    print(name, "FP32 iterations", st.iterations_fp32, "FP64", fp64, "residual", st.max_resid)
    assert st.fallback_used == 1
    assert st.iterations_fp32 > limit if limit == 3 else fp64 > (limit or 80) >= st.iterations_fp32
    assert np.all(np.abs(mixed - lam) <= 1e-10 * lam[-1])
    bx = fem.mass @ x
    res = np.linalg.norm(fem.stiffness @ x - bx * mixed, axis=0) / np.linalg.norm(bx, axis=0)
    assert np.all(res <= 1e-8 * np.maximum(np.abs(mixed), 1e-2 * mixed[-1]))


def test_eigenpairs_the_same_with_and_without_the_cycle():
    """The mixed-precision solve shares one hierarchy between its phases; an
    explicit degree keeps the polynomial."""
    fem = _eig_problem("cap")
    lam, _ = fem.eigs(k=12)
    for opts in ({"precision": "mixed"}, {"poly_degree": 11}, {"poly_degree": 1}):
        other, _ = fem.eigs(k=12, **opts)
        assert np.all(np.abs(other - lam) <= 1e-10 * lam[-1])

"""GPU tests of kg_poisson_solve (FP32 multigrid inside FP64 defect
correction).  The checks do not use the solver's own residual: the 9-point
operator is applied here in FP64 numpy to the returned solution, and that
operator is itself pinned by a textbook property (exact for polynomials of
degree <= 3).

* Manufactured solution: f = A u* for a known u* (zero boundary); the solver
  must return u* to within the conditioning of A at the requested residual.
* Random right-hand side in [-1, 1): ||f - A u||_2 / ||f||_2 < 1e-10, with
  the residual falling at every FP64 correction.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def apply_A(u, h):
    """(A u) = (20 u - 4 sum_axis - sum_diag) / (6 h^2) on the interior."""
    a = np.zeros_like(u)
    c = u[1:-1, 1:-1]
    ax = u[1:-1, :-2] + u[1:-1, 2:] + u[:-2, 1:-1] + u[2:, 1:-1]
    dg = u[:-2, :-2] + u[:-2, 2:] + u[2:, :-2] + u[2:, 2:]
    a[1:-1, 1:-1] = (20 * c - 4 * ax - dg) / (6 * h * h)
    return a


def test_operator_is_exact_for_quadratics():
    """A(x^2 + y^2) = -4 in the interior (a textbook property of the
    9-point Mehrstellen operator on polynomials of degree <= 3)."""
    n = 16
    h = 1.0 / n
    x = np.arange(n + 1) * h
    X, Y = np.meshgrid(x, x)
    a = apply_A(X ** 2 + Y ** 2 + 3 * X * Y + X ** 3, h)
    np.testing.assert_allclose(a[1:-1, 1:-1], -4 - 6 * X[1:-1, 1:-1], rtol=0, atol=1e-9)


@pytest.mark.parametrize("n", [8, 64, 256])
def test_poisson_manufactured_solution(gpu_ctx, kgmod, n):
    rng = np.random.default_rng(n)
    h = 1.0 / n
    x = np.arange(n + 1) * h
    X, Y = np.meshgrid(x, x)
    ustar = np.sin(np.pi * X) * np.sin(2 * np.pi * Y) + 0.1 * X * (1 - X) * Y * (1 - Y) * rng.uniform(-1, 1)
    ustar[0, :] = ustar[-1, :] = ustar[:, 0] = ustar[:, -1] = 0
    f = apply_A(ustar, h)
    df, du = gpu_ctx.array(f), gpu_ctx.array(np.zeros_like(f))
    rep = kgmod.poisson_solve(gpu_ctx, n, df, du, tol=1e-10)
    u = du.download()
    r = f - apply_A(u, h)
    assert np.linalg.norm(r) / np.linalg.norm(f) < 2e-10, rep
    assert np.max(np.abs(u - ustar)) < 1e-8 * np.max(np.abs(ustar)) * n * n, rep
    assert rep["rel_residual"] < 1e-10 and rep["outer"] >= 1
    df.free()
    du.free()


def test_poisson_random_rhs(gpu_ctx, kgmod):
    n = 1024
    rng = np.random.default_rng(7)
    f = rng.uniform(-1, 1, (n + 1, n + 1))
    f[0, :] = f[-1, :] = f[:, 0] = f[:, -1] = 0
    df, du = gpu_ctx.array(f), gpu_ctx.array(np.zeros_like(f))
    rep = kgmod.poisson_solve(gpu_ctx, n, df, du, tol=1e-10)
    u = du.download()
    r = f - apply_A(u, 1.0 / n)
    assert np.linalg.norm(r) / np.linalg.norm(f) < 2e-10, rep
    # each FP32 correction gains digits: the history decreases monotonically
    hist = rep["history"]
    assert all(b < a for a, b in zip(hist, hist[1:])), hist
    assert rep["outer"] <= 8, rep
    df.free()
    du.free()


def test_poisson_random_rhs_8192(gpu_ctx, kgmod):
    """The full-size configuration: 8192^2 cells (8193^2 vertices), random
    right-hand side in [-1, 1) with a zero boundary, to a relative residual
    of 1e-10.  The residual is recomputed here in FP64 numpy from the
    downloaded solution, independently of the solver's own norm."""
    n = 8192
    rng = np.random.default_rng(8192)
    f = rng.uniform(-1, 1, (n + 1, n + 1))
    f[0, :] = f[-1, :] = f[:, 0] = f[:, -1] = 0
    df, du = gpu_ctx.array(f), gpu_ctx.array(np.zeros_like(f))
    rep = kgmod.poisson_solve(gpu_ctx, n, df, du, tol=1e-10)
    u = du.download()
    df.free()
    du.free()
    r = f - apply_A(u, 1.0 / n)
    rel = np.linalg.norm(r) / np.linalg.norm(f)
    assert rel < 1e-10, (rel, rep)
    # the solver's norm and the independent one agree up to the rounding of
    # the two FP64 evaluations (different summation orders)
    assert abs(rel - rep["rel_residual"]) <= 0.1 * rel + 1e-12, (rel, rep["rel_residual"])
    hist = rep["history"]
    assert all(b < a for a, b in zip(hist, hist[1:])), hist
    assert rep["outer"] <= 8 and rep["levels"] == 13, rep


def test_poisson_first_residual_norm(gpu_ctx, kgmod):
    """From u = 0 the first recorded residual is ||f interior||_2 / ||f||_2:
    the solver's fused residual pass sums r^2 over every interior point and
    leaves the boundary (where r = 0) out.  f is nonzero on the boundary here,
    so the ratio is below 1."""
    n = 512
    rng = np.random.default_rng(11)
    f = rng.uniform(-1, 1, (n + 1, n + 1))
    df, du = gpu_ctx.array(f), gpu_ctx.array(np.zeros_like(f))
    rep = kgmod.poisson_solve(gpu_ctx, n, df, du, tol=1e-6)
    want = np.linalg.norm(f[1:-1, 1:-1]) / np.linalg.norm(f)
    assert want < 0.999
    assert abs(rep["history"][0] - want) <= 1e-13 * want, (rep["history"][0], want)


def test_poisson_rejects_bad_arguments(gpu_ctx, kgmod):
    a = gpu_ctx.empty((9 * 9,), np.float64)
    b = gpu_ctx.empty((9 * 9,), np.float64)
    with pytest.raises(kgmod.KGError):
        kgmod.poisson_solve(gpu_ctx, 6, a, b)          # not a power of two
    with pytest.raises(kgmod.KGError):
        kgmod.poisson_solve(gpu_ctx, 8, a, a)          # f aliases u


# ---- one correction against the same V-cycles in numpy, bit for bit ----
F = np.float32


def around(u):
    """Centre, the axis neighbours' sum and the diagonal neighbours' sum of
    the interior, in the order W + S + E + N and SW + NW + SE + NE."""
    ax = u[1:-1, :-2] + u[:-2, 1:-1] + u[1:-1, 2:] + u[2:, 1:-1]
    dg = u[:-2, :-2] + u[2:, :-2] + u[:-2, 2:] + u[2:, 2:]
    return u[1:-1, 1:-1], ax, dg


def sweeps(u, f, h):
    for _ in range(2):
        c, ax, dg = around(u)
        u = np.pad(F(1 - 0.8) * c + F(0.8 / 5) * ax + F(0.8 / 20) * dg + F(3 * 0.8 * h * h / 10) * f[1:-1, 1:-1], 1)
    return u


def vcycle(u, f):
    n = u.shape[0] - 1
    h = 1.0 / n
    if n == 2:
        return np.pad(F(6 * h * h / 20) * f[1:-1, 1:-1], 1)
    u = sweeps(u, f, h)
    c, ax, dg = around(u)
    r = np.pad(f[1:-1, 1:-1] - (F(20) * c - F(4) * ax - dg) * F(1 / (6 * h * h)), 1)
    R = lambda dy, dx: r[2 + dy:n - 1 + dy:2, 2 + dx:n - 1 + dx:2]  # noqa: E731
    fc = np.pad((F(4) * R(0, 0) + F(2) * (R(0, -1) + R(0, 1) + R(-1, 0) + R(1, 0)) +
                 (R(-1, -1) + R(-1, 1) + R(1, -1) + R(1, 1))) * F(0.0625), 1)
    a = vcycle(np.zeros_like(fc), fc)
    e = np.zeros_like(u)
    e[::2, ::2] = a
    e[::2, 1::2] = F(0.5) * (a[:, :-1] + a[:, 1:])
    e[1::2, ::2] = F(0.5) * (a[:-1] + a[1:])
    e[1::2, 1::2] = F(0.25) * (a[:-1, :-1] + a[:-1, 1:] + a[1:, :-1] + a[1:, 1:])
    u = u.copy()
    u[1:-1, 1:-1] += e[1:-1, 1:-1]
    return sweeps(u, f, h)


@pytest.mark.parametrize("cycles", [1, 2])
@pytest.mark.parametrize("n", [2, 4, 8, 16, 32, 64, 128, 256, 512, 1024, 2048])
def test_poisson_one_correction(gpu_ctx, kgmod, n, cycles):
    """u after one correction from a random guess: n up to 128 is the coarse
    kernel's alone; 256 columns and up take 2 or more pieces of 240, 1 to 3
    workgroups side by side and every count of rows per wave.  FP32
    arithmetic is IEEE on both sides, so the two agree bit for bit."""
    rng = np.random.default_rng(n)
    f = rng.uniform(-1, 1, (n + 1, n + 1))
    u0 = rng.uniform(-1, 1, (n + 1, n + 1))
    u0[[0, -1]] = u0[:, [0, -1]] = 0
    c, ax, dg = around(u0)
    r = np.pad(f[1:-1, 1:-1] - (20 * c - 4 * ax - dg) * (1 / (6 * (1.0 / n) ** 2)), 1).astype(F)
    e = np.zeros_like(r)
    for _ in range(cycles):
        e = vcycle(e, r)
    want = u0 + e
    for noalloc in (False, True) if n <= kgmod.POISSON_NOALLOC_MAX_N else (False,):
        df, du = gpu_ctx.array(f), gpu_ctx.array(u0)
        try:
            kgmod.poisson_solve(gpu_ctx, n, df, du, tol=1e-30, max_outer=1, vcycles=cycles, noalloc=noalloc)
        except kgmod.KGError as err:
            assert "relative residual" in str(err)
        np.testing.assert_array_equal(du.download().reshape(want.shape), want)
        df.free()
        du.free()


@pytest.mark.parametrize("n", [2, 64, 128, 256, 1024])
def test_poisson_leaves_the_boundary(gpu_ctx, kgmod, n):
    """Not a bit of u's boundary changes: -0.0 stays, and values beside it."""
    rng = np.random.default_rng(n)
    u0 = np.zeros((n + 1, n + 1))
    for edge in (np.s_[0], np.s_[-1], np.s_[:, 0], np.s_[:, -1]):
        u0[edge] = np.where(rng.random(n + 1) < 0.5, -0.0, 5e-324)
    df, du = gpu_ctx.array(rng.uniform(-1, 1, u0.shape)), gpu_ctx.array(u0)
    try:
        kgmod.poisson_solve(gpu_ctx, n, df, du, tol=1e-30, max_outer=2, vcycles=1)
    except kgmod.KGError as err:
        assert "relative residual" in str(err)
    u = du.download().reshape(u0.shape)
    df.free()
    du.free()
    for edge in (np.s_[0], np.s_[-1], np.s_[:, 0], np.s_[:, -1]):
        assert np.array_equal(u[edge].view(np.uint64), u0[edge].view(np.uint64))
    assert np.any(u[1:-1, 1:-1] != 0)


@pytest.mark.parametrize("cycles", [1, 2])
def test_poisson_one_correction_16_rows_a_wave(gpu_ctx, kgmod, cycles):
    """4096 cells: 16 rows per wave, the shape of the finest levels from here up
    (256 to 2048 cells take 2, 4 and 8)."""
    test_poisson_one_correction(gpu_ctx, kgmod, 4096, cycles)

"""CSR products and Jacobi steps against FP64 NumPy sums: right-hand-side
counts on both sides of every vector width, lane count and tile of the block
kernel, rows that are empty, shorter and longer than a pass, and all value
and vector types."""
import numpy as np
import pytest
import scipy.sparse

pytestmark = pytest.mark.gpu


def _matrix(m, n, rng, dtype):
    """Row lengths 0, 1, 3, 63 .. 65, 127 .. 129, 255 .. 257, 511 .. 513, n."""
    lens = [0, 1, 2, 3, 4, 5, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, n]
    rows = [np.sort(rng.permutation(n)[:lens[i % len(lens)]]) for i in range(m)]
    indptr = np.concatenate([[0], np.cumsum([r.size for r in rows])])
    idx = np.concatenate(rows)
    return scipy.sparse.csr_matrix((rng.uniform(0.1, 1.0, idx.size).astype(dtype), idx, indptr),
                                   shape=(m, n))


KS = [1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 33, 64, 65, 127, 128, 129, 130, 255, 256, 257, 300]


@pytest.mark.parametrize("k", KS)
@pytest.mark.parametrize("adt,xdt", [("f64", "f64"), ("f32", "f64"), ("f64", "f32"),
                                     ("f32", "f32"), ("bf16", "f32"), ("f16", "f32")])
def test_products_and_jacobi_steps(adt, xdt, k):
    import torch
    from fluxpy_amd import _kernels
    from fluxpy_amd.solve import _CsrOperator
    torch.cuda.set_device(0)
    n = 600
    rng = np.random.default_rng(k)
    A = _matrix(n, n, rng, np.float64 if adt == "f64" else np.float32)
    csr = _kernels.DeviceCSR.from_scipy(A)
    if adt in ("bf16", "f16"):
        csr = csr.astype(torch.bfloat16 if adt == "bf16" else torch.float16)
    vals = csr.data.double().cpu().numpy()
    Ad = scipy.sparse.csr_matrix((vals, A.indices, A.indptr), shape=A.shape)
    xt = torch.float64 if xdt == "f64" else torch.float32
    X = torch.from_numpy(rng.standard_normal((n, k))).cuda().to(xt)
    E = torch.from_numpy(rng.standard_normal((n, k))).cuda().to(xt)
    rho = torch.from_numpy(rng.uniform(0.1, 0.2, n)).cuda().to(xt)
    Xh, Eh, rh = (v.double().cpu().numpy() for v in (X, E, rho))
    # |sum error| <= terms x eps x sum of |a x| in the accumulation type, one
    # rounding of the result; every product within (2 + terms / 64) eps works
    # out looser than the sums need
    acc64 = "f64" in (adt, xdt)
    eps_acc, eps_out = np.finfo(np.float64 if acc64 else np.float32).eps, \
        np.finfo(np.float64 if xdt == "f64" else np.float32).eps
    absA = abs(Ad)
    bound = lambda a, y: 40 * eps_acc * a + 2 * eps_out * np.abs(y) + 1e-300
    want = Ad @ Xh
    got = csr.matmat(X).double().cpu().numpy()
    assert (np.abs(got - want) <= bound(absA @ np.abs(Xh), want)).all()
    op = _CsrOperator(csr)
    for r, rd in ((rho, rh[:, None]), (0.37, 0.37)):
        for left in (False, True):
            B1 = torch.full_like(X, float("nan"))
            cm = torch.full((k,), 9.0, dtype=torch.float64, device="cuda")
            op.jacobi_step(E, X, r, left, B1, cm)
            want = Eh + (rd * (Ad @ Xh) if left else Ad @ (rd * Xh))
            got = B1.double().cpu().numpy()
            assert (np.abs(got - want)
                    <= bound(absA @ np.abs(Xh) + np.abs(Eh), want)).all()
            assert np.array_equal(cm.cpu().numpy(), np.abs(got - Xh).max(0))


@pytest.mark.parametrize("k", [1, 3, 16])
@pytest.mark.parametrize("adt,xdt", [("f64", "f64"), ("f32", "f64"), ("f64", "f32"),
                                     ("f32", "f32"), ("bf16", "f32")])
@pytest.mark.parametrize("placement", ["left", "right", "scalar"])
def test_runs_equal_single_steps(adt, xdt, k, placement):
    """Runs of Jacobi steps return the iterate and the count of the loop that
    reads the maxima back after every step: convergence inside the first run,
    in a later one, at the first step, at an iteration limit, and columns
    with tolerances of their own."""
    import torch
    import warnings
    from fluxpy_amd import _kernels
    from fluxpy_amd.solve import _CsrOperator, _jacobi_runs
    torch.cuda.set_device(0)
    n = 600
    rng = np.random.default_rng(k)
    A = _matrix(n, n, rng, np.float64 if adt == "f64" else np.float32)
    A.data *= 0.9 / A.sum(1).max()
    csr = _kernels.DeviceCSR.from_scipy(A)
    if adt == "bf16":
        csr = csr.astype(torch.bfloat16)
    xt = torch.float64 if xdt == "f64" else torch.float32
    E = torch.from_numpy(rng.uniform(0, 1, (n, k))).cuda().to(xt)
    rho = 0.6 if placement == "scalar" else \
        torch.from_numpy(rng.uniform(0.5, 0.7, n)).cuda().to(xt)
    left = placement == "left"
    op = _CsrOperator(csr)

    def steps(tol, maxiter):
        B, B1 = E.clone(), torch.empty_like(E)
        cm = torch.empty(k, dtype=torch.float64, device="cuda")
        for it in range(1, maxiter + 1):
            op.jacobi_step(E, B, rho, left, B1, cm)
            if (cm.cpu().numpy() <= tol).all():
                break
            B, B1 = B1, B
        else:
            B = B1      # the loop breaks before its last swap
        return B, it

    eps = np.finfo(np.float64 if xdt == "f64" else np.float32).eps
    tols = [3.0, 1e-2, 3e-6] + ([1e-12] if xdt == "f64" else [])
    for tol, maxiter in [(x, 500) for x in tols] + [(1e-9, 4), (1e-9, 7), (1e-9, 1)]:
        cols = np.full(k, tol) * np.linspace(1.0, 3.0, k)
        for bound in (tol, cols, torch.from_numpy(cols).cuda()):
            lim = np.broadcast_to(tol if np.ndim(bound) == 0 else cols, (k,))
            want, it = steps(lim, maxiter)
            with warnings.catch_warnings():
                warnings.simplefilter("ignore")
                got, niter = _jacobi_runs(csr, E, rho, left, bound, maxiter)
            # the albedo may multiply elsewhere: a rounding per term and step,
            # summed over a contraction of 0.63
            assert niter == it
            d = (got - want).abs().max() / want.abs().max()
            assert d <= 30 * eps, (tol, maxiter, float(d))


def test_jacobi_of_no_columns_and_no_rows():
    """An empty batch with a tolerance of its own converges at once."""
    import torch
    from fluxpy_amd import _kernels
    from fluxpy_amd.solve import _jacobi_runs, solve_radiosity
    torch.cuda.set_device(0)
    A = scipy.sparse.csr_matrix(np.diag([0.1, 0.2, 0.3]))
    for E in (np.zeros((3, 0)), torch.zeros((3, 0), dtype=torch.float32, device="cuda")):
        B, niter = solve_radiosity(A, E, 0.3, tol=1e-6)
        assert B.shape == (3, 0) and B.dtype == E.dtype and niter == 1
    E = torch.zeros((0, 4), dtype=torch.float64, device="cuda")
    csr = _kernels.DeviceCSR.from_scipy(scipy.sparse.csr_matrix((0, 0)))
    B, niter = _jacobi_runs(csr, E, 0.3, False, 1e-6, 100)
    assert B.shape == (0, 4) and niter == 1


def test_tolerance_tensors_on_host_and_device():
    """The tolerance may be a tensor on either side, and a strided one."""
    import torch
    from fluxpy_amd.solve import solve_radiosity
    torch.cuda.set_device(0)
    A = scipy.sparse.random(300, 300, 0.2, "csr", random_state=1)
    A.data *= 0.9 / A.sum(1).max()
    E = np.random.default_rng(2).uniform(0, 1, (300, 3))
    cols = np.array([1e-3, 1e-9, 1e-6])
    want, it = solve_radiosity(A, E, 0.5, tol=cols)
    wide = torch.full((3, 4), 7.0, dtype=torch.float64)
    wide[:, 1] = torch.from_numpy(cols)
    for tol in (wide[:, 1], wide.cuda()[:, 1], torch.from_numpy(cols)):
        got, niter = solve_radiosity(A, E, 0.5, tol=tol)
        assert niter == it and np.array_equal(got, want)
    want, it = solve_radiosity(A, E, 0.5, tol=1e-9)
    for tol in (torch.tensor(1e-9, dtype=torch.float64),
                torch.tensor([1e-9], dtype=torch.float64).expand(3)):
        got, niter = solve_radiosity(A, E, 0.5, tol=tol)
        assert niter == it and np.array_equal(got, want)


def test_more_tiles_of_columns_than_a_grid_holds():
    """Two columns more than 65,535 full tiles of 128 FP64 columns."""
    import torch
    from fluxpy_amd import _kernels
    from fluxpy_amd.solve import _CsrOperator
    torch.cuda.set_device(0)
    k = 65535 * 128 + 2
    A = np.array([[0.0, 0.5], [0.25, 0.125]])
    csr = _kernels.DeviceCSR.from_scipy(scipy.sparse.csr_matrix(A))
    X = torch.arange(2 * k, dtype=torch.float64, device="cuda").reshape(2, k)
    want = torch.stack([0.5 * X[1], 0.25 * X[0] + 0.125 * X[1]])     # exact
    assert torch.equal(csr.matmat(X), want)
    B1, cm = torch.empty_like(X), torch.empty(k, dtype=torch.float64, device="cuda")
    _CsrOperator(csr).jacobi_step(X, X, 2.0, False, B1, cm)
    assert torch.equal(B1, X + 2.0 * want) and torch.equal(cm, (2.0 * want).abs().amax(0))


@pytest.mark.parametrize("k", [65, 130, 300])
def test_a_solve_that_overflows_does_not_converge(k):
    """With more than 64 columns a change that is not a number counts as the
    largest: an iteration that runs off to infinity (inf - inf) ends at its
    limit with a warning."""
    import torch
    from fluxpy_amd.solve import _CsrOperator, _jacobi_runs
    from fluxpy_amd import _kernels
    torch.cuda.set_device(0)
    csr = _kernels.DeviceCSR.from_scipy(scipy.sparse.csr_matrix(np.diag(np.full(70, 2.0 ** 100))))
    E = torch.ones((70, k), dtype=torch.float64, device="cuda")
    with pytest.warns(RuntimeWarning, match="did not converge in 40"):
        B, niter = _jacobi_runs(csr, E, 1.0, False, 1e-9, 40)
    assert niter == 40 and torch.isinf(B).all()
    X = E.clone()
    X[3, 5] = X[69, k - 1] = float("nan")
    cm = torch.empty(k, dtype=torch.float64, device="cuda")
    _CsrOperator(csr).jacobi_step(E, X, 1.0, False, torch.empty_like(E), cm)
    assert torch.isnan(cm).nonzero().reshape(-1).tolist() == [5, k - 1]

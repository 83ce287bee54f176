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

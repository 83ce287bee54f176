"""The batched symmetric eigensolver against LAPACK: odd and even sizes, the
smallest ones, both sides of the size that fits in LDS and of the widths at
which a wave holds more pairs (128, 256), graded and rank
deficient spectra, a diagonal matrix, and sizes mixed in one batch at odd
offsets."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(mats, max_sweeps=30):
    import torch
    from fluxpy_amd import _lib
    torch.cuda.set_device(0)
    ns = np.array([m.shape[0] for m in mats], dtype=np.int64)
    offA = np.concatenate([[0], np.cumsum(ns * ns)])
    offE = np.concatenate([[0], np.cumsum(ns)])
    A = torch.from_numpy(np.concatenate([m.ravel() for m in mats])).cuda()
    W, V = torch.empty_like(A), torch.empty_like(A)
    ev = torch.empty(int(offE[-1]), dtype=torch.float64, device="cuda")
    d_ns, d_oA, d_oE = (torch.from_numpy(x).cuda() for x in (ns, offA[:-1].copy(),
                                                             offE[:-1].copy()))
    _lib.call("flux_batched_syevj", len(mats), d_ns.data_ptr(), int(ns.max()), A.data_ptr(),
              d_oA.data_ptr(), W.data_ptr(), V.data_ptr(), ev.data_ptr(), d_oE.data_ptr(),
              max_sweeps, _lib.stream())
    V, ev = V.cpu().numpy(), ev.cpu().numpy()
    return [(ev[offE[b]:offE[b + 1]], V[offA[b]:offA[b + 1]].reshape(n, n))
            for b, n in enumerate(ns)]


def _matrix(n, kind, rng):
    if kind == "diagonal":
        return np.diag(rng.permutation(n) - n / 3.0)
    Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    if kind == "random":
        d = rng.standard_normal(n)
    elif kind == "graded":
        d = 10.0 ** -np.linspace(0, 14, n)
    else:
        d = np.where(np.arange(n) < max(1, n // 3), 1.0 + np.arange(n), 0.0)
    A = (Q * d) @ Q.T
    return 0.5 * (A + A.T)


@pytest.mark.parametrize("kind", ["random", "graded", "deficient", "diagonal"])
@pytest.mark.parametrize("ns", [(1,), (2, 1, 3), (5, 88, 17), (127, 128), (129, 88), (178, 31),
                                (179, 88), (256, 3), (257,)])
def test_syevj_against_lapack(ns, kind):
    rng = np.random.default_rng(sum(ns))
    mats = [_matrix(n, kind, rng) for n in ns]
    for A, (ev, V) in zip(mats, _run(mats)):
        n = A.shape[0]
        scale = max(np.abs(A).max() * n, 1e-300)
        # LAPACK and Jacobi are both backward stable: a few n eps |A|
        tol = 8 * n * np.finfo(float).eps * scale
        assert (np.diff(ev) <= 0).all()
        assert np.abs(ev - np.linalg.eigvalsh(A)[::-1]).max() <= tol
        assert np.abs(V.T @ V - np.eye(n)).max() <= 40 * n * np.finfo(float).eps
        assert np.abs(A @ V - V * ev).max() <= tol

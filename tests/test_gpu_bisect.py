"""Sturm counts of tridiagonal matrices that decouple, at points that are exactly an eigenvalue of
one of their blocks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS, TINY = np.finfo(float).eps, np.finfo(float).tiny


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a GPU"
    return t


def _diagonal(n, point, seed):
    """n values from -1 to 2, one of them exactly the given one of the 64 points at which the first
    multisection step counts; it stands first, the ends of the spectrum last."""
    d = np.linspace(-1.0, 2.0, n)
    widen = 2 * EPS * 2.0 * n + 2 * TINY
    lo, hi = -1.0 - widen, 2.0 + widen
    x = lo + (hi - lo) * float(point + 1) / 65.0
    inner = np.random.default_rng(seed).permutation(np.delete(d[1:-1], n // 2 - 1))
    return np.concatenate([[x], inner, [-1.0, 2.0]])


# off-diagonal 0 and 1e-25: counted in the ratio form; 1e-17: by the signs of the polynomials.  The
# eigenvalues are the diagonal in all three: the next term, e^2 / gap, is below 1e-31.
@pytest.mark.parametrize("off", [0.0, 1e-25, 1e-17])
@pytest.mark.parametrize("n,point,seed", [(2, 31, 0), (9, 16, 0), (40, 31, 0), (100, 16, 0), (300, 16, 1), (300, 63, 2)])
def test_points_on_an_eigenvalue(torch, n, point, seed, off):
    from apw import pw
    d = _diagonal(n, point, seed) if n > 2 else np.array([-1.0, 2.0])
    H = np.diag(d).astype(complex) + off * (np.eye(n, k=1) + np.eye(n, k=-1))
    ctx = pw.Context(0)
    dh = torch.from_numpy(np.ascontiguousarray(np.tril(H).T)).cuda()
    de = torch.zeros(n, dtype=torch.float64, device="cuda")
    dv = torch.zeros((n, n), dtype=torch.complex128, device="cuda")
    pw.dnevx_op(ctx, n, n, dh, n, de, dv)
    ctx.synchronize()
    e, V = de.cpu().numpy(), dv.cpu().numpy().T
    # bisection stops at 2 eps |lambda|; its points and counts are rounded once more
    assert np.abs(e - np.sort(d)).max() <= 8 * EPS * 2.0
    assert np.abs(H @ V - V * e).max() < 1e-12
    ctx.close()

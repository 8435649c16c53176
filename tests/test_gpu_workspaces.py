"""No result depends on what a work array held before the call: the context's work arrays are
filled with NaN and the call made again has to give the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a GPU"
    return t


# one-XCD reduction alone (64, 512); device-wide start with columns in LDS (513, 640, 704) and with
# rows split over waves (705, 1000)
@pytest.mark.parametrize("n", [64, 512, 513, 640, 704, 705, 1000])
def test_eigenproblem_on_filled_workspaces(torch, n):
    from apw import pw
    print(f"dnevx n={n}", flush=True)
    rng = np.random.default_rng(n)
    H = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    H = H + H.conj().T
    nband = max(1, n // 4)
    ctx = pw.Context(0)
    dh = torch.from_numpy(np.ascontiguousarray(np.tril(H).T)).cuda()

    def solve():
        de = torch.zeros(nband, dtype=torch.float64, device="cuda")
        dv = torch.zeros((nband, n), dtype=torch.complex128, device="cuda")
        pw.dnevx_op(ctx, n, n, dh, nband, de, dv)
        ctx.synchronize()
        return de.cpu().numpy(), dv.cpu().numpy()

    first = solve()
    ctx.fill_workspaces(float("nan"))
    again = solve()
    assert np.abs(first[0] - np.linalg.eigvalsh(H)[:nband]).max() < 1e-12 * n
    assert np.array_equal(first[0], again[0]) and np.array_equal(first[1], again[1])
    ctx.close()


@pytest.mark.parametrize("single", [False, True])
def test_split_product_on_filled_workspaces(torch, single):
    from apw import pw
    ctx = pw.Context(0)
    dt = torch.complex64 if single else torch.complex128
    m, n, k = 70, 45, 9001
    a = torch.randn((m, k), dtype=dt, device="cuda")
    b = torch.randn((n, k), dtype=dt, device="cuda")

    def product():
        out = torch.zeros((n, m), dtype=dt, device="cuda")
        pw.gemm_op(ctx, "C", "N", m, n, k, 1.0, a, k, b, k, 0.0, out, m)
        ctx.synchronize()
        return out.cpu().numpy()

    first = product()
    ctx.fill_workspaces(float("nan"))
    assert np.array_equal(first, product()) and np.isfinite(first).all()
    ctx.close()

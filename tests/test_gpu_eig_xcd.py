"""The subspace reduction on one XCD (n <= 512, and the last 512 columns of a larger matrix):
eigenpairs against LAPACK at the edges of its size classes, columns that need no reflector,
several streams at once, and contexts that come and go."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a GPU"
    return t


def _solve(torch, ctx, H, nband):
    from apw import pw
    n = H.shape[0]
    dh = torch.from_numpy(np.ascontiguousarray(np.tril(H).T)).cuda()
    de = torch.zeros(nband, dtype=torch.float64, device="cuda")
    dv = torch.zeros((n, n), dtype=torch.complex128, device="cuda")
    pw.dnevx_op(ctx, n, n, dh, nband, de, dv)
    ctx.synchronize()
    return de.cpu().numpy(), dv.cpu().numpy().T[:, :nband]


def _check(H, e, V):
    w = np.linalg.eigvalsh(H)
    scale = max(1.0, np.abs(w).max())
    assert np.abs(e - w[: len(e)]).max() < 1e-12 * scale
    assert np.abs(H @ V - V * e).max() < 1e-11 * scale
    assert np.abs(V.conj().T @ V - np.eye(len(e))).max() < 1e-11


def _hermitian(n, seed):
    rng = np.random.default_rng(seed)
    H = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    return H + H.conj().T


# rows per lane change at multiples of 64, columns per wave at multiples of 128, the device-wide
# start at 513; 514 leaves one column's step to it, 704 and 705 are its two forms
@pytest.mark.parametrize("n", [2, 3, 5, 63, 64, 65, 127, 128, 129, 192, 193, 256, 257, 320, 321, 384, 385, 448, 449,
                               511, 512, 513, 514, 576, 704, 705])
def test_size_classes(torch, n):
    from apw import pw
    ctx = pw.Context(0)
    H = _hermitian(n, n)
    _check(H, *_solve(torch, ctx, H, max(1, n // 4)))
    ctx.close()


@pytest.mark.parametrize("n,m", [(40, 0), (130, 0), (130, 70), (530, 9)])
def test_columns_without_reflector(torch, n, m):
    """A diagonal matrix with a dense m x m block: zero columns (tau = 0) around real ones."""
    from apw import pw
    ctx = pw.Context(0)
    H = np.diag(np.linspace(-3.0, 5.0, n)).astype(complex)
    H[n - m:, n - m:] += _hermitian(m, 7) * 0.1
    _check(H, *_solve(torch, ctx, H, n // 3))
    ctx.close()


def test_streams_at_once(torch):
    """Reductions of several contexts in flight together, of one-XCD and device-wide sizes, give
    what each gives alone."""
    from apw import pw
    sizes = [(96, 0), (200, 1), (512, 2), (600, 3), (200, 4), (48, 5)]
    mats = [_hermitian(n, 100 + s) for n, s in sizes]
    ctx = [pw.Context(0) for _ in sizes]
    alone = [_solve(torch, c, H, 12) for c, H in zip(ctx, mats)]
    got = [None] * len(sizes)

    def work(i):
        for _ in range(4):
            got[i] = _solve(torch, ctx[i], mats[i], 12)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    [t.start() for t in threads]
    [t.join() for t in threads]
    for a, g in zip(alone, got):
        assert np.array_equal(a[0], g[0]) and np.array_equal(a[1], g[1])
    [c.close() for c in ctx]


def test_contexts_come_and_go(torch):
    """A destroyed stream's reductions are forgotten: later ones on other streams are not held up
    or failed by them."""
    from apw import pw
    H = _hermitian(70, 3)
    keep = pw.Context(0)
    want = _solve(torch, keep, H, 10)
    for _ in range(20):
        ctx = pw.Context(0)
        e, V = _solve(torch, ctx, H, 10)
        ctx.close()
        assert np.array_equal(e, want[0]) and np.array_equal(V, want[1])
        assert np.array_equal(_solve(torch, keep, H, 10)[0], want[0])
    keep.close()


@pytest.mark.parametrize("n", [48, 130])
def test_stream_kept_to_half_of_the_cus(torch, n):
    """On a caller's stream with a CU mask the workgroups of one XCD need not be resident together:
    such a context takes the device-wide reduction (12 and 32 workgroups here)."""
    import ctypes as C
    from apw import pw
    torch.zeros(1, device="cuda")
    hip = C.CDLL("libamdhip64.so")
    stream = C.c_void_p()
    mask = (C.c_uint32 * 8)(*([0xffffffff] * 4 + [0] * 4))
    assert hip.hipExtStreamCreateWithCUMask(C.byref(stream), 8, mask) == 0
    H = _hermitian(n, n)
    ctx = pw.Context(0, stream=stream.value)
    _check(H, *_solve(torch, ctx, H, n // 4))
    ctx.close()
    assert hip.hipStreamDestroy(stream) == 0

"""The pipelined FP64 and FP32 products against numpy at the edges of their tiles: m and n around
64 and 16, k around the step of 8 (c64: 16) and the three stages, every op pair, split and
unsplit, leading dimensions with NaN in the padding (which no result may meet), odd ones, and
operands aligned to half an element."""
import json

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a GPU"
    return t


@pytest.fixture()
def tuner():
    from apw import pw
    pw.tune_clear()
    yield pw
    pw.tune_set_mode(pw.TUNE_FIXED)
    pw.tune_clear()


class _At:
    """Device memory at a byte offset into a tensor."""
    dtype = None

    def __init__(self, t, off):
        self.t, self.off = t, off

    def data_ptr(self):
        return self.t.data_ptr() + self.off


def _check(torch, pw, ops, m, n, k, pad, half=False, single=False, alpha=0.7 - 0.2j, beta=0.3 + 0.1j):
    real, cplx = (np.float32, np.complex64) if single else (np.float64, np.complex128)
    off = int(half)                              # in reals
    ctx = pw.Context(0)
    rng = np.random.default_rng(1000 * m + 10 * n + k)

    def crand(*shape):
        return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(cplx)

    def operand(op, rows, cols):                 # op(X) is rows x cols; stored column-major, padded
        r, c = (rows, cols) if op == "N" else (cols, rows)
        x = crand(c, r)
        full = np.full((c, r + pad), np.nan + 1j * np.nan, dtype=cplx)
        full[:, :r] = x
        flat = torch.from_numpy(full.reshape(-1).view(real)).cuda()
        buf = torch.full((flat.numel() + 2,), float("nan"), dtype=flat.dtype, device="cuda")
        buf[off: off + flat.numel()] = flat
        x = x.astype(np.complex128)
        y = x.T if op == "N" else x
        return (y.conj() if op == "C" else y), _At(buf, off * flat.element_size()), r + pad

    a, da, lda = operand(ops[0], m, k)
    b, db, ldb = operand(ops[1], k, n)
    c0 = crand(n, m + pad)
    dc = torch.from_numpy(c0).cuda()
    pw.gemm_op(ctx, ops[0], ops[1], m, n, k, alpha, da, lda, db, ldb, beta, dc, m + pad)
    ctx.synchronize()
    got = dc.cpu().numpy()
    ctx.close()
    want = alpha * (a @ b) + beta * c0[:, :m].T
    mag = abs(alpha) * (np.abs(a) @ np.abs(b)) + abs(beta) * np.abs(c0[:, :m].T)
    # the three-product form sums terms of up to twice the size: 8 eps per term, added at random
    assert (np.abs(got[:, :m].T - want) <= 8 * np.sqrt(k) * np.finfo(real).eps * mag).all(), (ops, m, n, k)
    assert np.array_equal(got[:, m:], c0[:, m:])     # nothing past the m rows


@pytest.mark.parametrize("ops", ["NN", "NT", "NC", "TN", "TT", "TC", "CN", "CT", "CC"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (64, 64, 8), (65, 17, 23), (63, 33, 40), (130, 49, 33), (127, 81, 57),
                                   (66, 50, 129)])
@pytest.mark.parametrize("single", [False, True])
def test_edges(torch, tuner, ops, m, n, k, single):
    _check(torch, tuner, ops, m, n, k, pad=3, single=single)
    _check(torch, tuner, ops, m, n, k, pad=0, single=single)


@pytest.mark.parametrize("ops,m,n,k", [("CN", 64, 24, 2371), ("CN", 129, 97, 5003), ("NN", 1000, 130, 77),
                                       ("NN", 8197, 193, 129), ("CN", 33, 16, 128), ("CC", 70, 66, 1025)])
@pytest.mark.parametrize("plan", [None, (12, 0), (12, 1), (12, 3), (13, 0), (13, 2)])
@pytest.mark.parametrize("single", [False, True])
def test_plans(torch, tuner, tmp_path, ops, m, n, k, plan, single):
    pw = tuner
    if plan:
        pw.tune_set_mode(pw.TUNE_MEASURE)
        _check(torch, pw, ops, m, n, k, pad=0, single=single)
        (key, _, _), = pw.tune_entries()
        path = tmp_path / "plan.json"
        entry = json.dumps({"key": key, "choice": list(plan), "us": 1.0})
        path.write_text('{"version": 1, "entries": [\n' + entry + "\n]}\n")
        pw.tune_clear()
        assert pw.tune_load(str(path)) == 1
        pw.tune_set_mode(pw.TUNE_CACHE)
    _check(torch, pw, ops, m, n, k, pad=1, single=single)


@pytest.mark.parametrize("ops,m,n,k", [("CN", 65, 33, 1000), ("NN", 333, 20, 41)])
@pytest.mark.parametrize("single", [False, True])
def test_half_aligned(torch, tuner, ops, m, n, k, single):
    _check(torch, tuner, ops, m, n, k, pad=1, half=True, single=single)


def test_many_columns(torch, tuner):
    """More n-tiles than a grid's second dimension holds."""
    _check(torch, tuner, "NN", 2, 65535 * 64 + 70, 3, pad=0)


@pytest.mark.parametrize("m,n,k", [(541, 13, 7106), (64, 64, 72), (300, 100, 40000)])
@pytest.mark.parametrize("single", [False, True])
def test_same_bits(torch, tuner, m, n, k, single):
    """Repeated calls with other work between them: every fill of LDS is waited for."""
    pw = tuner
    ctx = pw.Context(0)
    g = torch.Generator(device="cuda").manual_seed(5)
    dt = torch.complex64 if single else torch.complex128
    a, b = (torch.randn(r, k, dtype=dt, generator=g, device="cuda") for r in (m, n))
    outs = []
    for i in range(40):
        c = torch.zeros((n, m), dtype=dt, device="cuda")
        pw.gemm_op(ctx, "C", "N", m, n, k, 1.0, a, k, b, k, 0.0, c, m)
        if i % 3 == 0:
            torch.randn(1 << 22, device="cuda").sum()
        outs.append(c)
    ctx.synchronize()
    ctx.close()
    want = (b.to(torch.complex128).cpu().numpy() @ a.to(torch.complex128).cpu().numpy().conj().T)
    got = outs[0].to(torch.complex128).cpu().numpy()
    eps = np.finfo(np.float32 if single else np.float64).eps
    assert np.abs(got - want).max() <= 8 * eps * np.sqrt(k) * 2 * np.sqrt(k)
    assert all(torch.equal(o, outs[0]) for o in outs[1:])


# splits of 32 to 63 of k: up to one workgroup a CU (256), the last split short
@pytest.mark.parametrize("ops", ["CN", "NN", "TC"])
@pytest.mark.parametrize("m,n,k", [(5, 3, 128), (96, 96, 700), (130, 33, 161), (512, 96, 1031), (1000, 1000, 255)])
@pytest.mark.parametrize("single", [False, True])
def test_short_splits(torch, tuner, ops, m, n, k, single):
    _check(torch, tuner, ops, m, n, k, pad=1, single=single)


# tall products on either side of the line between the two orders of tiles
@pytest.mark.parametrize("m,n,k", [(33000, 193, 32), (33000, 193, 33), (33000, 129, 24), (33000, 128, 24)])
@pytest.mark.parametrize("single", [False, True])
def test_orders_of_tall_products(torch, tuner, m, n, k, single):
    _check(torch, tuner, "NN", m, n, k, pad=1, single=single)

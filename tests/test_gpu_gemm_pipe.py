"""The pipelined FP64 product against numpy at the edges of its tiles: m and n around 64 and
16, k around the step of 8 and the three stages, every op pair, split and unsplit, leading
dimensions with NaN in the padding (which no result may meet), and operands that are only
8-byte aligned (another kernel)."""
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

    def __init__(self, t, off=0):
        self.t, self.off = t, off

    def data_ptr(self):
        return self.t.data_ptr() + self.off


def _check(torch, pw, ops, m, n, k, pad, off=0, alpha=0.7 - 0.2j, beta=0.3 + 0.1j):
    ctx = pw.Context(0)
    rng = np.random.default_rng(1000 * m + 10 * n + k)

    def operand(op, rows, cols):                 # op(X) is rows x cols; stored column-major, padded
        r, c = (rows, cols) if op == "N" else (cols, rows)
        x = rng.standard_normal((c, r)) + 1j * rng.standard_normal((c, r))
        full = np.full((c, r + pad), np.nan + 1j * np.nan)
        full[:, :r] = x
        buf = torch.full((full.size * 2 + 2,), float("nan"), dtype=torch.float64, device="cuda")
        flat = torch.from_numpy(full.reshape(-1).view(np.float64)).cuda()
        buf[off // 8: off // 8 + flat.numel()] = flat
        y = x.T if op == "N" else x
        return (y.conj() if op == "C" else y), _At(buf, off), r + pad

    a, da, lda = operand(ops[0], m, k)
    b, db, ldb = operand(ops[1], k, n)
    c0 = rng.standard_normal((n, m + pad)) + 1j * rng.standard_normal((n, m + pad))
    dc = torch.from_numpy(c0).cuda()
    pw.gemm_op(ctx, ops[0], ops[1], m, n, k, alpha, da, lda, db, ldb, beta, dc, m + pad)
    ctx.synchronize()
    got = dc.cpu().numpy()
    ctx.close()
    want = alpha * (a @ b) + beta * c0[:, :m].T
    mag = abs(alpha) * (np.abs(a) @ np.abs(b)) + abs(beta) * np.abs(c0[:, :m].T)
    # the three-product form sums terms of up to twice the size: 8 eps per term, added at random
    assert (np.abs(got[:, :m].T - want) <= 8 * np.sqrt(k) * np.finfo(float).eps * mag).all(), (ops, m, n, k)
    assert np.array_equal(got[:, m:], c0[:, m:])     # nothing past the m rows


@pytest.mark.parametrize("ops", ["NN", "NT", "NC", "TN", "TT", "TC", "CN", "CT", "CC"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (64, 64, 8), (65, 17, 23), (63, 33, 40), (130, 49, 33), (127, 81, 57)])
def test_edges(torch, tuner, ops, m, n, k):
    _check(torch, tuner, ops, m, n, k, pad=3)


@pytest.mark.parametrize("ops,m,n,k", [("CN", 64, 24, 2371), ("CN", 129, 97, 5003), ("NN", 1000, 130, 77),
                                       ("NN", 8197, 193, 129), ("CN", 33, 16, 128), ("CC", 70, 66, 1025)])
@pytest.mark.parametrize("plan", [None, (12, 0), (12, 1), (12, 3), (13, 0), (13, 2)])
def test_plans(torch, tuner, tmp_path, ops, m, n, k, plan):
    pw = tuner
    if plan:
        pw.tune_set_mode(pw.TUNE_MEASURE)
        _check(torch, pw, ops, m, n, k, pad=0)
        (key, _, _), = pw.tune_entries()
        path = tmp_path / "plan.json"
        entry = json.dumps({"key": key, "choice": list(plan), "us": 1.0})
        path.write_text('{"version": 1, "entries": [\n' + entry + "\n]}\n")
        pw.tune_clear()
        assert pw.tune_load(str(path)) == 1
        pw.tune_set_mode(pw.TUNE_CACHE)
    _check(torch, pw, ops, m, n, k, pad=1)


@pytest.mark.parametrize("ops,m,n,k", [("CN", 65, 33, 1000), ("NN", 333, 20, 41)])
def test_8_byte_aligned(torch, tuner, ops, m, n, k):
    _check(torch, tuner, ops, m, n, k, pad=1, off=8)

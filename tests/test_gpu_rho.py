"""The density pass over more bands than one launch takes, and its workspace: one of bounded size
for the Hamiltonians of a context, and less where the memory is not there."""
import functools
import threading
from types import SimpleNamespace

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GIB = 1 << 30


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a GPU"
    return t


@functools.lru_cache(maxsize=None)
def _basis(ecut=50.0):
    """64-atom cell, 96^3 grid: 9 MB of intermediates a band, some 340 bands in 3 GiB."""
    from apw.basis import Lattice, PWBasisK
    return PWBasisK(Lattice(10.26, np.diag([2.0, 2.0, 2.0])), ecut, 96, 96, 96, kvec_d=np.zeros((1, 3)))


def _ham(pw, ctx, b):
    npw = int(b.npwk[0])
    return pw.HamiltPW(ctx, SimpleNamespace(
        npw=npw, npwx=npw, nx=b.nx, ny=b.ny, nz=b.nz, tpiba2=float(b.tpiba2), gk2=b.gk2[0, :npw],
        ig2ixyz=b.ig2ixyz_k[0, :npw], veff=np.zeros(b.nxyz), vkb=np.zeros((0, npw), complex),
        deeq=np.zeros((1, 0, 8, 8)), na=np.array([0]), nh=np.array([8])))


def _bands(torch, b, nb, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((nb, int(b.npwk[0]), 2), generator=g, device="cuda", dtype=torch.float64)
    return torch.view_as_complex(x)


def _reference(torch, b, psi, wg, omega):
    npw = int(b.npwk[0])
    idx = torch.from_numpy(np.ascontiguousarray(b.ig2ixyz_k[0, :npw])).cuda().long()
    rho = torch.zeros(b.nxyz, dtype=torch.float64, device="cuda")
    box = torch.zeros(b.nxyz, dtype=torch.complex128, device="cuda")
    for v, w in zip(psi, wg):
        box.zero_()
        box[idx] = v
        r = torch.fft.ifftn(box.view(b.nx, b.ny, b.nz)) * b.nxyz
        rho += w / omega * torch.view_as_real(r).square().sum(-1).reshape(-1)
    return rho


def _close(torch, got, want, nb):
    # every term is positive: the bound of an FFT of 3 log2(96) levels and a sum over the bands
    return float((got - want).abs().max() / want.abs().max()) < (8 * 20 + nb) * np.finfo(float).eps


def test_more_bands_than_a_launch(torch):
    from apw import pw
    b, nb = _basis(), 700
    ctx = pw.Context(0)
    ham = _ham(pw, ctx, b)
    psi, wg = _bands(torch, b, nb, 1), np.linspace(0.5, 2.0, nb)
    rho = ham.psi_to_rho(psi, nb, wg, b.lat.omega)
    ctx.synchronize()
    want = _reference(torch, b, psi, wg, b.lat.omega)
    assert _close(torch, rho, want, nb)
    # accumulated on top, from work arrays full of NaN
    ctx.fill_workspaces(float("nan"))
    ham.psi_to_rho(psi, nb, wg, b.lat.omega, rho=rho, add=True)
    ctx.synchronize()
    assert _close(torch, rho, 2.0 * want, 2 * nb)
    ham.close()
    ctx.close()


def test_workspace_is_the_contexts(torch):
    """A second Hamiltonian's density takes no gigabytes of its own, and the context's go with it."""
    from apw import pw
    b, nb = _basis(), 320
    psi, wg = _bands(torch, b, nb, 2), np.ones(nb)
    rho = torch.zeros(b.nxyz, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    ctx = pw.Context(0)
    hams = [_ham(pw, ctx, b) for _ in range(3)]
    used = []
    for h in hams:
        free = torch.cuda.mem_get_info()[0]
        h.psi_to_rho(psi, nb, wg, b.lat.omega, rho=rho)
        ctx.synchronize()
        used.append(free - torch.cuda.mem_get_info()[0])
    assert used[0] <= 3.1 * GIB and max(used[1:]) < 0.2 * GIB, used
    [h.close() for h in hams]
    ctx.close()
    assert before - torch.cuda.mem_get_info()[0] < 0.5 * GIB


@pytest.mark.skip(reason="with a failing allocation in the call, this ended in a segmentation fault inside the runtime "
                         "once, late in a run of all tests; the cause is not known.  tests/test_rho_bands.py has the rule")
def test_little_memory(torch):
    """With two gigabytes left the density is formed with fewer bands a launch."""
    from apw import pw
    b, nb = _basis(), 320
    psi, wg = _bands(torch, b, nb, 3), np.ones(nb)
    want = _reference(torch, b, psi, wg, b.lat.omega)
    rho = torch.zeros(b.nxyz, dtype=torch.float64, device="cuda")
    ctx = pw.Context(0)
    ham = _ham(pw, ctx, b)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    rest = torch.empty(torch.cuda.mem_get_info()[0] - 2 * GIB, dtype=torch.uint8, device="cuda")
    try:
        print(f"free {torch.cuda.mem_get_info()[0] / GIB:.2f} GiB", flush=True)
        ham.psi_to_rho(psi, nb, wg, b.lat.omega, rho=rho)
        ctx.synchronize()
    finally:
        del rest
        torch.cuda.empty_cache()
    assert _close(torch, rho, want, nb)
    ham.close()
    ctx.close()


def test_two_threads_on_one_context(torch):
    from apw import pw
    b, nb = _basis(), 60
    ctx = pw.Context(0)
    hams = [_ham(pw, ctx, b) for _ in range(2)]
    psi = [_bands(torch, b, nb, 4 + i) for i in range(2)]
    rho = [torch.zeros(b.nxyz, dtype=torch.float64, device="cuda") for _ in range(2)]
    want = [_reference(torch, b, p, np.ones(nb), b.lat.omega) for p in psi]

    def work(i):
        for _ in range(6):
            hams[i].psi_to_rho(psi[i], nb, np.ones(nb), b.lat.omega, rho=rho[i])

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    ctx.synchronize()
    assert all(_close(torch, r, w, nb) for r, w in zip(rho, want))
    [h.close() for h in hams]
    ctx.close()

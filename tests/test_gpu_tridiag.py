"""Hermitian eigensolver at the edges of its kernels: the one-wave Jacobi kernel
(n <= 16) and, through the divide and conquer, the Householder tridiagonalisations
(register-resident n <= 256, spread over many workgroups and panels above), on
structured matrices and on both sides of each batch rule."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng(gpu_lib):
    from muspinsim_amd.engine import SpinEngine
    return SpinEngine("cuda:0")


def _herm(rng, n):
    X = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    return (X + X.conj().T) / 2


def _check(eng, Hs, method=None):
    """Backward error of order n eps ||H|| and orthonormal eigenvectors; the
    strict upper triangle, which the solver must not read, is NaN."""
    from muspinsim_amd import _native as N
    n = Hs.shape[1]
    low = Hs.copy()
    low[:, np.triu_indices(n, 1)[0], np.triu_indices(n, 1)[1]] = np.nan
    E, U, info = eng.eigh(torch.as_tensor(low).cuda(),
                          method=N.MSP_EIGH_DC if method is None else method)
    assert np.all(info.cpu().numpy() == 0)
    _accurate(Hs, E.cpu().numpy(), U.cpu().numpy())


def _accurate(Hs, E, U):
    n = Hs.shape[1]
    nrm = np.maximum(np.abs(E).max(1), 1e-300)
    assert np.all(np.abs(E - np.linalg.eigvalsh(Hs)).max(1) <= 1e-14 * n * nrm)
    assert np.all(np.abs(Hs @ U - U * E[:, None, :]).max((1, 2)) <= 1e-14 * n * nrm)
    UU = np.conj(np.swapaxes(U, 1, 2)) @ U
    assert np.abs(UU - np.eye(n)).max() <= 1e-14 * max(n, 10)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 8, 9, 11, 12, 13, 15, 16, 17, 24, 25, 31, 32, 33, 48, 49, 64, 65,
                               80, 81, 95, 96, 97, 108, 112, 113, 127, 128, 129, 160, 161, 191,
                               192, 193, 200, 223, 224, 225, 255, 256, 257])
def test_structured(eng, n):
    rng = np.random.default_rng(n)
    tri = np.diag(rng.normal(size=n)) + 0j
    i = np.arange(n - 1)
    tri[i + 1, i] = rng.normal(size=n - 1) + 1j * rng.normal(size=n - 1)
    tri[i, i + 1] = np.conj(tri[i + 1, i])
    v = rng.normal(size=n) + 1j * rng.normal(size=n)
    half = np.zeros((n, n), dtype=complex)     # two uncoupled blocks: a zero column on the way
    m = n // 2
    half[:m, :m], half[m:, m:] = _herm(rng, m), _herm(rng, n - m)
    Hs = np.array([_herm(rng, n), 1e6 * _herm(rng, n), np.zeros((n, n)) + 0j,
                   np.diag(rng.normal(size=n)) + 0j, tri, np.outer(v, v.conj()),
                   _herm(rng, n).real + 0j, half,
                   1e-120 * _herm(rng, n), 1e120 * _herm(rng, n)])
    _check(eng, Hs)
    if n <= 16:
        from muspinsim_amd import _native as N
        _check(eng, Hs, N.MSP_EIGH_AUTO)
        _check(eng, Hs[:1], N.MSP_EIGH_AUTO)


@pytest.mark.parametrize("n", [40, 90])
@pytest.mark.parametrize("batch", [512, 513])
def test_batch_rule(eng, n, batch):
    rng = np.random.default_rng(n + batch)
    _check(eng, np.array([_herm(rng, n) for _ in range(batch)]))


@pytest.mark.parametrize("n", [257, 264, 265, 319, 320, 321, 384, 511, 513, 700, 1023, 1024])
def test_few_large(eng, n):
    rng = np.random.default_rng(n)
    v = rng.normal(size=n) + 1j * rng.normal(size=n)
    half = np.zeros((n, n), dtype=complex)
    m = n // 2
    half[:m, :m], half[m:, m:] = _herm(rng, m), _herm(rng, n - m)
    for Hs in ([_herm(rng, n)], [half, np.diag(rng.normal(size=n)) + 0j, np.outer(v, v.conj())]):
        _check(eng, np.array(Hs))


@pytest.mark.parametrize("n", [1, 2, 4, 5, 8, 9, 16])
def test_small_non_finite(eng, n):
    """n <= 16: a matrix with a NaN or infinite entry reports info != 0 with NaN
    eigenvalues and vectors; the matrices that share its wave are unaffected."""
    from muspinsim_amd import _native as N
    rng = np.random.default_rng(n)
    good = np.array([_herm(rng, n) for _ in range(16)])
    Hs = good.copy()
    bad = {1: (n - 1, 0, np.nan), 4: (0, 0, np.nan), 6: (n - 1, n - 1, np.inf),
           9: (n - 1, 0, -np.inf), 15: (n // 2, 0, complex(0.0 if n > 1 else np.nan, np.nan))}
    for k, (i, j, x) in bad.items():
        Hs[k, i, j] = x
    for method in (N.MSP_EIGH_DC, N.MSP_EIGH_AUTO):
        E0, U0, _ = eng.eigh(torch.as_tensor(good).cuda(), method=method)
        E, U, info = eng.eigh(torch.as_tensor(Hs).cuda(), method=method)
        for k in range(len(Hs)):
            if k in bad:
                assert int(info[k]) != 0
                assert torch.isnan(E[k]).all() and torch.isnan(torch.view_as_real(U[k])).all()
            else:
                assert int(info[k]) == 0
                assert torch.equal(E[k], E0[k]) and torch.equal(U[k], U0[k])


@pytest.mark.parametrize("n,sweeps", [(8, 7), (12, 8), (16, 8)])
def test_small_norms(eng, n, sweeps):
    """Rotations of the n <= 16 solver are unit to within rounding: a vector goes
    through n - 1 of them per sweep, so its squared norm is off by at most about
    eps / 2 times the root of their number (rms; a biased rotation adds up to
    their number instead, twice as much here)."""
    from muspinsim_amd import _native as N
    rng = np.random.default_rng(n)
    X = rng.normal(size=(4000, n, n)) + 1j * rng.normal(size=(4000, n, n))
    _, U, _ = eng.eigh(torch.as_tensor(X + X.conj().swapaxes(1, 2)).cuda(), method=N.MSP_EIGH_DC)
    U = U.cpu().numpy()
    off = (U.real.astype(np.longdouble) ** 2 + U.imag.astype(np.longdouble) ** 2).sum(1) - 1
    assert np.sqrt(float((off ** 2).mean())) <= 1.4 * 2.0 ** -53 * np.sqrt(sweeps * (n - 1))


@pytest.mark.parametrize("n,batch", [(257, 32), (257, 33), (512, 96), (512, 97), (513, 96), (513, 97),
                                     (1023, 193), (1024, 192), (1024, 193)])
def test_large_batch_rule(eng, n, batch):
    """Both sides of the line between the spread reduction (batch <= 192 and 4
    batch <= n - 128) and the panel kernel (panels in LDS up to n = 512, in the
    workspace above): three matrices in turn, checked once, every copy alike."""
    from muspinsim_amd import _native as N
    rng = np.random.default_rng(n)
    H = np.array([_herm(rng, n) for _ in range(2)] + [np.diag(rng.normal(size=n)) + 0j])
    k = torch.arange(batch, device="cuda") % 3
    low = np.where(np.tri(n, dtype=bool), H, np.nan)
    E, U, info = eng.eigh(torch.as_tensor(low).cuda()[k], method=N.MSP_EIGH_DC)
    assert int(info.abs().max()) == 0
    assert torch.equal(E, E[:3][k])
    for b in range(3, batch):
        assert torch.equal(U[b], U[b % 3])
    _accurate(H, E[:3].cpu().numpy(), U[:3].cpu().numpy())


def test_large_on_two_streams(eng):
    """Two spread reductions side by side on two streams, each with its own
    workspace, as dimension groups of one plan run them."""
    from muspinsim_amd import _native as N
    rng = np.random.default_rng(5)
    Hs = [torch.as_tensor(np.array([_herm(rng, n) for _ in range(4)])).cuda() for n in (300, 420)]
    alone = [eng.eigh(H.clone(), method=N.MSP_EIGH_DC) for H in Hs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in Hs]
    for _ in range(3):
        out = []
        for s, H in zip(streams, Hs):
            with torch.cuda.stream(s):
                out.append(eng.eigh(H.clone(), method=N.MSP_EIGH_DC))
        torch.cuda.synchronize()
        for (E, U, _), (E0, U0, _) in zip(out, alone):
            assert torch.equal(E, E0) and torch.equal(U, U0)

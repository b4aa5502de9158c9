"""Mode decomposition of general complex matrices (msp_lindblad_modes without
eigenvectors) against numpy's eigendecomposition: sizes around the LDS form's
limits, numbers of operators on both sides of its limit, and matrices with zero
reflectors, early deflation, exceptional shifts and extreme scales."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng(gpu_lib):
    from muspinsim_amd.engine import SpinEngine
    return SpinEngine("cuda:0")


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a, dtype=complex)).cuda()


def _matrices(rng, N):
    G = rng.normal(size=(N, N)) + 1j * rng.normal(size=(N, N))
    D = np.diag(np.arange(1, N + 1) * (0.1 + 0.2j))
    block = G.copy()
    block[N // 2:, : N // 2] = 0.0
    cyc = np.roll(np.eye(N), 1, axis=0) + 0j       # every Wilkinson shift starts at zero
    return [G, G + G.conj().T, -1j * (G + G.conj().T), D, D + np.triu(G, 1) / N, block, cyc,
            1e100 * G, 1e-100 * G]


@pytest.mark.parametrize("N", [4, 8, 9, 10, 16, 17, 36, 63, 64, 65])
def test_amplitudes(eng, N):
    rng = np.random.default_rng(N)
    Ms = np.array(_matrices(rng, N))
    for k in (1, 2, 3, 4):
        r = rng.normal(size=(len(Ms), N)) + 1j * rng.normal(size=(len(Ms), N))
        u = rng.normal(size=(len(Ms), k, N)) + 1j * rng.normal(size=(len(Ms), k, N))
        lam, amp, c, _ = eng.lindblad_modes(_dev(Ms), _dev(r), _dev(u), want_c=True)
        lam, amp = lam.cpu().numpy(), amp.cpu().numpy()
        for b, M in enumerate(Ms):
            w, V = np.linalg.eig(M)
            cond = np.linalg.cond(V)
            if cond > 1e6:
                continue
            s = np.abs(M).max()
            # backward error of order N eps ||M||: eigenvalues to cond(V) times it
            tol = 1e-15 * N * N * cond
            assert np.abs(np.sort_complex(np.round(lam[b] / s, 9)) -
                          np.sort_complex(np.round(w / s, 9))).max() <= max(tol, 3e-9)
            # u^T f(M) r is independent of order and scaling of the modes
            ref = np.linalg.solve(V, r[b])
            for f in (lambda x: np.exp(x / s / N), lambda x: 1.0 / (x / s - 3.0j * N)):
                want = (u[b] @ V) @ (ref * f(w))
                got = amp[b] @ f(lam[b])
                scale = np.abs(u[b]).sum(1) * np.abs(r[b]).max() * np.abs(f(w)).max()
                assert np.all(np.abs(got - want) <= tol * scale)


def test_zero_matrix_and_no_operators(eng):
    N = 16
    r = np.ones((1, N))
    lam, _, c, _ = eng.lindblad_modes(_dev(np.zeros((1, N, N))), _dev(r), None, want_c=True)
    assert np.all(lam.cpu().numpy() == 0) and np.allclose(c.cpu().numpy(), r)


@pytest.mark.parametrize("N", [9, 16, 36, 64])
def test_eigenvalue_rounding(eng, N):
    """Rotations of the QR sweeps are unit to within rounding: an eigenvalue of a
    normal matrix goes through two per sweep and about 2.5 N sweeps, so it is off
    by about eps / 2 times the root of their number (rms, relative to the norm;
    biased rotations add up to their number instead)."""
    rng = np.random.default_rng(N)
    G = rng.normal(size=(200, N, N)) + 1j * rng.normal(size=(200, N, N))
    G = G + np.conj(np.swapaxes(G, 1, 2))
    one = np.ones((200, N))
    lam, _, _, _ = eng.lindblad_modes(_dev(1j * G), _dev(one), _dev(one[:, None]))
    lam = lam.cpu().numpy()
    ref = np.linalg.eigvalsh(G)
    scale = np.abs(ref).max(1, keepdims=True)
    err = np.sqrt((((np.sort(lam.imag, 1) - ref) / scale) ** 2).mean())
    assert err <= 2.0 ** -53 * np.sqrt(2 * 2.5 * N)
    assert np.sqrt(((lam.real / scale) ** 2).mean()) <= 2.0 ** -53 * np.sqrt(2 * 2.5 * N)


@pytest.mark.parametrize("N", [16, 20, 21])
@pytest.mark.parametrize("nb", [2048, 2049])
def test_batch_rule(eng, N, nb):
    """Both sides of the batch rule up to N = 20: four normal matrices in turn
    (condition 1), each copy against numpy."""
    rng = np.random.default_rng(N)
    G = rng.normal(size=(4, N, N)) + 1j * rng.normal(size=(4, N, N))
    G = G + np.conj(np.swapaxes(G, 1, 2))
    r = rng.normal(size=(4, N)) + 1j * rng.normal(size=(4, N))
    u = rng.normal(size=(4, 2, N)) + 1j * rng.normal(size=(4, 2, N))
    k = np.arange(nb) % 4
    lam, amp, _, _ = eng.lindblad_modes(_dev(1j * G[k]), _dev(r[k]), _dev(u[k]))
    w, V = np.linalg.eigh(G)
    s = np.abs(w).max()
    want = np.einsum("bqi,bim,bm,bjm,bj->bq", u, V, np.exp(1j * w / s), V.conj(), r)
    got = (amp.cpu().numpy() * np.exp(lam.cpu().numpy() / s)[:, None]).sum(2)
    tol = 1e-15 * N * N * np.linalg.norm(r, axis=1).max() * np.linalg.norm(u, axis=2).max()
    assert np.abs(got - want[k]).max() <= tol

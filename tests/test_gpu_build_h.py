"""Hamiltonian build from the terms against the oracle: an element per thread, and
with packed spin digits one or several (4 < n <= 32, and n > 256 with many
elements), on both sides of each rule, digits up to the packed limit of 15 and above it, full
matrices and lower triangles."""

import numpy as np
import pytest
import torch

from oracle import physics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lower", [False, True])
@pytest.mark.parametrize("Is,nb", [([0.5], 1), ([0.5, 0.5], 3), ([2.0], 3), ([7.5], 3), ([8.0], 3),
                                   ([0.5, 1.5], 1024), ([0.5, 1.5], 1025), ([0.5, 0.5, 1.0, 0.5], 9),
                                   ([0.5, 7.0], 9000), ([0.5] * 5, 1023), ([0.5] * 5, 1024),
                                   ([0.5, 8.0], 1030),
                                   ([0.5, 0.5, 1.5], 9000), ([0.5, 1.0, 0.5], 5000), ([0.5] * 8, 3),
                                   ([0.5] * 8, 40), ([0.5, 3.5, 0.5, 1.0], 70), ([7.5, 0.5], 600),
                                   ([0.5, 8.5], 600),
                                   # from 32,768 workgroups of 256 elements on
                                   ([0.5, 1.0, 1.0, 2.5, 1.0], 79), ([0.5, 1.0, 1.0, 2.5, 1.0], 80),
                                   ([0.5, 8.5, 3.5], 102), ([0.5] * 9, 31), ([0.5] * 9, 32)])
def test_from_terms(gpu_lib, Is, nb, lower):
    from muspinsim_amd import _native as N
    from muspinsim_amd.engine import SpinEngine, SystemDesc, pack_systems
    rng = np.random.default_rng(len(Is) + nb)
    systems = []
    for _ in range(2):
        terms = [("linear", 0, 0, rng.normal(size=3))]
        for i in range(len(Is)):
            for j in range(i if Is[i] >= 1 else i + 1, len(Is)):
                M = rng.normal(size=(3, 3)) * 10
                M[rng.random((3, 3)) < 0.2] = 0.0
                terms.append(("bilinear", i, j, (M + M.T) / 2 if i == j else M))
        systems.append(SystemDesc(Is=list(Is), gammas=list(rng.normal(size=len(Is)) * 100),
                                  terms=terms))
    eng = SpinEngine("cuda:0")
    n = systems[0].n
    sysarr, termarr = pack_systems(systems)
    dsys, dterms = eng._bytes_view(sysarr), eng._bytes_view(termarr)
    B = rng.normal(size=(3, 3))
    sid = torch.as_tensor(np.arange(nb, dtype=np.int32) % 2).cuda()
    Br = torch.as_tensor(B[np.arange(nb) % 3]).cuda()
    H = torch.full((nb, n, n), float("nan"), dtype=torch.complex128, device="cuda")
    fn = gpu_lib.msp_build_h_lower if lower else gpu_lib.msp_build_h
    N.check(fn(n, nb, dsys.data_ptr(), dterms.data_ptr(), sid.data_ptr(), Br.data_ptr(), None, 1,
               H.data_ptr(), eng.stream()))
    H = H.cpu().numpy()
    part = np.tril_indices(n) if lower else np.indices((n, n)).reshape(2, -1)
    for k in range(min(nb, 6)):
        S = systems[k % 2]
        ref = physics.hamiltonian(S.Is, S.terms) + physics.zeeman(S.Is, S.gammas, B[k % 3])
        # at most 9 products per pair of spins, each rounded a few times
        assert np.abs((H[k] - ref)[part[0], part[1]]).max() <= 1e-15 * 9 * len(Is) ** 2 * np.abs(ref).max()
        for m in range(k, nb, 6):
            assert np.array_equal(H[m], H[k], equal_nan=True)

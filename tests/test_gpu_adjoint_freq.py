"""Frequency sums of the adjoint, R_jk = sum_t r cos w_jk t and S_jk = sum_t r t
sin w_jk t, against numpy at the edges of the two kernels' tiles (16 x 16 and 64
times for few instances, 64 x 64 and 8 times for many) and on both sides of the
rule between them."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nt", [(1, 5), (3, 1), (15, 8), (16, 9), (17, 16), (48, 17), (63, 40),
                                  (64, 33), (65, 7), (80, 24), (128, 15), (130, 31), (16, 0)])
@pytest.mark.parametrize("nb", [3, 0])
def test_frequency_sums(gpu_lib, n, nt, nb):
    """nb = 0: the smallest batch of the matrix form, and one below it."""
    if nb == 0 and n > 16:
        first = (720 if n <= 48 else 1152) // ((n + 15) // 16) ** 2 + 1
        _compare(gpu_lib, n, nt, first - 1)
        _compare(gpu_lib, n, nt, first)
    else:
        _compare(gpu_lib, n, nt, nb or 700)


def _compare(gpu_lib, n, nt, nb):
    from muspinsim_amd import _native as N
    rng = np.random.default_rng(100 * n + nt)
    slots = 2
    E = np.sort(rng.normal(0, 30.0, (nb, n)), axis=1)
    t = rng.uniform(0, 10.0, nt)
    r = rng.normal(size=(slots, nt))
    slot = (1 - np.arange(nb) % 2).astype(np.int32)
    w = rng.uniform(0.5, 2.0, nb)
    d = [torch.as_tensor(a).cuda() for a in (E, np.append(t, 0.0), np.append(r.ravel(), 0.0), slot, w)]
    R = torch.full((nb, n, n), np.nan, dtype=torch.float64, device="cuda")
    S = torch.full_like(R, np.nan)
    st = torch.cuda.current_stream().cuda_stream
    N.check(gpu_lib.msp_adjoint_freq(n, nb, nt, d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(),
                                     d[3].data_ptr(), d[4].data_ptr(), 0.25, R.data_ptr(),
                                     S.data_ptr(), st))
    arg = 2 * np.pi * (E[:, :, None] - E[:, None, :])[..., None] * t
    ref_r = 0.25 * w[:, None, None] * (r[slot][:, None, None, :] * np.cos(arg)).sum(-1)
    ref_s = 0.25 * w[:, None, None] * (r[slot][:, None, None, :] * t * np.sin(arg)).sum(-1)
    # phases of up to 2 pi 200 MHz 10 us carry a relative rounding of 2^-52 each
    tol = 1e-15 * (2 * np.pi * 200.0 * 10.0) * np.abs(r).sum() + 1e-14
    assert np.abs(R.cpu().numpy() - ref_r).max() <= tol
    assert np.abs(S.cpu().numpy() - ref_s).max() <= 10.0 * tol

"""The sampler's search over leaves of 256 amplitudes: one leaf, as many as a
round of 64 probes holds, one more round, and leaves of probability zero."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("n,log_nz", [(3, 2), (8, 5), (9, 0), (13, 4), (14, 9), (15, 3), (20, 12), (21, 7)])
def test_samples_of_equal_weights_are_exact(dev, n, log_nz):
    """2^log_nz amplitudes of weight 1/4 at random places, the rest zero: every
    sum is exact, so the index for u is the floor(u * count)-th of them."""
    import torch
    import blackwell_kernels as bk
    rng = np.random.default_rng(n)
    count = 1 << log_nz
    at = np.sort(rng.choice(1 << n, count, replace=False))
    psi = np.zeros(1 << n, np.complex64)
    psi[at] = 0.5 * np.exp(0.5j * np.pi * rng.integers(0, 4, count)).round()
    u = np.concatenate([np.arange(count) / count, (np.arange(count) + 0.75) / count, [0.0, 1 - 2.0 ** -30]])
    got = bk.sample_with_uniforms(torch.from_numpy(psi).to(dev), torch.from_numpy(u).to(dev)).cpu().numpy()
    assert np.array_equal(got, at[np.floor(u * count).astype(int)])
    again = bk.sample_with_uniforms(torch.zeros(1 << n, dtype=torch.complex64, device=dev),
                                    torch.from_numpy(u).to(dev)).cpu().numpy()
    assert not again.any()                               # no probability anywhere: index 0

"""Measure kernels (Meyer-Wallach, stabiliser entropy) at the edges of their
ranges: widths around the 16-value register groups, the 12-qubit chunk and
the block's state groups, batches that do not fill a block or the XCDs.

References are numpy in complex128 from the same state values, so the
tolerance is double rounding in both precisions: a sum of 2^n products of a
normalised state is off by at most about 2^n eps times their mean size, far
below 1e-13; the stabiliser sums are 4^n terms of a size-1 total."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _states(n, batch, dtype, seed):
    import torch
    rng = np.random.default_rng(seed)
    s = rng.standard_normal((batch, 1 << n)) + 1j * rng.standard_normal((batch, 1 << n))
    s /= np.linalg.norm(s, axis=1, keepdims=True)
    t = torch.as_tensor(s.astype(dtype), device="cuda")
    return t, t.cpu().numpy().astype(np.complex128)


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n,batch", [(1, 5), (2, 3), (3, 300), (4, 257), (5, 130), (6, 1), (7, 33), (8, 17), (9, 9),
                                     (10, 5), (11, 3), (12, 2), (13, 3), (14, 9), (16, 8), (17, 11), (21, 1)])
def test_meyer_wallach_widths_and_batches(n, batch, dtype):
    from pyramaterised_amd import engine as E
    t, s = _states(n, batch, dtype, 100 * n + batch)
    rho, q = E.mw(t, n)
    ref = np.zeros((batch, n, 4))
    for k in range(n):
        v = s.reshape(batch, 1 << k, 2, 1 << (n - 1 - k))
        a, b = v[:, :, 0], v[:, :, 1]
        ref[:, k, 0] = (abs(a) ** 2).sum(axis=(1, 2))
        ref[:, k, 1] = (abs(b) ** 2).sum(axis=(1, 2))
        r = (a * b.conj()).sum(axis=(1, 2))
        ref[:, k, 2], ref[:, k, 3] = r.real, r.imag
    Q = 2 * (1 - (ref[..., 0] ** 2 + ref[..., 1] ** 2 + 2 * (ref[..., 2] ** 2 + ref[..., 3] ** 2)).mean(axis=1))
    assert np.max(np.abs(rho.cpu().numpy() - ref)) < 1e-13
    assert np.max(np.abs(q.cpu().numpy() - Q)) < 1e-13


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("n,batch", [(1, 9), (2, 65), (3, 7), (4, 17), (5, 5), (6, 3), (7, 2), (8, 3), (9, 2),
                                     (10, 2), (11, 1), (12, 1), (13, 1)])
@pytest.mark.parametrize("alpha", [2.0, 0.5, 3.0])
def test_stabiliser_sum_widths(n, batch, dtype, alpha):
    from pyramaterised_amd import engine as E
    t, s = _states(n, batch, dtype, 7 * n + batch)
    got = E.magic_sum(t, n, alpha).cpu().numpy()
    D = 1 << n
    idx = np.arange(D)
    ref = np.zeros(batch)
    for b in range(batch):
        for j0 in range(0, D, 256):  # X parts in blocks
            j = idx[j0:j0 + 256]
            f = s[b].conj()[None, :] * s[b][idx[None, :] ^ j[:, None]]
            for bit in range(n):
                v = f.reshape(len(j), -1, 2, 1 << bit)
                f = np.stack([v[:, :, 0] + v[:, :, 1], v[:, :, 0] - v[:, :, 1]], axis=2)
            ref[b] += ((np.abs(f) ** 2 / D) ** alpha).sum()
    # rounding of F is about n eps of the largest term; 4^n terms |F| sum to
    # at most 2^n times the result at alpha = 1/2
    assert np.max(np.abs(got / ref - 1)) < 1e-11

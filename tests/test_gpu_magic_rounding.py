"""Rounding of the stabiliser Renyi sums at alpha = 1/2, where every term has
the factor 2^{-n/2}, against 80-bit sums: over many states the errors have no
common part.  With u = 2^-53 each result is rounded to
within u, rms 0.41 u and independently, so the mean relative error of 4000
states is 0.007 u; a factor rounded once and used in every term alike would
put its own error there (the double next to sqrt(1/2) is 0.62 u off)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


@pytest.mark.parametrize("n,batch", [(3, 4000), (4, 4000), (5, 4000), (6, 1000), (7, 500), (9, 40)])
def test_no_common_error(n, batch):
    from pyramaterised_amd import engine as E
    rng = np.random.default_rng(n)
    d = 1 << n
    s = rng.normal(size=(batch, d)) + 1j * rng.normal(size=(batch, d))
    s /= np.linalg.norm(s, axis=1, keepdims=True)
    got = E.magic_sum(torch.as_tensor(s, device="cuda"), n, 0.5).cpu().numpy().astype(np.longdouble)
    j = np.arange(d)
    x = s.astype(np.clongdouble)
    want = np.zeros(batch, dtype=np.longdouble)
    for m in range(d):  # <psi|X^m Z^i|psi> for every i
        f = (x.conj() * x[:, j ^ m])[:, None, :]
        for b in range(n):
            v = f.reshape(batch, -1, 2, 1 << b)
            f = np.stack([v[:, :, 0] + v[:, :, 1], v[:, :, 0] - v[:, :, 1]], axis=2)
        want += (np.abs(f) / np.sqrt(np.longdouble(d))).reshape(batch, -1).sum(axis=1)
    rel = ((got - want) / want).astype(np.float64)
    # five standard errors of independent roundings, three of them per result
    assert abs(rel.mean()) < 5 * 0.41 * U * np.sqrt(3 / batch) + 0.05 * U, rel.mean() / U
    assert np.sqrt(np.mean(rel ** 2)) < 2 * U

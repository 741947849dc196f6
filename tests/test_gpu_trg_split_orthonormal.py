"""TRG splits whose smallest kept singular values are 1e-3 .. 1e-7 of the largest: kept vectors orthonormal to rounding, and
the gradient through them, for full spectra (up to 192 rows in all) and truncated ones, square and not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(m, mp, kk, smin):
    rng = np.random.default_rng(m + mp)
    n = min(m, mp)
    Q, _ = np.linalg.qr(rng.standard_normal((m, n)))
    P, _ = np.linalg.qr(rng.standard_normal((mp, n)))
    i = np.arange(n)
    s = np.where(i < kk, smin ** (i / (kk - 1)), 0.5 * smin)   # a gap after the kept values
    return Q, s, P


@pytest.mark.parametrize("smin", [1e-3, 1e-4, 1e-5, 2e-6, 1e-7])
@pytest.mark.parametrize("d1,d2,d3,d4,kk", [(8, 8, 8, 8, 16), (6, 9, 8, 11, 13), (16, 16, 16, 16, 32), (12, 11, 13, 17, 17),
                                            (24, 24, 24, 24, 32)])
def test_split_orthonormal(ctx, d1, d2, d3, d4, kk, smin):
    import tnad
    print(f"case: trg_svd {d1}x{d2}x{d3}x{d4} kept={kk} smin={smin:g}", flush=True)
    m, mp = d1 * d2, d3 * d4
    Q, s, P = _matrix(m, mp, kk, smin)
    M = (Q * s) @ P.T
    t = np.asfortranarray(M.reshape(d1, d2, d3, d4, order="F"))
    u, v = tnad.trg_svd(t, kk, 1e-16, ctx=ctx)
    assert u.shape[2] == kk
    u, v = u.reshape(m, kk, order="F"), v.reshape(kk, mp, order="F")
    U, V = u / np.linalg.norm(u, axis=0), v.T / np.linalg.norm(v, axis=1)
    # a sum of m rounded products of unit vectors: m eps / 2 at most
    assert np.abs(U.T @ U - np.eye(kk)).max() < max(m, mp) * 1.2e-16
    assert np.abs(V.T @ V - np.eye(kk)).max() < max(m, mp) * 1.2e-16
    # gradient of <W, u v>: u v = h(M), h(s) = s for the kept values and 0 for the others, so with C = Q^T W P the gradient is
    # the divided differences of h on the symmetric and antisymmetric parts of C (square case)
    if m != mp:
        return
    W = np.random.default_rng(3).standard_normal((m, mp))
    bar = tnad.trg_svd_back(t, kk, 1e-16, (W @ v.T).reshape((d1, d2, kk), order="F"),
                            (u.T @ W).reshape((kk, d3, d4), order="F"), ctx=ctx).reshape(m, mp, order="F")
    C = Q.T @ W @ P
    h = np.where(np.arange(m) < kk, s, 0.0)
    dm, sm = s[:, None] - s[None, :], s[:, None] + s[None, :]
    same = dm == 0.0
    odd = np.where(same, np.where(np.arange(m) < kk, 1.0, 0.0)[:, None], (h[:, None] - h[None, :]) / np.where(same, 1.0, dm))
    G = Q @ (odd * (C + C.T) / 2 + (h[:, None] + h[None, :]) / sm * (C - C.T) / 2) @ P.T
    # M itself carries rounding of eps s_0, which turns the vectors of the smallest kept values by eps s_0 / smin; a hundredfold
    # of that covers the sums over the kept pairs
    assert np.abs(bar - G).max() < 1e-14 / smin * np.abs(G).max() + 1e-12

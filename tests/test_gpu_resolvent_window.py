"""The resolvent's iteration narrows to the columns still active: right-hand sides whose active columns lie at both ends, in the
middle, at one end."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _back(ctx, A, chi, k, G):
    n = len(A)
    G = np.asfortranarray(G)
    out = np.zeros((n, n), order="F")
    ctx.check(ctx.lib.tnad_svd_back_sym(ctx.h, C.c_void_p(A.ctypes.data), n, chi, k, C.c_void_p(G.ctypes.data),
                                        C.c_void_p(out.ctypes.data)))
    return out


@pytest.mark.parametrize("cols", [[0, 1, 39], [0, 39], [17, 18, 19, 25], [0, 1, 2], [39], list(range(40))])
def test_active_columns(ctx, cols):
    print(f"case: svd_back_sym n=256 chi=40 cotangent columns {cols}", flush=True)
    n, chi, k = 256, 40, 90
    rng = np.random.default_rng(7)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    lam = 0.97 ** np.arange(n) * np.where(np.arange(n) % 3, 1.0, -1.0)
    A = np.asfortranarray((Q * lam) @ Q.T)
    A = np.asfortranarray(0.5 * (A + A.T))
    full = rng.standard_normal((n, chi))
    G = np.zeros((n, chi))
    G[:, cols] = full[:, cols]
    got = _back(ctx, A, chi, k, G)
    # every column's solve is independent of the others', and the adjoint linear in G; the solves stop at a relative residual of
    # 1e-13 each, over spectral gaps down to 3 % of the value
    ref = sum(_back(ctx, A, chi, k, np.where(np.arange(chi) == j, full, 0.0)) for j in cols)
    assert np.abs(got).max() > 0.0
    assert np.abs(got - ref).max() < 1e-10 * np.abs(ref).max()

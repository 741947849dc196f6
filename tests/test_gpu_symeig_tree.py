"""The full eigensolver at the edges of its instances (a half of the tridiagonal matrix per workgroup, up to 48, 72 and
96 rows) and of its merge tree, on matrices that stress the merges: rank one (nodes of rounding noise of noise), close
poles with equal weights, exact multiplets, heavy deflation."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 4, 5, 6, 7, 9, 13, 31, 63, 80, 95, 96, 97, 127, 144, 145, 146, 191, 192]


def _matrix(kind, n):
    rng = np.random.default_rng(n)
    i = np.arange(n)
    if kind == "ones":
        return np.ones((n, n))
    if kind == "outer":
        return np.outer(np.cos(i), np.cos(i))
    if kind == "wilkinson":         # periodic Wilkinson blocks: clusters agreeing to 1e-14
        return np.diag(np.abs(10.0 - i % 21)) + np.diag(np.ones(n - 1), 1) + np.diag(np.ones(n - 1), -1)
    if kind == "multiplets":
        Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
        A = (Q * ((i * 7) % 5 - 2.0)) @ Q.T
    elif kind == "graded":
        A = rng.standard_normal((n, n)) * np.exp(-0.3 * (i[:, None] + i[None, :]))
    elif kind == "split":           # two halves that all but decouple
        A = rng.standard_normal((n, n))
        A[: n // 2, n // 2:] *= 1e-14
        A[n // 2:, : n // 2] *= 1e-14
    else:
        A = rng.standard_normal((n, n))
    return 0.5 * (A + A.T)


@pytest.mark.parametrize("kind", ["ones", "outer", "wilkinson", "multiplets", "graded", "split", "random"])
@pytest.mark.parametrize("n", SIZES)
def test_full_spectrum(ctx, n, kind):
    print(f"case: symeig full n={n} {kind}", flush=True)
    A = np.asfortranarray(_matrix(kind, n))
    ev, U, count = np.empty(n), np.empty((n, n), order="F"), C.c_int(0)
    ctx.check(ctx.lib.tnad_symeig(ctx.h, C.c_void_p(A.ctypes.data), n, n, n, C.c_void_p(ev.ctypes.data),
                                  C.c_void_p(U.ctypes.data), C.byref(count)))
    assert count.value == n
    # backward stable with Householder and divide and conquer: errors of a few n eps of the matrix's norm
    tol = 10 * (n + 5) * 2.0 ** -52
    norm = max(np.abs(ev).max(), 1e-300)
    assert np.abs(U.T @ U - np.eye(n)).max() < tol
    assert np.abs(A @ U - U * ev).max() < tol * norm
    assert np.abs(np.sort(ev) - np.linalg.eigvalsh(A)).max() < tol * norm

"""The truncated eigensolver (n > 192) on spectra where its orthogonal iteration can go wrong: ten and more
decades (the first product's block is numerically dependent), a rank below the block width, exact multiplets
and +- pairs across the kept edge, a slowly decaying spectrum, the widest block."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(kind, n, want, rng):
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    sgn = np.sign(rng.standard_normal(n))
    i = np.arange(n)
    if kind == "graded":            # fourteen decades over the matrix, ~1e-9 at the kept edge
        lam = sgn * 10.0 ** (-9.0 * i / want)
        lam[np.abs(lam) < 1e-14] = 0.0
    elif kind == "low_rank":        # rank below the kept count
        lam = np.where(i < want // 2, sgn * (1.0 + i), 0.0)
    elif kind == "pairs":           # (+s, -s), as the augmented matrix of a split; a gap after the kept edge
        lam = np.where(i < want, 1.0, 0.05) * 0.93 ** (i // 2) * np.where(i % 2, -1.0, 1.0)
    elif kind == "multiplets":      # exact four-fold values, a gap after the kept edge
        lam = np.where(i < want, 1.0, 0.1) * 0.9 ** (i // 4)
    else:                           # slow decay: many products
        lam = sgn * 1.0 / (1.0 + i) ** 2
    A = (Q * lam) @ Q.T
    return 0.5 * (A + A.T), lam


# block widths at the edges of the Cholesky kernel's 16-column blocks, down to a single block
EDGES = [(200, 1, 1), (200, 3, 5), (200, 8, 16), (200, 8, 17), (300, 20, 95), (300, 20, 97), (400, 100, 191)]


@pytest.mark.parametrize("n,want,k,kind", [(n, w, k, kind) for n, w, k in [(193, 16, 40), (333, 37, 83), (576, 80, 192)]
                                           for kind in ("graded", "low_rank", "pairs", "multiplets", "slow")]
                         + [e + ("graded",) for e in EDGES])
def test_symeig_truncated_hard_spectra(ctx, n, want, k, kind):
    print(f"case: symeig truncated {kind} n={n} want={want} k={k}", flush=True)
    A, lam = _matrix(kind, n, want, np.random.default_rng(n))
    A = np.asfortranarray(A)
    ev, X, got = np.zeros(k), np.zeros((n, k), order="F"), C.c_int(0)
    ctx.check(ctx.lib.tnad_symeig(ctx.h, C.c_void_p(A.ctypes.data), n, want, k, C.c_void_p(ev.ctypes.data),
                                  C.c_void_p(X.ctypes.data), C.byref(got)))
    assert got.value == k
    s0 = np.abs(lam).max()
    ref = np.sort(np.abs(lam))[::-1][:want]
    X = X[:, :want]
    # the iteration stops at a residual of 1e-13 |theta_0|; eigenvalues are off by at most that (Weyl) plus
    # the rounding of A itself (n eps); the block is orthonormal to 1e-12 before the last rotation
    assert np.max(np.abs(np.abs(ev[:want]) - ref)) <= 1e-12 * s0
    assert np.max(np.linalg.norm(A @ X - X * ev[:want], axis=0)) <= 5e-13 * s0
    assert np.max(np.abs(X.T @ X - np.eye(want))) <= 1e-11

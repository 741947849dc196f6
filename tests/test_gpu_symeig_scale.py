"""The eigensolvers on matrices far from unit norm: squares of their entries leave the range of a double."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _symeig(ctx, A, want, k):
    n = len(A)
    A = np.asfortranarray(A)
    ev, X, got = np.zeros(k), np.zeros((n, k), order="F"), C.c_int(0)
    ctx.check(ctx.lib.tnad_symeig(ctx.h, C.c_void_p(A.ctypes.data), n, want, k, C.c_void_p(ev.ctypes.data),
                                  C.c_void_p(X.ctypes.data), C.byref(got)))
    assert got.value == k
    return ev, X


@pytest.mark.parametrize("kind,power", [("random", p) for p in (-1000, -500, -440, 500, 1000)]
                         + [("graded", p) for p in (-800, -440, 800)])
@pytest.mark.parametrize("n", [2, 8, 63, 97, 192])
def test_full_spectrum_scales(ctx, n, kind, power):
    # a power of two changes no rounding, so the result is that of the matrix of order one to the bit
    print(f"case: symeig full n={n} {kind} 2^{power}", flush=True)
    rng = np.random.default_rng(n)
    i = np.arange(n)
    A = rng.standard_normal((n, n)) * (np.exp(-0.3 * (i[:, None] + i[None, :])) if kind == "graded" else 1.0)
    A = A + A.T
    ev, U = _symeig(ctx, A, n, n)
    evs, Us = _symeig(ctx, np.ldexp(A, power), n, n)
    assert np.array_equal(evs, np.ldexp(ev, power))
    assert np.array_equal(Us, U)


@pytest.mark.parametrize("power", [-500, -440, -350, 350, 500])
@pytest.mark.parametrize("kind", ["graded", "slow"])
@pytest.mark.parametrize("n,want,k", [(200, 8, 17), (333, 37, 83)])
def test_truncated_scales(ctx, n, want, k, kind, power):
    print(f"case: symeig truncated n={n} want={want} k={k} {kind} 2^{power}", flush=True)
    Q, _ = np.linalg.qr(np.random.default_rng(n).standard_normal((n, n)))
    i = np.arange(n)
    A = (Q * (10.0 ** (-9.0 * i / want) if kind == "graded" else 1.0 / (1.0 + i) ** 2)) @ Q.T
    A = A + A.T
    ev, X = _symeig(ctx, A, want, k)
    evs, Xs = _symeig(ctx, np.ldexp(A, power), want, k)
    assert np.array_equal(evs, np.ldexp(ev, power))
    assert np.array_equal(Xs, X)


def test_truncated_zero(ctx):
    ev, X = _symeig(ctx, np.zeros((200, 200)), 8, 17)
    assert np.array_equal(ev, np.zeros(17))
    assert np.abs(X.T @ X - np.eye(17)).max() < 1e-11

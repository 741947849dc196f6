"""Inputs that are not numbers end in an error, in the kernels that look for a largest entry too: a column or a tensor of
NaNs has none."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["entry", "row", "all", "inf"])
@pytest.mark.parametrize("n,want,k", [(200, 8, 16), (333, 37, 83)])
def test_symeig_truncated_nonfinite(ctx, n, want, k, where):
    import tnad
    print(f"case: symeig truncated {where} n={n} want={want} k={k}", flush=True)
    A = np.random.default_rng(n).standard_normal((n, n))
    A = np.asfortranarray(A + A.T)
    if where == "entry":
        A[5, 5] = np.nan
    elif where == "row":
        A[5, :] = A[:, 5] = np.nan
    else:
        A[:] = np.nan if where == "all" else np.inf
    ev, X, got = np.zeros(k), np.zeros((n, k), order="F"), C.c_int(0)
    with pytest.raises(tnad.TnadError) as e:
        ctx.check(ctx.lib.tnad_symeig(ctx.h, C.c_void_p(A.ctypes.data), n, want, k, C.c_void_p(ev.ctypes.data),
                                      C.c_void_p(X.ctypes.data), C.byref(got)))
    assert "NaN" in str(e.value)


@pytest.mark.parametrize("where", ["entry", "all"])
@pytest.mark.parametrize("dtype", [float, complex])
def test_trg_nan(ctx, dtype, where):
    import tnad
    print(f"case: trg {dtype.__name__} {where}", flush=True)
    a = np.ones((2, 2, 2, 2), dtype=dtype)
    a[0, 1, 0, 1] = np.nan
    if where == "all":
        a[:] = np.nan
    with pytest.raises(tnad.TnadError):
        tnad.trg_and_grad(a, 4, 3, ctx=ctx)


@pytest.mark.parametrize("n", [1, 8, 97, 192])
def test_symeig_full_nan(ctx, n):
    # every eigenpair is written (a NaN has no rank among the values), so nothing of an earlier call shows
    print(f"case: symeig full NaN n={n}", flush=True)
    A = np.full((n, n), np.nan, order="F")
    ev, U, count = np.zeros(n), np.zeros((n, n), order="F"), C.c_int(0)
    ctx.check(ctx.lib.tnad_symeig(ctx.h, C.c_void_p(A.ctypes.data), n, n, n, C.c_void_p(ev.ctypes.data),
                                  C.c_void_p(U.ctypes.data), C.byref(count)))
    assert np.isnan(ev).all()
    if n > 1:
        assert np.isnan(U).all()

"""FP64 contractions with few output tiles (every wave multiplies a whole tile over its share of K): edges of the
tiles, of the 16-element K steps and of the waves' shares, for every way an operand can be laid out, against NumPy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAYOUTS = ["ik,kj->ij", "ki,kj->ij", "ik,jk->ij", "ki,jk->ij"]
# one of each tile (16 x 16 up to 32 x 48 per workgroup), remainders on every index, K below a step, one step, not all
# waves, all waves, several rounds
SIZES = [(1, 1, 1), (2, 2, 2), (16, 16, 16), (17, 15, 33), (31, 47, 127), (33, 49, 129), (64, 2, 200), (1, 70, 257),
         (513, 17, 130), (96, 96, 2048), (2047, 45, 1030), (2048, 192, 520), (640, 641, 272), (1024, 512, 256)]


def _check(got, A, B, ref, extra=0.0):
    # a sum of K products in any order, in FP64: |error| <= (K + 2) 2^-53 sum |a||b|, and NumPy's the same
    k = A.shape[1]
    bound = 2 * (k + 2) * 2.0 ** -53 * (np.abs(A) @ np.abs(B) + extra)
    assert np.all(np.abs(got - ref) <= bound)


@pytest.mark.parametrize("spec", LAYOUTS)
@pytest.mark.parametrize("m,n,k", SIZES)
def test_layouts_and_edges(ctx, spec, m, n, k):
    import tnad
    print(f"case: slab {spec} {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(m + 7 * n + 11 * k)
    A, B, C0 = rng.standard_normal((m, k)), rng.standard_normal((k, n)), rng.standard_normal((m, n))
    a = A if spec[:2] == "ik" else np.asfortranarray(A.T)
    b = B if spec[3:5] == "kj" else np.asfortranarray(B.T)
    _check(tnad.contract(spec, a, b, ctx=ctx), A, B, A @ B)
    _check(tnad.contract(spec, a, b, ctx=ctx, alpha=-0.5, beta=2.0, Cin=C0), A, B, 2.0 * C0 - 0.5 * (A @ B),
           2.0 * np.abs(C0))


# composite indices: a K of two runs whose inner extent is odd, even, a multiple of 16; rows of two runs, even and odd
@pytest.mark.parametrize("spec", ["abcd,cdef->abef", "cdab,cdef->abef", "acbd,edfc->abef", "dacb,fdec->bafe"])
@pytest.mark.parametrize("ext", [dict(a=3, b=5, c=7, d=3, e=5, f=4), dict(a=6, b=4, c=2, d=9, e=8, f=3),
                                 dict(a=16, b=9, c=16, d=9, e=16, f=2)])
def test_composite_indices(ctx, spec, ext):
    import tnad
    print(f"case: slab {spec} {ext}", flush=True)
    ia, ib = spec.split("->")[0].split(",")
    rng = np.random.default_rng(5)
    A = rng.standard_normal([ext[c] for c in ia])
    B = rng.standard_normal([ext[c] for c in ib])
    ref = np.einsum(spec, A, B)
    mag = np.einsum(spec, np.abs(A), np.abs(B))
    got = tnad.contract(spec, A, B, ctx=ctx)
    assert np.all(np.abs(got - ref) <= 2 * (ext["c"] * ext["d"] + 2) * 2.0 ** -53 * mag)


# an infinity or a NaN reaches exactly the outputs it belongs to, also from the last row, column and k
@pytest.mark.parametrize("spec", LAYOUTS)
def test_nonfinite_values_stay_in_their_rows(ctx, spec):
    import tnad
    print(f"case: slab nonfinite {spec}", flush=True)
    m, n, k = 35, 18, 37
    rng = np.random.default_rng(2)
    A, B = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    A[m - 1, 3] = np.inf
    A[5, k - 1] = np.nan
    B[k - 1, n - 1] = -np.inf
    a = A if spec[:2] == "ik" else np.asfortranarray(A.T)
    b = B if spec[3:5] == "kj" else np.asfortranarray(B.T)
    got, ref = tnad.contract(spec, a, b, ctx=ctx), A @ B
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isposinf(got), np.isposinf(ref))
    assert np.array_equal(np.isneginf(got), np.isneginf(ref))
    ok = np.isfinite(ref)
    assert np.allclose(got[ok], ref[ok], rtol=0, atol=1e-13 * k)

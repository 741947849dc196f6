"""FP64 contractions over two indices that lie in different orders in the operands, and over a long K: values against
NumPy on both sides of every rule, and the time of a product that must not depend on the order they are named in."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# K below and at the length from which the order is chosen, and around the lengths from which a product may be left to the
# kernels that cut K over the grid; inner runs odd, even and of 32; outputs of one tile, of fewer than 32 and of more
KS = [(5, 51), (4, 64), (64, 4), (51, 30), (48, 32), (33, 93), (32, 96), (7, 585), (2, 4098)]
SPECS = ["ikl,lkj->ij", "kil,ljk->ij", "kli,lkj->ij", "kil,lkj->ij", "lik,klj->ij", "ikl,jlk->ij", "kli,jlk->ij"]


@pytest.mark.parametrize("spec", SPECS)
@pytest.mark.parametrize("k,l", KS)
@pytest.mark.parametrize("i,j", [(1, 7), (35, 18), (130, 260)])
def test_two_contracted_indices(ctx, spec, i, j, k, l):
    import tnad
    print(f"case: k order {spec} {i}x{j} K {k}x{l}", flush=True)
    ext = dict(i=i, j=j, k=k, l=l)
    ia, ib = spec.split("->")[0].split(",")
    rng = np.random.default_rng(i + 3 * j + 5 * k + 7 * l)
    A = rng.standard_normal([ext[c] for c in ia])
    B = rng.standard_normal([ext[c] for c in ib])
    got = tnad.contract(spec, A, B, ctx=ctx)
    # a sum of K products in any order, in FP64: |error| <= (K + 2) 2^-53 sum |a||b|, and NumPy's the same
    bound = 2 * (k * l + 2) * 2.0 ** -53 * np.einsum(spec, np.abs(A), np.abs(B), optimize=True)
    assert np.all(np.abs(got - np.einsum(spec, A, B, optimize=True)) <= bound)


@pytest.mark.parametrize("spec", ["ik,kj->ij", "ki,kj->ij", "ik,jk->ij", "ki,jk->ij"])
@pytest.mark.parametrize("i,j,k", [(5, 9, 3071), (5, 9, 3072), (64, 64, 3072), (63, 62, 4096), (64, 60, 4097),
                                   (250, 120, 3500), (256, 128, 3500), (1, 40, 4000)])
def test_long_k(ctx, spec, i, j, k):
    import tnad
    print(f"case: long K {spec} {i}x{j}x{k}", flush=True)
    rng = np.random.default_rng(i + j + k)
    A, B, C0 = rng.standard_normal((i, k)), rng.standard_normal((k, j)), rng.standard_normal((i, j))
    a = A if spec[:2] == "ik" else np.asfortranarray(A.T)
    b = B if spec[3:5] == "kj" else np.asfortranarray(B.T)
    got = tnad.contract(spec, a, b, ctx=ctx, alpha=-0.5, beta=2.0, Cin=C0)
    bound = 2 * (k + 2) * 2.0 ** -53 * (np.abs(A) @ np.abs(B) + 2.0 * np.abs(C0))
    assert np.all(np.abs(got - (2.0 * C0 - 0.5 * (A @ B))) <= bound)


# the first operand contiguous along its rows, the second along either contracted index: the same bytes in runs of even
# length, so far less than a factor of two apart (read in the first operand's order only, the second call touched a line of
# memory per element and took 2.8 times as long)
def test_time_does_not_depend_on_the_order(ctx):
    import tnad
    e = dict(i=2304, j=180, k=50, l=32)
    t = {}
    for spec in ("ikl,klj->ij", "ikl,lkj->ij"):
        print(f"case: time {spec}", flush=True)
        t[spec] = min(tnad.time_contract(spec, e, "fp64", reps=20, ctx=ctx) for _ in range(5))
    assert max(t.values()) < 2 * min(t.values())

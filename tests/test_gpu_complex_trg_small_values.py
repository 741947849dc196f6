"""Complex TRG gradients where the kept singular values reach down to 1e-9 .. 1e-13 of the largest: the kept vectors must
come out orthonormal there as in the real path (full spectra of up to 96 rows and truncated ones)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [117, 119, 124])
def test_real_weights_as_complex(ctx, seed):
    # Boltzmann weights as ComplexF64 give the real path's lnZ and gradient; that one is right to rounding here, and the
    # gradient well conditioned, so 1e-10 leaves five digits for the sums over the splits
    import tnad
    print(f"case: complex trg vertex gradient seed={seed} chi=16 niter=5", flush=True)
    a = np.exp(-2.0 * np.random.default_rng(seed).random((2, 2, 2, 2)))
    lnz, g = tnad.trg_and_grad(a, 16, 5, ctx=ctx)
    lnz_z, g_z = tnad.trg_and_grad(a + 0j, 16, 5, ctx=ctx)
    assert abs(lnz_z - lnz) < 1e-13 * abs(lnz)
    assert np.abs(g_z - g).max() < 1e-10 * np.abs(g).max()


def test_gauge_transformed_weights(ctx):
    # unitary changes of basis on the two kinds of bonds leave lnZ alone and turn the gradient with the tensor
    import tnad
    print("case: complex trg vertex gradient, unitary gauge, seed=117 chi=16 niter=5", flush=True)
    rng = np.random.default_rng(117)
    a = np.exp(-2.0 * rng.random((2, 2, 2, 2)))
    U, _ = np.linalg.qr(rng.standard_normal((2, 2)) + 1j * rng.standard_normal((2, 2)))
    V, _ = np.linalg.qr(rng.standard_normal((2, 2)) + 1j * rng.standard_normal((2, 2)))

    def turn(t):
        return np.einsum("urdl,ui,rj,dk,lm->ijkm", t, U, V, U.conj(), V.conj())
    lnz, g = tnad.trg_and_grad(a, 16, 5, ctx=ctx)
    lnz_z, g_z = tnad.trg_and_grad(np.asfortranarray(turn(a)), 16, 5, ctx=ctx)
    # (niter = 5 leaves the largest entry of a turned tensor another one, whose logarithm is taken out and put back)
    assert abs(lnz_z - lnz) < 1e-12 * abs(lnz)
    assert np.abs(g_z - turn(g)).max() < 1e-10 * np.abs(g).max()

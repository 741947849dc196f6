"""TRG gradients where the kept singular values reach down to 1e-9 .. 1e-13 of the largest: the +-s pairs of the
augmented matrix then mix at rounding level over s / s_0, and the kept vectors must still come out orthonormal."""
import numpy as np
import pytest

from oracle import tnad_oracle as O

pytestmark = pytest.mark.gpu


# Boltzmann weights of vertex models; the splits of these three keep values of 1e-9 .. 1e-13 of the largest, in full
# spectra (up to 192 rows) and in truncated ones.  The gradient itself is well conditioned (the weights are of
# order one), so it is right to rounding times a modest factor: 1e-10 leaves five digits of that.
@pytest.mark.parametrize("seed", [117, 119, 124])
def test_vertex_gradient_with_small_kept_values(ctx, seed):
    import tnad
    print(f"case: trg vertex gradient seed={seed} chi=32 niter=6", flush=True)
    a = np.exp(-2.0 * np.random.default_rng(seed).random((2, 2, 2, 2)))
    direc = np.random.default_rng(1).standard_normal(a.shape)
    lnz, abar = tnad.trg_and_grad(a, 32, 6, ctx=ctx)
    lnz_o, g_o = O.trg(a, 32, 6, with_grad_seed=direc)
    assert lnz == pytest.approx(lnz_o, rel=1e-13, abs=0)
    assert float(np.sum(abar * direc)) == pytest.approx(g_o, rel=1e-10)

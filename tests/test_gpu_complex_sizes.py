"""Complex energy and gradient against the oracle (same phase rule) over the range of corner matrices, n = 4 chi from
4 to 96: a single 16-lane group, sizes off and on the lane and tile edges, the largest whose vectors fill the LDS."""
import numpy as np
import pytest

from oracle import tnad_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chi,maxit", [(1, 1), (2, 2), (3, 3), (7, 2), (16, 2), (17, 1), (24, 1)])
def test_complex_energy_over_sizes(ctx, chi, maxit):
    import tnad
    print(f"case: complex energy chi={chi} maxit={maxit}", flush=True)
    rng = np.random.default_rng(100 + chi)
    h = O.hamiltonian_heisenberg()
    b = O.reshape_f(rng.standard_normal(32) + 1j * rng.standard_normal(32), (2, 2, 2, 2, 2))
    e, g = tnad.energy_and_grad(h, b, chi, 0.0, maxit, ctx=ctx)
    e_o, g_o, _ = O.energy_and_grad(h, b, chi, 0.0, maxit)
    # a few steps of well-separated spectra: rounding times the condition of the adjoint (the bounds of the
    # smaller sizes' test)
    assert abs(e - e_o) < 1e-11
    assert np.linalg.norm(g - g_o) < 1e-8 * np.linalg.norm(g_o)

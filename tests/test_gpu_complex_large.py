"""Complex contractions with large outputs: the cotangent of the double layer at bonds of 25 and 36 (up to 1296 x 1296)."""
import numpy as np
import pytest

from oracle import tnad_oracle as O

pytestmark = pytest.mark.gpu


def test_double_layer_bond_25_matches_real(ctx):
    import tnad
    print("case: complex energy gradient d=5 s=2 chi=3, two steps", flush=True)
    bulk, h = O.symmetrized_random_bulk(5, 2, 0, "uniform"), O.hamiltonian_heisenberg()
    e, g = tnad.energy_and_grad(h, bulk, 3, 0.0, 1, ctx=ctx)
    ez, gz = tnad.energy_and_grad(h.astype(complex), bulk.astype(complex), 3, 0.0, 1, ctx=ctx)
    assert abs(ez - e) < 1e-12 * abs(e)
    assert np.abs(gz - g).max() < 1e-10 * np.abs(g).max()


def test_double_layer_bond_36(ctx):
    import tnad
    print("case: complex energy gradient d=6 s=1 chi=2, one step", flush=True)
    bulk, h = O.symmetrized_random_bulk(6, 1, 0, "uniform"), np.ones((1, 1, 1, 1))
    ez, gz = tnad.energy_and_grad(h.astype(complex), bulk.astype(complex), 2, 0.0, 0, ctx=ctx)
    # with one physical state <h> / <1> is h itself, whatever the bulk: the gradient vanishes up to the rounding of its two
    # parts, each of the order of 1 / |bulk| (entries of order one)
    assert abs(ez - 1.0) < 1e-12
    assert np.abs(gz).max() < 1e-10

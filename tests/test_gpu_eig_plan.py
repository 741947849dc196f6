"""The product count that one CTMRG step's eigensolver hands to the next, where the tolerance cannot be reached."""
import pytest

from oracle import tnad_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eig_tol", [1e-17, 1e-16])
def test_products_do_not_grow_below_the_rounding_level(ctx, eig_tol):
    import tnad
    print(f"case: eig_tol={eig_tol:g} chi=64 D=4, 17 steps", flush=True)
    h, bulk = O.hamiltonian_heisenberg(), O.symmetrized_random_bulk(2, 2, 0, "uniform")

    def products(maxit):
        tnad.energy_and_grad(h, bulk, 64, 0.0, maxit, ctx=ctx, want_grad=False, eig_tol=eig_tol)
        st = ctx.stats()
        assert st["iters"] == maxit + 1
        return st["eig_iters_total"]

    # the first step finds the rounding level and notices it 8 products later; a later one starts from its count and may look
    # once more, at most 16 products on
    first = products(0)
    assert products(16) <= 17 * (first + 16)

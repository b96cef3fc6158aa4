"""What a linear solve that does not converge leaves: krylov_maxit bounds its iterations, attempt
without the coarse correction included, and the residuals that it reports are those of the
caller's start and of the vector that it returns."""
import numpy as np
import pytest

from cardiomechanics_amd import materials as MT
from cardiomechanics_amd import mesh as M
from cardiomechanics_amd.context import MechanicsContext

pytestmark = pytest.mark.gpu


def solve(method, precision, maxit, rtol):
    mesh = M.lv_mesh(2500)
    with MechanicsContext(mesh, [MT.lv_holzapfel()], krylov_method=method, precision=precision, krylov_maxit=maxit) as ctx:
        vals = (ctx.tangent(mesh.coords.ravel(), 0.0) + 4e6 * ctx.mass_matrix()).astype(ctx.value_dtype)
        A = ctx.bsr(vals.astype(np.float64)).tocsr()
        rng = np.random.default_rng(9)
        b, x0 = A @ rng.normal(size=ctx.n_dofs), 1e3 * rng.normal(size=ctx.n_dofs)
        x, st = ctx.linear_solve(vals, b, x0=x0, rtol=rtol)
    print(f"method {method}: {st.iterations} iterations of {maxit}, residual {st.final_residual:.6e} of {st.initial_residual:.6e}",
          flush=True)
    assert not st.converged
    start, end = np.linalg.norm(b - A @ x0), np.linalg.norm(b - A @ x)
    assert start > 10 * np.linalg.norm(b)
    assert abs(st.initial_residual - start) <= 1e-10 * start
    # both sides round sums of products as large as |A| |x|
    assert abs(st.final_residual - end) <= 1e-10 * end + 1e-13 * np.linalg.norm(abs(A) @ abs(x))
    return st


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("method", [0, 1, 2])
def test_iterations_spent(method, precision):
    assert solve(method, precision, 5, 1e-12).iterations == 5


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_tolerance_below_rounding(precision):
    """The recurrence reaches the tolerance, b - A x does not: given up after 50 restarts (some 4,000
    iterations), and again without the correction, from where the first attempt ended."""
    st = solve(2, precision, 100_000, 1e-19)
    assert 102 <= st.iterations < 100_000
    assert st.final_residual <= 1e-10 * st.initial_residual

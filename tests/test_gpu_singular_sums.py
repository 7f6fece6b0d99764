"""The singular faces' sums over a face's angular points (collocation), where the grouping of a wavefront's lanes changes:
1, 2, 3 and 4 points (4 lanes per face), 8, 15 and 20 (as many lanes as points; 8 to 3 faces per wavefront, so that a
vertex's faces take several batches) and 65 (64 lanes, one face at a time).  cqbem_laplace against the oracle: U, Bt and
Ba within 1e-13 (sums of at most 65^2 terms of one sign); P's finite-part rule cancels terms of 1/rho^2 with the innermost
rho shrinking as 1/points: 1e-10 at 10 points, times (points / 10)^2."""
import numpy as np
import pytest

from surfaceonlydeformables_amd import abi
from surfaceonlydeformables_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = abi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("order,sub", [(1, 1), (2, 1), (3, 1), (4, 1), (4, 2), (5, 3), (5, 4), (5, 13)])
def test_groups(ctx, oracle, order, sub):
    V, F = M.icosphere(1, 0.2)
    V = M.center(M.jitter(V, F, 0.01, 8), F)
    rho, nu, L, dt = 1000.0, 0.3, 16, 1e-3
    _, c1, c2 = M.material_speeds(5e5, nu, rho)
    R = 1e-10 ** (1 / (2 * L))
    print(f"singular sums {order * sub} points", flush=True)
    g = ctx.laplace(abi.make_mesh(V, F), abi.make_params(c1, c2, rho, nu, dt, R, L, order=order, subdivision=sub), 5)
    s = oracle.frequencies(L, R, dt, 2)[5]
    o = oracle.laplace(V, F, oracle.params(c1, c2, rho, nu, dt, R, L, order=order, subdiv=sub, nthreads=8), s)
    for k, tol in (("U", 1e-13), ("P", 1e-10 * max(1.0, (order * sub / 10) ** 2)), ("Bt", 1e-13), ("Ba", 1e-13)):
        assert np.linalg.norm(g[k] - o[k]) <= tol * np.linalg.norm(o[k]), k

"""cqbem_last_timings of a job with host outputs: the phases [1] to [5] follow one another on one stream (quadrature, B,
singular faces, transform on the device; preparation and the copies on the host), so that together they take no longer than
the whole call, up to the 1% and 50 us that the two clocks may differ by."""
import pytest

from surfaceonlydeformables_amd import abi
from surfaceonlydeformables_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("galerkin,order,sub", [(False, 5, 6), (True, 3, 1)])
def test_phases_add_up_to_no_more_than_the_call(galerkin, order, sub):
    V, F = M.icosphere(1 if galerkin else 2, 0.2)
    mesh = abi.make_mesh(M.center(M.jitter(V, F, 0.01, 2), F), F)
    _, c1, c2 = M.material_speeds(3e5, 0.33, 1000.0)
    L = 8
    p = abi.make_params(c1, c2, 1000.0, 0.33, 0.4 / (c2 * 6), 1e-10 ** (1 / (2 * L)), L, galerkin=galerkin, order=order,
                        subdivision=sub)
    ctx = abi.Context(0)
    for _ in range(3):  # the first call also loads the kernels
        print(f"phase times galerkin={galerkin}", flush=True)
        ctx.assemble(mesh, p)
        t = ctx.last_timings()
    ctx.close()
    phases = t["regular_gh"] + t["singular"] + t["transform"] + t["host"] + (0.0 if galerkin else t["regular_b"])
    print({k: round(v, 3) for k, v in t.items()}, f"phases {phases:.3f}", flush=True)
    assert t["regular_gh"] > 0.1 * (t["total"] if not galerkin else 0.0)
    assert phases <= 1.01 * t["total"] + 0.05

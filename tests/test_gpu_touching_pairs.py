"""The touching-pair kernels of the Galerkin path (one lane per direction of the Sauter-Schwab maps, moments along the last
coordinate) against the one-lane-per-rule-point kernels (CQBEM_GALERKIN_SINGULAR=lane), where their work division changes:
rules of 1 to 12 points per coordinate (a last group of 16 directions that is partly empty, or a single direction), item
counts that are no multiple of 4, G or H or B alone, and one or four waves per block.

Tolerances.  One frequency: both sum the same products; the entries carry a cancellation of at most 1/|z|^2 at the rule's
smallest distances, whose weights are below its square, so rounding stays within a few hundred 1.1e-16 of the matrix
norm: 1e-13, as for the existing comparison of the two.  Weights: the inverse transform multiplies that by up to
R^-(L-1) ~ 1e5: 1e-8 of the stack's norm."""
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


def params(L, order, sub, which=abi.ALL):
    _, c1, c2 = M.material_speeds(1e6, 0.35, 1100.0)
    return abi.make_params(c1, c2, 1100.0, 0.35, 5e-4, 1e-10 ** (1 / (2 * L)), L, order=order, subdivision=sub, galerkin=True,
                           which=which)


def mesh(name):
    V, F = {"ico1": lambda: M.icosphere(1, 0.1), "ico2": lambda: M.icosphere(2, 0.1), "cube2": lambda: M.cube(2, 0.1),
            "ragged": lambda: abi.decimate_mesh(*M.icosphere(1, 0.1), 46)}[name]()
    return M.center(M.jitter(V, F, 0.01, 3), F), F


def off(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def both(monkeypatch, run):
    out = []
    for variant in ("quad", "lane"):
        monkeypatch.setenv("CQBEM_GALERKIN_SINGULAR", variant)
        out.append(run())
    return out


@pytest.mark.parametrize("name,order,sub,which", [("ico1", 1, 1, abi.ALL), ("cube2", 4, 3, abi.ALL), ("ragged", 5, 1, abi.ALL),
                                                  ("ragged", 3, 1, abi.G), ("ragged", 3, 1, abi.H),
                                                  ("ragged", 2, 1, abi.B_TRANS | abi.B_ANGULAR)])
def test_one_frequency_against_the_lane_kernels(ctx, monkeypatch, name, order, sub, which):
    V, F = mesh(name)
    m = abi.make_mesh(V, F)
    for l in (0, 3):
        print(f"touching pairs {name} {order}x{sub} which={which} l={l}", flush=True)
        got, want = both(monkeypatch, lambda: ctx.laplace(m, params(8, order, sub, which), l))
        for k in want:
            assert (got[k] is None) == (want[k] is None)
            if want[k] is not None and np.linalg.norm(want[k]) > 0:
                assert off(got[k], want[k]) <= 1e-13, k


@pytest.mark.parametrize("name,L", [("ico2", 64), ("ragged", 9)])
def test_all_frequencies_against_the_lane_kernels(ctx, monkeypatch, name, L):
    """ico2 with 33 frequencies has enough items for one wave per block; the ragged mesh takes four."""
    V, F = mesh(name)
    m = abi.make_mesh(V, F)
    print(f"touching pairs {name} L={L}", flush=True)
    got, want = both(monkeypatch, lambda: ctx.assemble(m, params(L, 1, 1)))
    for k in want:
        assert off(got[k], want[k]) <= 1e-8, k

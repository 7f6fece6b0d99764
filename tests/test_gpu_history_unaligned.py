"""cqbem_history and cqbem_matvec where the 16-byte loads of the matrices are only 8-byte aligned (an odd n3, or buffers
that start at an odd double), at the edges of a wavefront's 128 columns, of the 512-column unrolled step and of the 4
rows of a wavefront; and where the steps are split over the waves of a block.  Sums of at most 5 x 2 x 1027 terms in another order: each of relative error below 1e-13 of the
norm (1e4 terms of random sign, 1.1e-16 each)."""
import numpy as np
import pytest

from surfaceonlydeformables_amd import abi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = abi.Context(0)
    yield c
    c.close()


def device(a, shift):
    """a on the device, starting `shift` doubles behind a 16-byte boundary."""
    import torch
    buf = torch.empty(a.size + 2, dtype=torch.float64, device="cuda:0")
    view = buf[shift:shift + a.size]
    view.copy_(torch.from_numpy(np.ascontiguousarray(a).reshape(-1)))
    return view


@pytest.mark.parametrize("n,m", [(8, 1), (64, 2), (64, 3), (129, 4), (390, 9), (1019, 5), (1022, 5), (1030, 2), (2049, 2),
                                 (3074, 1)])
def test_steps_over_the_waves_of_a_block(ctx, n, m):
    """m steps over 4 waves (fewer than, as many as and more than them), 2 and 4 rows per wave with ragged last rows, B's
    6 m products over the block; at the sizes where the rows per wave change.  The tolerance above."""
    import torch
    rng = np.random.default_rng(n + m)
    L, nh = m + 1, m + 2
    G, H, B = rng.standard_normal((L, n, n)), rng.standard_normal((L, n, n)), rng.standard_normal((L, n, 6))
    p, u, acc = rng.standard_normal((nh, n)), rng.standard_normal((nh, n)), rng.standard_normal((nh, 6))
    t = [device(a, 0) for a in (G, H, B, p, u, acc)]
    out = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    print(f"history over the waves n={n} m={m}", flush=True)
    ctx.history(n, L, t[0].data_ptr(), t[1].data_ptr(), t[2].data_ptr(), t[3].data_ptr(), t[4].data_ptr(), t[5].data_ptr(), nh,
                out.data_ptr())
    want = sum(G[i] @ p[nh - i] - H[i] @ u[nh - i] + B[i] @ acc[nh - i] for i in range(1, m + 1))
    assert np.linalg.norm(out.cpu().numpy() - want) <= 1e-13 * np.linalg.norm(want)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 3, 127, 129, 130, 511, 513, 514, 1027])
def test_unaligned(ctx, n, shift):
    import torch
    rng = np.random.default_rng(n)
    L, nh = 3, 2
    G, H = rng.standard_normal((L, n, n)), rng.standard_normal((L, n, n))
    p, u = rng.standard_normal((nh, n)), rng.standard_normal((nh, n))
    t = [device(a, shift) for a in (G, H, p, u)]
    out = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    print(f"unaligned history n={n} shift={shift}", flush=True)
    for g, h in ((1, 1), (1, 0), (0, 1)):
        ctx.history(n, L, t[0].data_ptr() if g else None, t[1].data_ptr() if h else None, None, t[2].data_ptr(),
                    t[3].data_ptr(), None, nh, out.data_ptr())
        want = sum(g * (G[i] @ p[nh - i]) - h * (H[i] @ u[nh - i]) for i in (1, 2))
        assert np.linalg.norm(out.cpu().numpy() - want) <= 1e-13 * max(np.linalg.norm(want), 1.0)
    ctx.matvec(n, t[0].data_ptr(), t[2].data_ptr(), out.data_ptr())
    want = G[0] @ p[0]
    assert np.linalg.norm(out.cpu().numpy() - want) <= 1e-13 * max(np.linalg.norm(want), 1.0)

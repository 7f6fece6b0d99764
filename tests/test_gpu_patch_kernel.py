"""The patch kernel of the regular-face G and H against the star kernel (CQBEM_COLLOC_KERNEL=star: one lane per column
vertex, every face evaluated once per corner, another formulation of the same sums) where the patch kernel's work
division changes: face counts at the edges of a 64-face chunk, of 1, 2 and several chunks per patch (a chunk shared by
4, 2 or 1 waves), of several patches, and rules of 1 to 63 points; every face touching the row point; and several rows
per block with a ragged last group.

Tolerances.  One Laplace-domain matrix: each point's entries carry some 30 roundings of 1.1e-16 and a cancellation
between the two waves' terms of at most 1/|z|^2 ~ 1e2, i.e. 4e-13 of the entry; 1e-12 of the matrix norm.  Weights:
the inverse transform multiplies that by up to R^-(L-1) ~ 1e5 on weights that are small beside the first ones, over
sums of Lf terms with independent errors; 1e-8 of the stack's norm."""
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


def sphere_with(nf):
    """A closed mesh of nf faces (nf even), of about unit-ratio triangles."""
    if nf == 4:
        V = np.array([(1, 1, 1), (1, -1, -1), (-1, 1, -1), (-1, -1, 1)], float) * 0.1
        return V, np.array([(0, 1, 2), (0, 3, 1), (0, 2, 3), (1, 3, 2)], np.int32)
    level = 1
    while 20 * 4 ** level < nf:
        level += 1
    V, F = M.icosphere(level, 0.2)
    V = M.jitter(V, F, 0.01, nf)
    return (V, F) if len(F) == nf else abi.decimate_mesh(V, F, nf)


def params(L, order, sub, which=abi.G | abi.H, bdf=abi.BDF2):
    _, c1, c2 = M.material_speeds(3e5, 0.33, 1000.0)
    return abi.make_params(c1, c2, 1000.0, 0.33, 0.4 / (c2 * max(L - 2, 4)), 1e-10 ** (1 / (2 * L)), L, bdf=bdf, order=order,
                           subdivision=sub, which=which)


def off(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("nf,order,sub", [(4, 5, 2), (20, 5, 2), (62, 5, 1), (64, 5, 2), (66, 4, 2), (126, 1, 1), (128, 5, 2),
                                          (130, 2, 1), (192, 3, 2), (258, 5, 2), (512, 5, 3), (520, 5, 2), (1100, 4, 1)])
def test_one_frequency_against_the_star_kernel(ctx, monkeypatch, nf, order, sub):
    V, F = sphere_with(nf)
    assert len(F) == nf
    V = M.center(V, F)
    mesh, L = abi.make_mesh(V, F), 16
    for which in (abi.G | abi.H, abi.G, abi.H):
        p = params(L, order, sub, which)
        for l in (0, 5):
            print(f"patch kernel nf={nf} rule {order}x{sub} which={which} l={l}", flush=True)
            monkeypatch.delenv("CQBEM_COLLOC_KERNEL", raising=False)
            got = ctx.laplace(mesh, p, l)
            monkeypatch.setenv("CQBEM_COLLOC_KERNEL", "star")
            want = ctx.laplace(mesh, p, l)
            for k in "UP":
                assert (got[k] is None) == (want[k] is None)
                if got[k] is not None:
                    assert off(got[k], want[k]) <= 1e-12, k


@pytest.mark.parametrize("nf,L", [(1280, 64), (1276, 61)])
def test_rows_per_block_against_the_star_kernel(ctx, monkeypatch, nf, L):
    """3 patches x 33 or 31 frequencies x 640-odd rows: 7 rows per block, the last group ragged."""
    V, F = sphere_with(nf)
    V = M.center(V, F)
    mesh, p = abi.make_mesh(V, F), params(L, 2, 1)
    print(f"patch kernel rows per block nf={nf} L={L}", flush=True)
    monkeypatch.delenv("CQBEM_COLLOC_KERNEL", raising=False)
    got = ctx.assemble(mesh, p, want=("G", "H"))
    monkeypatch.setenv("CQBEM_COLLOC_KERNEL", "star")
    want = ctx.assemble(mesh, p, want=("G", "H"))
    for k in "GH":
        assert off(got[k], want[k]) <= 1e-8, k


@pytest.mark.parametrize("galerkin", [False, True])
@pytest.mark.parametrize("L", [2, 3, 4, 18])
def test_real_frequencies_share_a_slot(ctx, galerkin, L):
    """At an even L the first and the last frequency (real s) share one slot of the regular-face kernels; cqbem_laplace
    computes each of them alone.  The weights must be the inverse transform of cqbem_laplace's matrices, plus
    B_trans (x) x_v in B_angular: each within 1e-12 of the sum of its terms' magnitudes (the per-entry rounding above,
    and a sum of at most 10 terms).  H from n = 1 (H_0 also holds the C matrix)."""
    V, F = M.icosphere(1, 0.2)
    V = M.center(M.jitter(V, F, 0.01, 3), F)
    mesh, p = abi.make_mesh(V, F), params(L, 4, 1)
    p.galerkin = int(galerkin)
    p.which |= abi.B_TRANS | abi.B_ANGULAR
    print(f"real frequencies L={L} galerkin={galerkin}", flush=True)
    got = ctx.assemble(mesh, p, want=("G", "H", "B_trans", "B_angular"))
    X = [ctx.laplace(mesh, p, l) for l in range(L // 2 + 1)]
    mult = np.array([1.0 if l in (0, L / 2) else 2.0 for l in range(L // 2 + 1)])
    ang = 2 * np.pi / L * np.outer(np.arange(L), np.arange(L // 2 + 1))
    scale = p.R ** -np.arange(L, dtype=float)[:, None] / L
    for k, name in (("U", "G"), ("P", "H"), ("Bt", "B_trans"), ("Ba", "B_angular")):
        S = np.stack([x[k].reshape(-1) for x in X])
        W = scale * ((mult * np.cos(ang)) @ S.real + (mult * np.sin(ang)) @ S.imag)
        mag = scale * (mult @ np.abs(S))
        if name == "B_trans":
            Wt, mt = W, mag
        elif name == "B_angular":
            x = np.repeat(V, 3, axis=0)[None, :, None, :]
            W = W + (Wt.reshape(L, -1, 3, 1) * x).reshape(L, -1)
            mag = mag + (mt.reshape(L, -1, 3, 1) * np.abs(x)).reshape(L, -1)
        first = name == "H"
        assert (np.abs(got[name].reshape(L, -1) - W) <= 1e-12 * mag)[first:].all(), name


@pytest.mark.parametrize("galerkin", [False, True])
@pytest.mark.parametrize("dt,R,l", [(1e-2, 0.5, 1), (1e-3, 0.5, 3), (2e-5, 0.9999, 1), (2e-5, 0.9999, 8), (1e-6, 0.9999, 1),
                                    (1e-6, 0.9999, 0)])
def test_tabulated_exponentials_over_arguments(ctx, oracle, galerkin, dt, R, l):
    """|s r / c| from below 1 to 1e4 over the mesh (up to 7 squarings of the tabulated values), complex and real s, against
    the oracle's exponentials.  Its arguments are rounded to half an ulp, so a value at |z| is good to |z| 1.1e-16 there;
    four times that (two exponentials, two roundings each) on top of the bounds of a moderate argument: 1e-13, and 1e-10
    for the finite-part rule of P."""
    L, rho = 16, 1000.0
    V, F = M.icosphere(1, 0.2)
    V = M.center(M.jitter(V, F, 0.01, 6), F)
    _, c1, c2 = M.material_speeds(1e6, 0.35, rho)
    s = oracle.frequencies(L, R, dt, 2)[l]
    z = abs(s) * 0.42 / c2
    print(f"exponentials dt={dt} l={l} |z|={z:.3g} galerkin={galerkin}", flush=True)
    g = ctx.laplace(abi.make_mesh(V, F), abi.make_params(c1, c2, rho, 0.35, dt, R, L, order=2, subdivision=1, galerkin=galerkin), l)
    o = oracle.laplace(V, F, oracle.params(c1, c2, rho, 0.35, dt, R, L, order=2, subdiv=1, galerkin=galerkin, nthreads=8), s)
    for k, tol in (("U", 1e-13), ("P", 1e-10), ("Bt", 1e-13), ("Ba", 1e-13)):
        assert off(g[k], o[k]) <= tol + 4 * z * 1.1e-16, k


@pytest.mark.parametrize("nf,L", [(62, 5), (62, 16), (66, 33)])
def test_transform_of_odd_sizes(ctx, nf, L):
    """99 or 105 rows: the transform's pairs of entries are unaligned and the last entry has none.  Against the transform of
    cqbem_laplace's matrices (1e-12 of the terms, as above), and in float storage the same weights rounded once."""
    import torch
    V, F = sphere_with(nf)
    V = M.center(V, F)
    n3 = 3 * len(V)
    assert n3 % 2 == 1
    mesh, p = abi.make_mesh(V, F), params(L, 2, 1, abi.G)
    print(f"transform of odd sizes n3={n3} L={L}", flush=True)
    got = ctx.assemble(mesh, p, want=("G",))["G"].reshape(L, -1)
    S = np.stack([ctx.laplace(mesh, p, l)["U"].reshape(-1) for l in range(L // 2 + 1)])
    mult = np.array([1.0 if l in (0, L / 2) else 2.0 for l in range(L // 2 + 1)])
    ang = 2 * np.pi / L * np.outer(np.arange(L), np.arange(L // 2 + 1))
    scale = p.R ** -np.arange(L, dtype=float)[:, None] / L
    W = scale * ((mult * np.cos(ang)) @ S.real + (mult * np.sin(ang)) @ S.imag)
    assert (np.abs(got - W) <= 1e-12 * scale * (mult @ np.abs(S))).all()
    p.storage = abi.STORE_F32
    out = torch.full((L * n3 * n3 + 1,), float("nan"), dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    ctx.assemble_device(mesh, p, {"G": out.data_ptr()})
    assert np.array_equal(out[:-1].cpu().numpy(), got.astype(np.float32).reshape(-1))
    assert bool(torch.isnan(out[-1]))  # nothing behind the last weight

"""Far rules of fewer points than the waves that share a chunk of the patch kernel (CQBEM_QUAD_BANDED with a far rule of 1
or 3 points beside a reference rule of 14 points or more, on a patch of one or two 64-face chunks).

- On the CPU: the points that the parts of a rule take are every point of the rule once and no other.
- On the GPU: each block of U and P equals, where the host plan says near, the reference rule's run bit for bit, and
  where it says far, a run with the far rule as the only rule.  Each point's entries carry some 30 roundings of 1.1e-16
  and a cancellation between the two waves' terms of at most 1/|z|^2 ~ 1e2, i.e. 4e-13; 1e-12 of the far blocks' norm."""
import os
import subprocess

import numpy as np
import pytest

from surfaceonlydeformables_amd import abi
from surfaceonlydeformables_amd import mesh as M

HERE = os.path.dirname(os.path.abspath(__file__))


def test_parts_take_every_point_once(tmp_path):
    out = tmp_path / "check"
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    r = subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O2", "-std=c++17", "-o", str(out),
                        os.path.join(HERE, "part_points_check.cpp")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    asked = [(n, s) for n in range(1, 60) for s in (1, 2, 4)]
    r = subprocess.run([str(out)], input="\n".join(f"{n} {s}" for n, s in asked) + "\n", capture_output=True, text=True,
                       timeout=60)
    for (n, s), line in zip(asked, r.stdout.strip().split("\n"), strict=True):
        parts = line.split("-")[:-1]
        assert len(parts) == s
        assert sorted(int(q) for p in parts for q in p.split()) == list(range(n)), (n, s)


def sphere(nf):
    V, F = M.icosphere(3, 0.2)
    V, F = abi.decimate_mesh(M.jitter(V, F, 0.01, nf), F, nf)
    return M.center(V, F), F


# last patches of 45 faces (one chunk, shared by 4 waves) and of 76 (two chunks, 2 waves each)
@pytest.mark.gpu
@pytest.mark.parametrize("nf,listed", [(530, 45), (554, 76)])
@pytest.mark.parametrize("far_order", [1, 2])
@pytest.mark.parametrize("order,sub", [(5, 2), (2, 4)])
def test_small_far_rules(nf, listed, far_order, order, sub):
    V, F = sphere(nf)
    assert len(F) == nf
    mesh, L, l, nv = abi.make_mesh(V, F), 16, 5, len(V)
    _, c1, c2 = M.material_speeds(3e5, 0.33, 1000.0)
    args = (c1, c2, 1000.0, 0.33, 0.4 / (c2 * (L - 2)), 1e-10 ** (1 / (2 * L)), L)
    which = abi.G | abi.H
    band = abi.make_params(*args, order=order, subdivision=sub, which=which, quad=abi.QUAD_BANDED, far_order=far_order,
                           far_subdivision=1, band_kappa=1e-300)
    pov, far = abi.band_plan(mesh, band)
    small = far.shape[1] - 1
    assert (pov[F] == small).any(axis=1).sum() == listed and far[:, small].any()
    ctx = abi.Context(0)
    print(f"far rule of order {far_order} beside {order}x{sub}, last patch of {listed} faces", flush=True)
    got = ctx.laplace(mesh, band, l)
    ref = ctx.laplace(mesh, abi.make_params(*args, order=order, subdivision=sub, which=which), l)
    low = ctx.laplace(mesh, abi.make_params(*args, order=far_order, subdivision=1, which=which), l)
    ctx.close()
    tile = far[:, pov]
    for k in ("U", "P"):
        g, r, w = (x[k].reshape(nv, 3, nv, 3).transpose(0, 2, 1, 3) for x in (got, ref, low))
        assert np.array_equal(g[~tile], r[~tile]), k
        assert np.linalg.norm(g[tile] - w[tile]) <= 1e-12 * np.linalg.norm(w[tile]), k

"""The regular kernels' exponentials e^{-s r / c} from the per-block table (cqbem_device.hpp: exp_pair), built for the host
from the same header and checked against mpmath at 120 bits.

Errors are of a complex value in units of 2^-53 of its modulus.  The table's value is a sum whose last rounding leaves at most
sqrt(2) and whose terms before it are |v| <= 1.3 times as large, with some four roundings: 6 at most anywhere.  The
direct functions' argument is rounded, so that their error grows with it.  The table must be no less exact than they are, in
the root mean square over every decade of |s r / c2|, for the pair and for what the kernels form from it: A1 - A2 with
A = (z + 1) e (twice s^2 A), up to 5% of sampling.  Frequencies beyond the table's reach take the direct functions."""
import math
import os
import random
import subprocess

import pytest

mp = pytest.importorskip("mpmath")

HERE = os.path.dirname(os.path.abspath(__file__))
ULP = 2.0 ** -53


@pytest.fixture(scope="module")
def check_bin(tmp_path_factory):
    out = tmp_path_factory.mktemp("exppair") / "check"
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    r = subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O2", "-std=c++17", "-o", str(out),
                        os.path.join(HERE, "exp_pair_check.cpp")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    return str(out)


def run(binary, sc1, sc2, reach, rs):
    text = f"{sc1.real!r} {sc1.imag!r} {sc2.real!r} {sc2.imag!r} {reach!r} {len(rs)}\n" + "\n".join(repr(r) for r in rs) + "\n"
    r = subprocess.run([binary], input=text, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    lines = r.stdout.strip().split("\n")
    rows = [[float.fromhex(t) for t in l.split()] for l in lines[1:]]
    return int(lines[0]), [[complex(v[2 * k], v[2 * k + 1]) for k in range(4)] for v in rows]


def off(got, want):
    return float(abs(mp.mpc(got) - want)) / ULP


def rms(v):
    return math.sqrt(sum(x * x for x in v) / len(v))


# |s reach / c2| and the angle of s; the last near the table's reach
@pytest.mark.parametrize("size", [1e-2, 1.0, 10.0, 40.0, 70.0, 98.0])
@pytest.mark.parametrize("angle", [0.3, 1.2, -1.5])
def test_no_less_exact_than_the_direct_functions(check_bin, size, angle):
    mp.mp.prec = 120
    reach, ratio = 0.37, 0.46
    sc2 = size / reach * complex(math.cos(angle), math.sin(angle))
    sc1 = sc2 * ratio
    rng = random.Random(int(size * 100) + int(angle * 10))
    top = size
    while top > max(size / 400, 1e-3):
        rs = [reach * math.exp(rng.uniform(math.log(top / 10 / size), math.log(top / size))) for _ in range(1500)] + [reach * top / size]
        beyond, rows = run(check_bin, sc1, sc2, reach, rs)
        assert not beyond
        err = {k: [] for k in ("table", "direct", "table dA", "direct dA")}
        for r, v in zip(rs, rows, strict=True):
            z1, z2 = mp.mpc(sc1) * mp.mpf(r), mp.mpc(sc2) * mp.mpf(r)
            e1, e2 = mp.exp(-z1), mp.exp(-z2)
            d = (z1 + 1) * e1 - (z2 + 1) * e2
            for name, a, b in (("table", v[0], v[1]), ("direct", v[2], v[3])):
                err[name] += [off(a, e1) / float(abs(e1)), off(b, e2) / float(abs(e2))]
                # the pair's own part of the difference: its later roundings are the same for both
                err[name + " dA"].append(off((z1 + 1) * mp.mpc(a) - (z2 + 1) * mp.mpc(b), d))
        print(f"|z2| up to {top:.3g}: table {rms(err['table']):.2f} (largest {max(err['table']):.2f}), direct "
              f"{rms(err['direct']):.2f} ({max(err['direct']):.2f}), dA {rms(err['table dA']):.2f} and {rms(err['direct dA']):.2f}")
        assert max(err["table"]) <= 6.0
        assert rms(err["table"]) <= 1.05 * rms(err["direct"])
        assert rms(err["table dA"]) <= 1.05 * rms(err["direct dA"])
        top /= 10


def test_beyond_the_reach(check_bin):
    reach = 0.37
    for size, want in ((1.0, 0), (98.0, 0), (110.0, 1), (1e5, 1)):
        sc2 = size / reach * complex(math.cos(1.1), math.sin(1.1))
        assert run(check_bin, sc2 * 0.5, sc2, reach, [0.1])[0] == want


def test_every_cell_and_the_ends(check_bin):
    """One distance in the middle and one at each end of every cell, and the whole reach."""
    mp.mp.prec = 120
    reach = 0.37
    sc2 = 90.0 / reach * complex(math.cos(1.0), math.sin(1.0))
    cells = 63 * 128 - 64
    h = reach / (cells - 1.5)
    rs = [h * (k + t) for k in range(0, cells - 2, 13) for t in (0.0, 0.5, 1 - 1e-9)] + [reach, h * 1e-6]
    _, rows = run(check_bin, sc2 * 0.6, sc2, reach, rs)
    for r, v in zip(rs, rows, strict=True):
        for sc, e in ((sc2 * 0.6, v[0]), (sc2, v[1])):
            want = mp.exp(-mp.mpc(sc) * mp.mpf(r))
            assert off(e, want) <= 6.0 * float(abs(want)), r

"""CPU checks of the pair kernels' shared arithmetic (host build): the box grid,
the Coulomb factors and the fused fixed-point product."""

import ctypes
import math
import subprocess
from fractions import Fraction
from pathlib import Path

import numpy as np
import pytest
from scipy.special import erfc

ROOT = Path(__file__).resolve().parents[1]
D = ctypes.c_double


@pytest.fixture(scope="module")
def pc(tmp_path_factory):
    out = tmp_path_factory.mktemp("pc") / "pair_check.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC",
                    f"-I{ROOT / 'timemachine_amd' / 'csrc'}", str(ROOT / "tests" / "native" / "pair_check.cpp"), "-o",
                    str(out)], check=True)
    lib = ctypes.CDLL(str(out))
    for name, n in (("pc_wrap", 2), ("pc_delta", 3), ("pc_frame_delta", 4), ("pc_edge", 1)):
        getattr(lib, name).restype = D
        getattr(lib, name).argtypes = [D] * n
    lib.pc_es.argtypes = [D, D, ctypes.POINTER(D)]
    lib.pc_product.restype = ctypes.c_uint64
    lib.pc_product.argtypes = [D, D]
    lib.pc_product3.argtypes = [D] * 5 + [ctypes.POINTER(ctypes.c_uint64)]
    return lib


@pytest.mark.parametrize("L", [2.65, 3.0, 4.0, 4.0000001, 7.07, 8.0, 33.3])
def test_displacements_on_the_box_grid_are_exact(pc, L):
    """Wrapped coordinates are within half a grid step (2^-53 of the power of two
    at or above L, plus the rounding of the wrap itself) of the periodic image,
    and the displacement of two atoms has the same bits from any images and from
    any frame that holds the pair unsplit: it is the exact rational difference."""
    rng = np.random.default_rng(1)
    top = 2.0 ** math.ceil(math.log2(L))
    edge = Fraction(pc.pc_edge(L))
    assert abs(float(edge) - L) <= top * 2.0**-53
    for _ in range(400):
        xi = rng.uniform(-3 * L, 3 * L)
        xj = xi + rng.uniform(-0.45 * L, 0.45 * L) + L * int(rng.integers(-2, 3))
        wi, wj = pc.pc_wrap(L, xi), pc.pc_wrap(L, xj)
        n = round((xi - wi) / L)
        assert abs(Fraction(wi) + n * edge - Fraction(xi)) <= Fraction(top) / 2**52
        d = Fraction(wi) - Fraction(wj)
        d -= round(d / edge) * edge
        assert Fraction(pc.pc_delta(L, xi, xj)) == d
        assert Fraction(pc.pc_delta(L, xj, xi)) == -d
        c = wi + rng.uniform(-0.02 * L, 0.02 * L)  # a block's centre lies among wrapped coordinates
        assert Fraction(pc.pc_frame_delta(L, xi, xj, c)) == d


@pytest.mark.parametrize("L", [3.1, 40.0, 999.0, 2.0**20 - 1, 2.0**20, 1.7e6, 1e9, 1e12])
def test_grid_error_stays_below_the_pair_terms(pc, L):
    """Pairs near the origin of a box of any size: the grid moves a displacement by
    at most 2^-52 times the power of two above L per axis, and by nothing from 2^20 nm on,
    where that would pass 2.4e-10 nm (a relative 3e-8 of the steepest pair force at 0.1 nm,
    the FP32 exponential of the Coulomb term has 1.2e-7)."""
    rng = np.random.default_rng(3)
    for _ in range(200):
        xi = rng.uniform(-2, 2)
        xj = xi + rng.uniform(-1.2, 1.2)
        got = Fraction(pc.pc_delta(L, xi, xj))
        if L < 2.0**20:
            assert abs(got - (Fraction(xi) - Fraction(xj))) <= Fraction(2.0 ** math.ceil(math.log2(L)) * 2.0**-52)
        else:
            assert got == Fraction(xi - xj)


def test_coulomb_factors(pc):
    """Force bracket and erfc against the closed forms over the fit's range
    (x up to 3): the FP32 exponential's 1.2e-7 and the fit's 2e-8. The paired
    evaluation has the single one's bits."""
    out = (D * 4)()
    for beta in (2.0, 1.3):
        for d in np.linspace(0.05, 1.5, 900):
            pc.pc_es(d * d, beta, out)
            x = beta * d
            bracket = erfc(x) + 2 * x / math.sqrt(math.pi) * math.exp(-x * x)
            assert abs(out[0] * d**3 / bracket - 1) < 1.4e-7
            assert abs(out[1] * d / erfc(x) - 1) < 1.4e-7
            assert out[2] == out[0] and out[3] == out[1]


def test_product_to_fixed_rounds_once(pc):
    """round(a b) to the nearest integer, ties to even, from the exact product."""
    rng = np.random.default_rng(2)
    out = (ctypes.c_uint64 * 3)()
    for _ in range(2000):
        a = float(rng.normal() * 2.0 ** rng.integers(0, 50))
        v = rng.uniform(-1.2, 1.2, 3)
        pc.pc_product3(a, 1.2, *v, out)
        for k in range(3):
            want = round(Fraction(a) * Fraction(float(v[k])))
            assert pc.pc_product(a, float(v[k])) == want % 2**64
            assert out[k] == want % 2**64
    # large products, overflow and NaN go the general way
    for a, b in ((2.0**51, 1.0), (2.0**40, 2.0**15), (-(2.0**61), 1.5), (2.0**62, 4.0), (math.nan, 1.0), (math.inf, 0.5)):
        want = 1 << 63 if not abs(a * b) < 2.0**63 else int(a * b) % 2**64
        assert pc.pc_product(a, b) == want
        pc.pc_product3(a, abs(b), b, b, b, out)
        assert list(out) == [want] * 3

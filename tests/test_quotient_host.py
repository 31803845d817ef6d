"""The host check that lets a mesh take FP64 quotients from reciprocals
(csrc/pf_quotient.hpp): where it agrees, the three operations give the
correctly rounded quotient (against integer division) for random dividends
and for those whose quotients lie nearest a rounding boundary; with a
reciprocal that is wrong it refuses."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "phonomena_amd", "csrc")
SOURCE = """
#include "%s/pf_quotient.hpp"
extern "C" int allowed(double b, double y) { return pf::quotients_exact(b, y); }
extern "C" int spacing_allowed(double h) { return pf::quotient_exact(h); }
extern "C" double quotient(double a, double b, double y) {
    const double q = a * y;
    return std::fma(std::fma(-b, q, a), y, q);
}
""" % CSRC


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("quotient")
    (d / "q.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", "-o", str(d / "q.so"),
                    str(d / "q.cpp")], check=True)
    so = ctypes.CDLL(str(d / "q.so"))
    so.allowed.argtypes = [ctypes.c_double] * 2
    so.spacing_allowed.argtypes = [ctypes.c_double]
    so.quotient.argtypes = [ctypes.c_double] * 3
    so.quotient.restype = ctypes.c_double
    return so


def _rounded(A, B):
    """RN(A / B) of two 53-bit integers, by integer division."""
    w = 53 if A < B else 52  # the quotient's 53 bits
    q, r = divmod(A << w, B)
    q += 2 * r > B or (2 * r == B and q & 1)
    return float(q) * 2.0 ** -w


def _near_boundaries(B, most):
    """53-bit dividends with A 2^w = B M + t, M odd of 54 bits, 0 < |t| <= most."""
    z = (B & -B).bit_length() - 1
    out = []
    for w in (53, 54):
        for t in range(-most, most + 1):
            if t == 0 or t % (1 << z):
                continue
            mod = 1 << (w - z)
            M = (-(t >> z) * pow(B >> z, -1, mod)) % mod
            while M < 1 << 54:
                if M >= 1 << 53 and M & 1 and (B * M + t) >> w << w == B * M + t:
                    A = (B * M + t) >> w
                    if 1 << 52 <= A < 1 << 53:
                        out.append(A)
                M += mod
    return out


def _divisors():
    rng = np.random.default_rng(11)
    special = [(1 << 52) + 1, (1 << 53) - 1, 3 << 51, 5 << 50, (1 << 52) + (1 << 26), (1 << 53) - (1 << 5),
               (1 << 53) - (1 << 4), (1 << 52) + (1 << 4), (1 << 52) + (1 << 5), 0x1999999999999a, 0x13333333333333,
               0x1a36e2eb1c432d, 6369051672525773, (1 << 52) + 3]  # 0.1, 0.3 x 2, 1e-4, sqrt(2), ...
    return special + [int(v) for v in rng.integers(1 << 52, 1 << 53, 150)]


def test_quotients_are_correctly_rounded_where_allowed(lib):
    rng = np.random.default_rng(12)
    allowed = 0
    for B in _divisors():
        b = float(B)
        y = 1.0 / b
        if not lib.allowed(b, y):
            continue
        allowed += 1
        for A in _near_boundaries(B, 48) + [int(v) for v in rng.integers(1 << 52, 1 << 53, 50)]:
            assert lib.quotient(float(A), b, y) == _rounded(A, B), (A, B)
    assert allowed > 0


def test_every_dividend_it_tries_is_one_of_the_nearest(lib):
    """The check decides by the dividends up to |t| = 16: perturbing the
    reciprocal until one of them fails must make it refuse, and only then."""
    refused = agreed = 0
    for B in _divisors():
        b = float(B)
        near = _near_boundaries(B, 16)
        for rel in (0.0, 2.0 ** -51, 2.0 ** -45, -2.0 ** -40, 2.0 ** -30, -2.0 ** -26):
            y = 1.0 / b * (1.0 + rel)
            fails = any(lib.quotient(float(A), b, y) != _rounded(A, B) for A in near)
            if B & 31:
                assert bool(lib.allowed(b, y)) == (not fails), (B, rel)
            refused += fails
            agreed += not fails
    assert refused > 100 and agreed > 100


def test_spacings_are_judged_by_their_significand(lib):
    rng = np.random.default_rng(13)
    for h in np.exp(rng.uniform(np.log(1e-12), np.log(1e5), 2000)):
        assert lib.spacing_allowed(h)  # none that fails is known
        assert lib.spacing_allowed(h * 2.0 ** 37)

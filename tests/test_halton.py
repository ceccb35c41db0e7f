"""Halton sampler: the reference's radical inverse (src/util.cpp:22-32) and
the scrambled extension, pinned by closed forms, the stratification
property and an exact rational evaluation; product == oracle bit for bit."""
import os
import shutil
import subprocess
from fractions import Fraction

import numpy as np
import pytest

from globillum_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_radical_inverse_known_values(oracle):
    # closed form: base 2, n = 1..8 and base 3, n = 1..3
    exp2 = [0.5, 0.25, 0.75, 0.125, 0.625, 0.375, 0.875, 0.0625]
    assert [oracle.radical_inverse(n, 2) for n in range(1, 9)] == exp2
    assert oracle.radical_inverse(1, 3) == pytest.approx(1 / 3, rel=1e-7)
    assert oracle.radical_inverse(2, 3) == pytest.approx(2 / 3, rel=1e-7)
    assert oracle.radical_inverse(3, 3) == pytest.approx(1 / 9, rel=1e-7)
    assert oracle.radical_inverse(0, 5) == 0.0


def test_primes(oracle):
    first = [2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31, 37, 41, 43, 47]
    assert [oracle.prime(d) for d in range(15)] == first
    assert oracle.prime(227) == 1439 and oracle.prime(99) == 541  # 228th, 100th prime


@pytest.mark.parametrize("dim,seed", [(0, 0), (1, 7), (5, 3), (40, 11), (227, 1)])
def test_permutation_is_bijection(oracle, dim, seed):
    p = oracle.halton_perm(dim, seed)
    assert sorted(p.tolist()) == list(range(oracle.prime(dim)))


def test_permutations_depend_on_seed(oracle):
    assert not np.array_equal(oracle.halton_perm(30, 0), oracle.halton_perm(30, 1))
    assert np.array_equal(oracle.halton_perm(30, 5), oracle.halton_perm(30, 5))


def _exact(n, p, perm):
    """sum_k perm[d_k] p^-(k+1) + perm[0] p^-K / (p-1), as a rational."""
    r = Fraction(0)
    k = 0
    while n > 0:
        n, d = divmod(n, p)
        r += Fraction(int(perm[d]), p ** (k + 1))
        k += 1
    return r + Fraction(int(perm[0]), (p - 1) * p ** k)


@pytest.mark.parametrize("dim", [0, 1, 2, 7, 33, 100])
def test_scrambled_matches_exact_rational(oracle, dim):
    rng = np.random.default_rng(dim)
    p = oracle.prime(dim)
    perm = oracle.halton_perm(dim, 9)
    for n in [0, 1, 2, p - 1, p, p * p + 3] + rng.integers(0, 2 ** 32, 50).tolist():
        got = np.float32(oracle.halton_sample(int(n), dim, 9))
        ref = np.float32(float(_exact(int(n), p, perm)))
        assert abs(int(got.view(np.int32)) - int(ref.view(np.int32))) <= 1, (n, got, ref)


@pytest.mark.parametrize("dim", [0, 1, 3, 9])
def test_scrambled_stratification(oracle, dim):
    # the first p^2 points of a scrambled van der Corput sequence are
    # j/p^2 + tail with j = perm[d0]*p + perm[d1] running over all cells and
    # tail = perm[0]/(p-1)/p^2 (the digits beyond the second)
    p = oracle.prime(dim)
    m = p * p
    perm0 = int(oracle.halton_perm(dim, 4)[0])
    v = np.array([oracle.halton_sample(n, dim, 4) for n in range(m)], np.float64)
    cells = np.rint(v * m - perm0 / (p - 1)).astype(int)
    assert np.all(np.abs(v * m - perm0 / (p - 1) - cells) < 1e-4 * m)
    assert sorted(cells.tolist()) == list(range(m))


def test_product_matches_oracle_bitwise(oracle):
    lib = _lib.load()
    rng = np.random.default_rng(1)
    for _ in range(400):
        n = int(rng.integers(0, 2 ** 32))
        dim = int(rng.integers(0, 228))
        seed = int(rng.integers(0, 2 ** 31))
        a = np.float32(lib.gi_halton_sample(n, dim, seed))
        b = np.float32(oracle.halton_sample(n, dim, seed))
        assert a.view(np.uint32) == b.view(np.uint32)
    for n, base in [(1, 2), (77, 3), (12345, 7), (2 ** 31 + 5, 13)]:
        assert np.float32(lib.gi_radical_inverse(n, base)) == np.float32(oracle.radical_inverse(n, base))
    perm = np.zeros(oracle.prime(50), np.uint16)
    assert lib.gi_halton_permutation(50, 17, _lib.ptr(perm)) == 0
    assert np.array_equal(perm, oracle.halton_perm(50, 17))
    assert lib.gi_halton_prime(-1) == -1 and lib.gi_halton_prime(227) == 1439


@pytest.fixture(scope="module")
def sampler_check(tmp_path_factory):
    hipcc = next((c for c in ("/opt/rocm/bin/hipcc", shutil.which("hipcc")) if c and os.path.exists(c)), None)
    if hipcc is None:
        pytest.skip("hipcc not found")
    exe = str(tmp_path_factory.mktemp("sampler") / "sampler_check")
    r = subprocess.run([hipcc, "-O2", "-std=c++17", "-ffp-contract=off", "-x", "c++", "-D__HIP_PLATFORM_AMD__",
                        os.path.join(ROOT, "tests", "csrc", "sampler_check.cpp"),
                        os.path.join(ROOT, "globillum_amd", "csrc", "bvh_build.cpp"), "-pthread", "-o", exe],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    return exe


@pytest.mark.parametrize("seed", [0, 7, 2 ** 32 - 1])
def test_kernel_sampler_on_the_host(sampler_check, seed):
    """The kernels' sampler function and tables, compiled for the host
    (tests/csrc/sampler_check.cpp): the bounds they rest on hold for every
    dimension of a depth-32 render, and the values are the digit loop's at the
    chunks' boundaries, the ends of the range and 20000 random indices each."""
    r = subprocess.run([sampler_check, str(seed), "20000"], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and "bad: bounds 0 edges 0 random 0" in r.stdout, r.stdout[-2000:]


@pytest.mark.parametrize("dim", [0, 1, 2, 53, 54, 227])
def test_digit_split_keeps_the_rational(oracle, dim):
    """Counting leading zeros as digits, up to a fixed number of them, leaves
    A / B as it is (the kernels' splits always count as many)."""
    p = oracle.prime(dim)
    perm = oracle.halton_perm(dim, 7).astype(np.int64)
    rng = np.random.default_rng(dim)
    for n in [0, 1, p - 1, p, 2 ** 32 - 1] + [int(x) for x in rng.integers(0, 2 ** 32, 8)]:
        exact = _exact(n, p, perm)
        k = 0
        while p ** k < 2 ** 32:
            k += 1
        for digits in range(k, k + 3):
            rev, x = 0, n
            for _ in range(digits):
                rev = rev * p + int(perm[x % p])
                x //= p
            assert x == 0 and Fraction(rev * (p - 1) + int(perm[0]), p ** digits * (p - 1)) == exact

"""The precision of the contractions on bf16 parts: bounds against 64 bits that hold with all six products of the parts
and fail where any one of them is missing.  The emulation below shows that they fail; it runs on the CPU.

Data that makes every product count: numbers whose second part is 0.996 of the largest there is (2^-8 of the number)
and whose third part is half of the largest, all of the sign of the number, so that what a missing product leaves out of a
sum of n terms has the sign of the terms."""
import numpy as np
import pytest

import orc_binding as ob

SIZES = [(22, 40), (64, 128)]
SCALE = -2.8853900817779268  # GEMM1 contracts x with this times W1
ALL = ("hh", "hm", "mh", "hl", "lh", "mm")

# h = tanh(p) from FP32 arithmetic: the sum p rounds once per product of the parts (6 per 24 or 32 terms) and its error is
# multiplied by at most 1, exp2, 1 + e, the reciprocal and 2 s - 1 add about 2^-23 each: 4e-7 for |p| <= 2.
# With one product missing p is off by 7.5e-6 of itself or more (in h: 4e-6).
BOUND_ACTIVATION = 1e-6
# a product of two FP32 numbers, relative: u = s - s^2 carries an error of s of about 1e-7 times |1 - 2 s| / u <= 4 for
# |p| <= 2, and half a dozen factors round to 2^-24 each: 8e-7 (measured 2.7e-7 and 5.1e-7).  With one product missing:
# 4e-6 or more.
BOUND_PRODUCT = 2e-6
TARGET = 40.0  # far from every prediction: the residual has no cancellation


def telling_numbers(rng, shape, exponents):
    """Random sign and power of two, significand 1 + 0x7f3f / 2^23."""
    bits = (rng.integers(0, 2, shape).astype(np.uint32) << np.uint32(31)) | np.uint32(0x7F3F)
    bits |= (127 + rng.choice(exponents, shape)).astype(np.uint32) << np.uint32(23)
    return bits.view(np.float32)


def make(d0, d1, n, seed):
    rng = np.random.default_rng(seed)
    X = telling_numbers(rng, (n, d0), [-1, 0])
    low = -3 if d0 == 22 else -4
    W1 = (telling_numbers(rng, (d0, d1), [low, low + 1]) / np.float32(SCALE)).astype(np.float32)
    b1 = (telling_numbers(rng, d1, [-2, -1]) / np.float32(SCALE)).astype(np.float32)
    w2 = rng.uniform(0.5, 1.0, d1).astype(np.float32)
    return X, W1, b1, w2


def params(W1, b1, w2):
    return np.concatenate([W1.ravel(), b1, w2, [0.0]]).astype(np.float32)


# ---- emulation -----------------------------------------------------------------------------------------------------
def bf16(x):
    b = x.astype(np.float32).view(np.uint32)
    b = (b + np.uint32(0x7FFF) + ((b >> np.uint32(16)) & np.uint32(1))) & np.uint32(0xFFFF0000)
    return b.view(np.float32).astype(np.float64)


def parts(x):
    h = bf16(x)
    m = bf16(x - h)
    return dict(h=h, m=m, l=x - h - m)


def contract(A, B, products):
    a, b = parts(A), parts(B)
    return sum(a[p[0]] @ b[p[1]] for p in products)


def activation_error(d0, d1, products):
    X, W1, b1, _ = (v.astype(np.float64) for v in make(d0, d1, 64, d0))
    p = X @ W1 + b1
    t = contract(X, W1 * SCALE, products) + b1 * SCALE
    h = 2.0 / (1.0 + 2.0**t) - 1.0
    return np.abs(h - np.tanh(p)).max()


def product_error(d0, d1, products):
    X, W1, b1, w2 = (v.astype(np.float64) for v in make(d0, d1, 16, d0 + 1))
    h = np.tanh(X @ W1 + b1)
    g = (TARGET - h @ w2)[:, None]
    u = (1 - h * h) / 4
    worst = 0.0
    for r in range(16):
        A, B = ((u * g), X) if d0 == 22 else (u, X * g)
        A, B = A[r].astype(np.float32).astype(np.float64), B[r].astype(np.float32).astype(np.float64)
        exact = np.outer(A, B)
        worst = max(worst, (np.abs(contract(A[:, None], B[None], products) - exact) / np.abs(exact)).max())
    return worst


@pytest.mark.parametrize("d0,d1", SIZES)
def test_the_bounds_need_every_product(d0, d1):
    assert activation_error(d0, d1, ALL) < BOUND_ACTIVATION / 4
    assert product_error(d0, d1, ALL) < BOUND_PRODUCT / 4
    for missing in ALL:
        rest = [p for p in ALL if p != missing]
        assert activation_error(d0, d1, rest) > 2 * BOUND_ACTIVATION, missing
        assert product_error(d0, d1, rest) > 2 * BOUND_PRODUCT, missing


# ---- the kernels ---------------------------------------------------------------------------------------------------
def sampler(pkg, lib, d0, d1, n, X, y, launch):
    model = lib.default_model(d0=d0, d1=d1, n=n, lik_kind=pkg.LIK_GAUSSIAN, lik_scale=1.0, prior_scale=1e6)
    s = lib.create(model, lib.default_hmc(), launch, 1, 1)
    s.set_window_data(0, X, y)
    return s


@pytest.mark.gpu
@pytest.mark.parametrize("d0,d1", SIZES)
def test_first_contraction(pkg, lib, d0, d1):
    """One hidden unit at a time through the rows' log-likelihood."""
    n = 64
    X, W1, b1, _ = make(d0, d1, n, d0)
    h = np.tanh(X.astype(np.float64) @ W1 + b1)
    s = sampler(pkg, lib, d0, d1, n, X, np.ones(n, np.float32), lib.default_launch())
    worst = 0.0
    for c in range(d1):
        w2 = np.zeros(d1, np.float32)
        w2[c] = 1.0
        ell = s.eval(0, params(W1, b1, w2))[0].astype(np.float64)
        d = 1.0 - h[:, c]
        want = -0.5 * d * d - 0.5 * np.log(2 * np.pi)
        # ell itself is rounded a few times
        off = (np.abs(ell - want) - 4 * 2.0**-24 * np.abs(want)).clip(0) / d
        worst = max(worst, off[d > 0.25].max())
    s.close()
    assert worst <= BOUND_ACTIVATION, worst


@pytest.mark.gpu
@pytest.mark.parametrize("d0,d1", SIZES)
def test_second_contraction(pkg, lib, d0, d1):
    """Rows of zeros but for one: the gradient of W1 is an outer product, each entry one product of two numbers.  Every
    row of a tile takes its turn."""
    X, W1, b1, w2 = make(d0, d1, 16, d0 + 1)
    worst = 0.0
    for r in range(16):
        Xr = np.zeros_like(X)
        Xr[r] = X[r]
        s = sampler(pkg, lib, d0, d1, 16, Xr, np.full(16, TARGET, np.float32), lib.default_launch())
        grad = s.eval(0, params(W1, b1, w2))[2][: d0 * d1].reshape(d0, d1).astype(np.float64)
        s.close()
        x, w = X[r].astype(np.float64), w2.astype(np.float64)
        h = np.tanh(x @ W1 + b1)
        want = np.outer(x, (1 - h * h) * w * (TARGET - h @ w)) - W1.astype(np.float64) * 1e-12
        worst = max(worst, (np.abs(grad - want) / np.abs(want)).max())
    assert worst <= BOUND_PRODUCT, worst

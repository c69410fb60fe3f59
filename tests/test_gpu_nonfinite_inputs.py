"""Features and first-layer weights that have no bf16 parts (infinite, or beyond the largest bf16 number) on the layers
that contract parts: FP32 arithmetic throughout, as in the oracle.  An infinite feature saturates the hidden units of
its row and leaves every other row alone."""
import numpy as np
import pytest

import orc_binding as ob
from hipmem import DevBuf

pytestmark = pytest.mark.gpu

HUGE = np.float32(3.4e38)  # finite; rounds to an infinite bf16 number


def student(lib, n, d0, d1):
    return lib.default_model(d0=d0, d1=d1, n=n), ob.Model(d0, d1, n, ob.LIK_STUDENT_T, 100.0, 2.2, 200.0)


def window(orc, d0, d1, n):
    X, y, th = orc.gen_window(n, 0, n, d0=d0, d1=d1, teacher_scale=0.15, noise_sigma=5.0)
    return X, y, (0.8 * th).astype(np.float32)


def check(got, want, what, rel=1e-5):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    assert (np.isnan(got) == np.isnan(want)).all(), (what, np.flatnonzero(np.isnan(got) != np.isnan(want))[:8])
    ok = ~np.isnan(want)
    np.testing.assert_allclose(got[ok], want[ok], rtol=rel, atol=rel * np.abs(want[ok]).max(), err_msg=what)


# n = 1000 at one workgroup: runs of 7 and 8 tiles; 100 at one: one tile per wave; at the default: every wave one tile
@pytest.mark.parametrize("d0,d1,n,G,threads", [(d0, d1, n, G, 0) for d0, d1 in [(22, 40), (64, 128)] for n, G in
                                               [(5, 1), (100, 1), (1000, 1), (1000, 0), (4099, 3)]] +
                         [(64, 128, 500, 1, 256)])
def test_features_without_parts(lib, orc, d0, d1, n, G, threads):
    model, om = student(lib, n, d0, d1)
    X, y, w = window(orc, d0, d1, n)
    s = lib.create(model, lib.default_hmc(seed=3), lib.default_launch(cus_per_chain=G, threads=threads), 1, 1)
    plain = orc.eval_f32(om, X, y, w)
    for value in (np.inf, -np.inf, HUGE, -HUGE):
        Xv = X.copy()
        rows = sorted({0, n // 3, n // 2, n - 1})  # the last one in the ragged tile
        for i, r in enumerate(rows):
            Xv[r, (0, d0 // 2, 17, d0 - 1)[i]] = value
        s.set_window_data(0, Xv, y)
        ell, prior, grad = s.eval(0, w)
        want = orc.eval_f32(om, Xv, y, w)
        assert np.isfinite(want[0]).all()
        check(ell, want[0], "rows, %g" % value)
        assert prior.tobytes() == want[1].tobytes()
        check(grad, want[2], "gradient, %g" % value)
        assert np.isnan(grad).any() == bool(np.isinf(value))
    # two infinities that cancel, an infinity on a zero weight, a NaN: those rows only
    Xv, wv = X.copy(), w.copy()
    wv[: 2 * d1] = np.abs(wv[: 2 * d1]) + np.float32(1e-3)
    wv[2 * d1 + 1] = 0.0
    Xv[0, :2] = np.inf, -np.inf
    Xv[n // 2, 2] = np.inf
    Xv[n - 1, 3] = np.nan
    s.set_window_data(0, Xv, y)
    check(s.eval(0, wv)[0], orc.eval_f32(om, Xv, y, wv)[0], "NaN rows")
    s.set_window_data(0, X, y)
    check(s.eval(0, w)[2], plain[2], "the same window without them")
    s.close()


@pytest.mark.parametrize("d0,d1", [(22, 40), (64, 128)])
def test_weights_without_parts(lib, orc, d0, d1):
    n = 300
    model, om = student(lib, n, d0, d1)
    X, y, w = window(orc, d0, d1, n)
    X[n // 2, 3] = 0.0
    X[7, 3] = np.float32(1e-38)
    s = lib.create(model, lib.default_hmc(seed=3), lib.default_launch(), 1, 1)
    s.set_window_data(0, X, y)
    for p, value in ((3 * d1 + 1, np.inf), (3 * d1 + d1 - 1, -np.inf), (3 * d1 + 5, HUGE / 2), (d0 * d1 + 2, np.inf),
                     (3 * d1 + 9, np.float32(1e37))):
        v = w.copy()
        v[p] = value
        check(s.eval(0, v)[0], orc.eval_f32(om, X, y, v)[0], "weight %d = %g" % (p, value))
    v = w.copy()
    v[3 * d1 + 1], v[4 * d1 + 1] = np.inf, -np.inf  # cancel in the rows whose features have the same sign
    want = orc.eval_f32(om, X, y, v)[0]
    assert np.isnan(want).any() and np.isfinite(want).any()
    check(s.eval(0, v)[0], want, "opposite infinities")
    s.close()


@pytest.mark.parametrize("d0,d1", [(22, 40), (64, 128)])
def test_final_losses_with_an_infinite_feature(lib, orc, d0, d1):
    """Its gradient is NaN, every proposal is rejected, and the losses are those of the start."""
    n = 500
    model, om = student(lib, n, d0, d1)
    X, y, w = window(orc, d0, d1, n)
    X[123, 5] = np.inf
    hmc = lib.default_hmc(leapfrog_steps=3, burn_in=0, n_samples=3, seed=4, eps0=1e-3)
    s = lib.create(model, hmc, lib.default_launch(), 1, 1)
    s.set_window_data(0, X, y)
    s.init_chains(w)
    s.run(3)
    assert (s.get_samples(0) == w).all() and s.get_chain_state(0)["n_accepted"] == 0
    ell, prior = orc.eval_f32(om, X, y, w)[:2]
    want = (ell.sum(dtype=np.float64), prior.sum(dtype=np.float64))
    loss1, loss2, full = s.final_loss(0)
    for got, ref in ((loss1, want[0]), (loss2, want[1]), (full, sum(want))):
        assert abs(got - ref) <= 1e-5 * abs(ref)
    s.close()


@pytest.mark.parametrize("d0,d1", [(22, 40), (64, 128)])
@pytest.mark.parametrize("offset", [0, 4])
def test_step_operator_with_an_infinite_feature(lib, orc, d0, d1, offset):
    n = 200
    model, om = student(lib, n, d0, d1)
    P = lib.num_params(d0, d1)
    X, y, w = window(orc, d0, d1, n)
    X[50, 2] = -np.inf
    X[199, 20] = HUGE
    launch = lib.default_launch()
    dX, dy = DevBuf.from_numpy(X, offset_bytes=offset), DevBuf.from_numpy(y, offset_bytes=offset)
    dw, z = DevBuf.from_numpy(w), DevBuf.full(P, 0.0)
    outs, loss = [DevBuf.full(P, np.nan) for _ in range(4)], DevBuf.full(n + P, np.nan)
    wsb = lib.step_workspace_bytes(model, launch)
    ws = DevBuf.full(wsb // 4 + 16, 0, np.int32)
    lib.mcmc_step(model, launch, dX.data_ptr, dy.data_ptr, dw.ptr, outs[0].ptr, z.ptr, outs[1].ptr, z.ptr, outs[2].ptr,
                  outs[3].ptr, loss.ptr, ws.ptr, wsb, 0.0, 1, 0)
    lib.step_check(model, launch, ws.ptr, 0)
    ell, prior, grad, _ = orc.eval_f32(om, X, y, w)
    check(loss.numpy(n + P), np.concatenate([ell, prior]), "loss values")
    check(outs[2].numpy(P), grad, "gradient")

"""Calls that hand results to the host: final losses of more samples than one batch of sums holds, several threads that
read one sampler, rows on either side of the size that goes through page-locked memory."""
import threading

import numpy as np
import pytest

import orc_binding as ob

pytestmark = pytest.mark.gpu


def sampler(lib, n, keep, L=1, launch=None, windows=1, chains=1, seed=5):
    model = lib.default_model(n=n)
    hmc = lib.default_hmc(leapfrog_steps=L, burn_in=0, n_samples=keep, seed=seed, eps0=1e-3)
    s = lib.create(model, hmc, launch or lib.default_launch(), windows, chains)
    th = [s.generate_window(w, teacher_scale=0.1, noise_sigma=1.0) for w in range(windows)]
    s.init_chains((0.9 * th[0]).astype(np.float32))
    s.run(keep)
    return s


def test_final_loss_of_more_samples_than_one_batch(lib, orc):
    n, keep = 3, 33001  # one chunk of rows: 32768 samples fill the sums once
    s = sampler(lib, n, keep, launch=lib.default_launch(transitions_per_launch=1000))
    om = ob.Model(22, 40, n, ob.LIK_STUDENT_T, 100.0, 2.2, 200.0)
    X, y = s.get_window_data(0)
    sums = []
    for w in s.get_samples(0):
        ell, prior = orc.eval_f64(om, X, y, w.astype(np.float64))[:2]
        sums.append((ell.sum(), prior.sum()))
    want = np.mean(sums, 0)
    loss1, loss2, full = s.final_loss(0)
    # each sample's sums are rounded to FP32, from FP32 rows of a few roundings each
    for got, ref in ((loss1, want[0]), (loss2, want[1]), (full, want.sum())):
        assert abs(got - ref) <= 16 * 2.0**-24 * abs(ref)
    s.close()


@pytest.mark.parametrize("losses_by", ["forward kernel", "whole evaluations"])
def test_threads_that_read_one_sampler(pkg, lib, losses_by):
    n, keep, chains = 2000, 6, 8
    layer = {"forward kernel": pkg.LAYER_MFMA, "whole evaluations": pkg.LAYER_FFMA}[losses_by]
    s = sampler(lib, n, keep, L=3, windows=2, chains=4, launch=lib.default_launch(layer=layer))
    rng = np.random.default_rng(0)
    ws = [(s.get_samples(0)[0] + rng.normal(0, 0.01, s.P)).astype(np.float32) for _ in range(chains)]

    def read(c):
        state = s.get_chain_state(c)
        ell, prior, grad = s.eval(c % 2, ws[c])
        return (s.get_samples(c).tobytes(), state["w"].tobytes(), state["grad"].tobytes(), state["eps"],
                state["n_accepted"], ell.tobytes(), prior.tobytes(), grad.tobytes())

    want, losses = [read(c) for c in range(chains)], {c: s.final_loss(c) for c in (3, 5)}
    wrong = []

    def work(c):
        for _ in range(40):
            if read(c) != want[c]:
                wrong.append(c)

    def work_losses(c):
        for _ in range(40):
            if s.final_loss(c) != losses[c]:
                wrong.append("losses")

    threads = [threading.Thread(target=work, args=(c,)) for c in range(chains)]
    threads += [threading.Thread(target=work_losses, args=(c,)) for c in losses]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong
    s.close()


@pytest.mark.parametrize("n", [(1 << 20) - 3, (1 << 20) + 5])
def test_rows_of_an_evaluation_whatever_their_number(lib, orc, n):
    model, om = lib.default_model(n=n), ob.Model(22, 40, n, ob.LIK_STUDENT_T, 100.0, 2.2, 200.0)
    s = lib.create(model, lib.default_hmc(seed=2), lib.default_launch(), 1, 1)
    th = s.generate_window(0, teacher_scale=0.1, noise_sigma=1.0)
    w = (0.9 * th).astype(np.float32)
    X, y = s.get_window_data(0)
    ell, prior, grad = s.eval(0, w)
    want = orc.eval_f32(om, X, y, w)
    np.testing.assert_allclose(ell, want[0], rtol=1e-5, atol=1e-5)
    assert prior.tobytes() == want[1].tobytes()
    assert np.abs(grad - want[2]).max() <= 1e-5 * np.abs(want[2]).max()
    s.close()

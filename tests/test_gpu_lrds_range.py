"""The replay where dv/dw times a signal leaves fp32's range and only the Frobenius clip
brings it back: the clip's factor of the tick itself, and of a later tick.

The reference here works as the entry point's contract does, in fp32 per operation: the
history is scaled by the factors so far, then multiplied by the signals (a product past
the range is infinite), clip ticks zero what is not finite.  Sums are taken in fp64, so a
result's own error is what fp32 sums of m = K_len bn products leave, sqrt(m) 2^-24 of the
largest partial sum; sixteen times that is allowed, over the ticks that carry it on."""
import numpy as np
import pytest

from heliox_amd import Sim, build_config

pytestmark = pytest.mark.gpu

F = np.float32


def replay32(it, dv, dp, blocks, dL, po, pre, dt, thr, every):
    n, ticks = it.shape[0], dL.shape[0]
    K_len = blocks[0].shape[2]
    K = np.zeros((n, n, K_len))
    s = 0
    for b in blocks:
        K[s:s + b.shape[0], s:s + b.shape[0]] = b
        s += b.shape[0]
    hist, sig, gs, dw = [np.zeros((n, n), F)], [F(1)], F(1), np.zeros(n)
    for t in range(1, ticks + 1):
        acc, base = np.zeros((n, n)), np.zeros((n, n))
        for tau in range(max(0, t - K_len), t):
            tap = K[:, :, K_len - t + tau]
            base += tap * it[:, tau + 1].astype(np.float64)[:, None]
            D = hist[tau]
            P = np.where(pre >= 0, D[:, np.maximum(pre, 0)], F(0))
            X = D * (sig[tau] * dv[:, tau + 1]) + P * (sig[tau] * dp[:, tau + 1])
            for j in range(n):                      # the taps of j's own block only
                k = np.nonzero(np.any(K[j] != 0, axis=1))[0]
                acc[:, j] += X[:, k].astype(np.float64) @ tap[j, k]
        out = (acc.astype(F) * F(dt) + base.astype(F) * F(dt) * gs).astype(F)
        sig.append(F(1))
        hist.append(out)
        if t % every == 0:
            out[~np.isfinite(out)] = 0
            l2 = np.sqrt(np.sum(out.astype(np.float64) ** 2))
            if l2 > thr:
                f = F(thr / l2)
                sig = [x * f for x in sig]
                gs *= f
                dw *= f
        dw += (out[:, po] * sig[-1]).astype(np.float64) @ dL[t - 1]
    return dw / ticks


@pytest.mark.parametrize("every,hot", [(1, "all"), (2, "second")])
def test_product_past_the_range_comes_back_with_the_clip(gpu_lib, every, hot):
    print(f"case lrds range every={every} hot={hot}", flush=True)
    rng = np.random.default_rng(every)
    bns, K_len, ticks = (6, 7), 3, 7
    n = sum(bns)
    blocks = [rng.uniform(0.2, 1.0, (b, b, K_len)).astype(F) for b in bns]
    it, dv, dp = (rng.uniform(0.1, 1.0, (n, ticks + 1)).astype(F) for _ in range(3))
    cols = np.arange(n) if hot == "all" else np.arange(bns[0], n)
    it[:, 3] *= F(1e30)                             # tick 3 is large, its products infinite
    dv[cols, 4] *= F(1e11)
    dp[cols, 4] *= F(1e11)
    pre = np.where(np.arange(n) < bns[0], rng.integers(-1, bns[0], n), rng.integers(bns[0], n, n)).astype(np.int32)
    po = np.array([0, 4, bns[0], n - 1], np.int32)
    dL = rng.normal(0, 1, (ticks, 4)).astype(F)
    with np.errstate(all="ignore"):
        want = replay32(it, dv, dp, blocks, dL, po, pre, 0.1, 1.0, every)
    assert np.all(np.isfinite(want)) and np.all(want != 0)
    g = Sim()
    g.load_model_from_spec(build_config(1, 1, 10.0))
    assert g.set_dense_blocks_f32(blocks) == K_len
    dw, dx = np.zeros(n, F), np.zeros((1, ticks), F)
    rc = g.replay_compute_dw_dx_from_signals_into(it, dv, dp, dL, po, np.zeros(1, np.int32), pre, dw, dx, 0.1, True,
                                                  eps=4.0, grad_l2norm_threshold=1.0, clip_check_every=every)
    assert rc == 0, g.last_error()
    err, scale = float(np.max(np.abs(dw - want))), float(np.max(np.abs(want)))
    tol = 16 * np.sqrt(K_len * max(bns)) * 2.0 ** -24 * ticks
    print(f"  dw max err {err:.3e} scale {scale:.3e} tol {tol:.1e}", flush=True)
    assert err <= tol * scale

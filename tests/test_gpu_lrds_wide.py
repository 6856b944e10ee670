"""Replays whose dv/dw slice has more than 2^32 elements, or whose correction has more
workgroups than one row of its grid, against the oracle.

All kernels are zero but those of a few blocks (the first, one in the middle, the last
two), so nothing else ever leaves zero: the oracle runs the few blocks alone, and every
other entry of dw has to be exactly 0.  The same bound as at the tile edges: an entry is
an fp32 sum of m = K_len (bn + 1) products, sqrt(m) 2^-24 of the largest partial sum,
sixteen times that."""
import numpy as np
import pytest

from heliox_amd import Sim, build_config
from oracle import lrds

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sim(gpu_lib):
    g = Sim()
    g.load_model_from_spec(build_config(1, 1, 10.0))
    yield g
    g.clear_dense_blocks()          # gives the slices back


@pytest.mark.parametrize("bn,nblk,last,K_len,percise,thr", [
    (32, 2048, 3, 2, False, 0.5),        # N = 65539: N^2 = 2^32 + 393225
    (32, 2048, 3, 2, True, 0.5),
    (32, 2043, 31, 2, False, 0.4),       # N = 65407: the last in 32 bits
    (2, 32769, 1, 1, True, 0.08),        # 32770 column tiles of 513 row tiles, 256 threads each
])
def test_wide_replay_matches_oracle(sim, bn, nblk, last, K_len, percise, thr):
    N, ksteps = bn * nblk + last, 5
    print(f"case lrds wide N={N} bn={bn} percise={percise}", flush=True)
    rng = np.random.default_rng(N + percise)
    bns = [bn] * nblk + [last]
    live = [0, nblk // 2, nblk - 1, nblk]
    zero = np.zeros((bn, bn, K_len), np.float32)
    blocks = [zero] * nblk + [None]
    for b in live:
        blocks[b] = (rng.normal(0, 1, (bns[b], bns[b], K_len)) * 0.3 / np.sqrt(bns[b])).astype(np.float32)
    cols = np.concatenate([np.arange(b * bn, b * bn + bns[b]) for b in live])
    n = cols.size
    it, dv, dp = (rng.normal(0, s, (N, ksteps + 1)).astype(np.float32) for s in (1.0, 0.3, 0.3))
    # a pre link within the live columns, to a dead column (0 ever) or none
    sub_pre = np.where(rng.random(n) < 0.6, rng.integers(0, n, n), -1)
    pre = rng.integers(-1, N, N).astype(np.int32)
    pre[cols] = np.where(sub_pre >= 0, cols[sub_pre], np.where(rng.random(n) < 0.5, bn, -1))
    out, inp = rng.permutation(n)[:min(n, 9)], np.array([0, n - 1])
    dL = rng.normal(0, 1, (ksteps, out.size)).astype(np.float32)
    assert sim.set_dense_blocks_f32(blocks) == K_len
    dw, dx = np.full(N, 7.0, np.float32), np.zeros((2, ksteps), np.float32)
    rc = sim.replay_compute_dw_dx_from_signals_into(
        it, dv, dp, dL, cols[out].astype(np.int32), cols[inp].astype(np.int32), pre, dw, dx, 0.1, percise,
        grad_scale=1.3, eps=4.0, grad_l2norm_threshold=thr)
    assert rc == 0, sim.last_error()
    rdw, rdx, hist = lrds.replay(it[cols], dv[cols], dp[cols], [blocks[b] for b in live], dL, out, sub_pre, dt=0.1,
                                 percise=percise, pinput=inp, grad_scale=1.3, eps=4.0, grad_l2norm_threshold=thr,
                                 clip_strategy=1, variant="signals", keep_history=True)
    assert any(np.linalg.norm(h) > thr * 0.999 for h in hist)         # the clip acts
    tol = 16 * np.sqrt(K_len * (bn + 1)) * 2.0 ** -24
    for name, a, r in (("dw", dw[cols], rdw), ("dx", dx, rdx)):
        err, scale = float(np.max(np.abs(a - r))), float(np.max(np.abs(r)))
        print(f"  {name} max err {err:.3e} scale {scale:.3e} tol {tol:.1e}", flush=True)
        assert err <= tol * scale + 1e-9
    assert not np.any(np.delete(dw, cols))

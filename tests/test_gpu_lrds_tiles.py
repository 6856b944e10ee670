"""The replay's correction GEMM at the edges of its tiles and splits, against the oracle:
column tiles of 32, 64 and 128 and one more or less, rows that do not fill a 128-row tile,
block widths that are not a multiple of 4 (padded rows), reductions of one chunk, of a few
(one per split) and of many, several taps per chunk, more ticks than one launch of the base
term makes, and an infinite signal on clip ticks.

An entry of dv/dw is an fp32 sum of m = K_len (bn + 1) products whose rounding errors add
up like a random walk, sqrt(m) 2^-24 of the largest partial sum; the bound allows sixteen
times that, relative to the largest result."""
import numpy as np
import pytest

from heliox_amd import Sim, build_config
from oracle import lrds

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sim(gpu_lib):
    g = Sim()
    g.load_model_from_spec(build_config(1, 1, 10.0))
    return g


CASES = [
    # bns, K_len, ksteps, percise, thr, infinite signal
    ((1,), 1, 3, True, 1e6, False),
    ((1, 2, 3), 4, 10, True, 1e6, False),
    ((31,), 2, 9, True, 1e6, False),
    ((32, 32), 3, 8, True, 0.05, False),
    ((33, 30), 2, 17, True, 1e6, False),
    ((63, 65), 2, 6, True, 1e6, False),
    ((127, 2), 1, 5, True, 1e6, False),
    ((128, 128, 1), 2, 9, True, 1e6, False),
    ((130,), 3, 7, True, 1e6, False),
    ((5,) * 40, 16, 25, True, 0.5, False),
    ((16, 17), 64, 70, True, 1e6, False),
    ((70, 58), 6, 19, False, 0.05, False),
    ((40, 23), 5, 12, True, 1.0, True),
    # more than one element a thread where the splits are summed: 4, 8 and 16
    ((200, 199, 131), 2, 7, True, 0.3, False),
    ((128,) * 8 + (77,), 2, 5, True, 0.3, False),
    ((300,) * 7 + (1,), 2, 4, False, 0.3, False),
    ((125,) * 12, 1, 3, True, 1e6, False),       # a tile for more than every other CU: no split
    ((20,) * 70, 1, 3, True, 1e6, False),        # the same with 32-column tiles
]


@pytest.mark.parametrize("bns,K_len,ksteps,percise,thr,inf", CASES)
def test_replay_at_tile_edges_matches_oracle(sim, bns, K_len, ksteps, percise, thr, inf):
    print(f"case lrds tiles bns={bns[:3]}x{len(bns)} K_len={K_len} ksteps={ksteps} percise={percise} thr={thr}",
          flush=True)
    rng = np.random.default_rng(len(bns) * 1000 + bns[0] + K_len)
    N, T = int(sum(bns)), ksteps + 1
    blocks = [(rng.normal(0, 1, (bn, bn, K_len)) * 0.3 / np.sqrt(bn)).astype(np.float32) for bn in bns]
    it, dv, dp = (rng.normal(0, s, (N, T)).astype(np.float32) for s in (1.0, 0.3, 0.3))
    if inf:
        dv[3, 4] = np.inf
    pre = np.where(rng.random(N) < 0.6, rng.integers(0, N, N), -1).astype(np.int32)
    po = np.sort(rng.choice(N, min(N, 9), replace=False)).astype(np.int32)
    pin = np.sort(rng.choice(N, min(N, 3), replace=False)).astype(np.int32)
    dL = rng.normal(0, 1, (ksteps, po.size)).astype(np.float32)
    assert sim.set_dense_blocks_f32(blocks) == K_len
    dw, dx = np.zeros(N, np.float32), np.zeros((pin.size, ksteps), np.float32)
    rc = sim.replay_compute_dw_dx_from_signals_into(it, dv, dp, dL, po, pin, pre, dw, dx, 0.1, percise, grad_scale=1.3,
                                                    eps=4.0, grad_l2norm_threshold=thr)
    assert rc == 0, sim.last_error()
    with np.errstate(all="ignore"):
        rdw, rdx, _ = lrds.replay(it, dv, dp, blocks, dL, po, pre, dt=0.1, percise=percise, pinput=pin, grad_scale=1.3,
                                  eps=4.0, grad_l2norm_threshold=thr, clip_strategy=1, variant="signals")
    assert np.all(np.isfinite(rdw)) and np.all(np.isfinite(rdx))
    # timed, dx runs apart from the correction: the same bits
    dw2, dx2 = np.zeros_like(dw), np.zeros_like(dx)
    sim.set_replay_timing(True)
    rc = sim.replay_compute_dw_dx_from_signals_into(it, dv, dp, dL, po, pin, pre, dw2, dx2, 0.1, percise, grad_scale=1.3,
                                                    eps=4.0, grad_l2norm_threshold=thr)
    ms, ticks = sim.replay_kernel_time()
    sim.set_replay_timing(False)
    assert rc == 0 and ms > 0 and ticks == ksteps
    assert np.array_equal(dw, dw2) and np.array_equal(dx, dx2)
    tol = 16 * np.sqrt(K_len * (max(bns) + 1)) * 2.0 ** -24
    for name, a, r in (("dw", dw, rdw), ("dx", dx, rdx)):
        err, scale = float(np.max(np.abs(a - r))), float(np.max(np.abs(r)))
        print(f"  {name} max err {err:.3e} scale {scale:.3e} tol {tol:.1e}", flush=True)
        assert err <= tol * scale + 1e-9


def test_base_term_of_fewer_ticks_where_memory_is_short(gpu_lib):
    """One block of 4000 columns: a tick's base terms are 64 MB, eight ticks' 512; with about
    700 MB free the replay (448 MB beside them) makes fewer at a time, and the same bits."""
    import ctypes as C

    print("case lrds base ticks in short memory", flush=True)
    rng = np.random.default_rng(4)
    N, ksteps = 4000, 9
    block = (rng.standard_normal((N, N, 1), np.float32) * np.float32(0.3 / np.sqrt(N)))
    it, dv, dp = (rng.normal(0, 0.3, (N, ksteps + 1)).astype(np.float32) for _ in range(3))
    pre = rng.integers(-1, N, N).astype(np.int32)
    po, pin = np.arange(0, N, 500, dtype=np.int32), np.array([3], np.int32)
    dL = rng.normal(0, 1, (ksteps, po.size)).astype(np.float32)
    out = []
    for short in (False, True):
        g = Sim()
        g.load_model_from_spec(build_config(1, 1, 10.0))
        with open("/proc/self/maps") as f:      # the runtime that the library runs on
            paths = {line.split()[-1] for line in f if "libamdhip64" in line}
        hip = C.CDLL(sorted(paths, key=lambda p: "torch" in p)[0])
        hold, free, total = C.c_void_p(), C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        if short:
            assert hip.hipMalloc(C.byref(hold), C.c_size_t(free.value - (700 << 20))) == 0
        dw, dx = np.zeros(N, np.float32), np.zeros((1, ksteps), np.float32)
        assert g.set_dense_blocks_f32([block]) == 1
        rc = g.replay_compute_dw_dx_from_signals_into(it, dv, dp, dL, po, pin, pre, dw, dx, 0.1, True, eps=4.0)
        why = g.last_error()
        g.clear_dense_blocks()
        if short:
            assert hip.hipFree(hold) == 0
        assert rc == 0, why
        out.append((dw, dx))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1]) and np.any(out[0][0])


def test_signal_buffers_serve_problems_of_other_sizes(gpu_lib):
    """One program replays problems of growing and shrinking sizes, with and without the
    precise term; each gives a fresh program's bits."""
    print("case lrds signal buffers", flush=True)
    rng = np.random.default_rng(8)
    kept = Sim()
    kept.load_model_from_spec(build_config(1, 1, 10.0))
    blocks, last = None, 0
    for n, ksteps, percise in [(40, 6, True), (40, 30, False), (200, 30, False), (200, 29, True), (40, 6, True),
                               (12, 4, False), (12, 5, True), (12, 60, True)]:
        if n != last:
            blocks, last = [(rng.normal(0, 0.1, (n // 2, n // 2, 3))).astype(np.float32) for _ in range(2)], n
            assert kept.set_dense_blocks_f32(blocks) == 3
        it, dv, dp = (rng.normal(0, 0.5, (n, ksteps + 1)).astype(np.float32) for _ in range(3))
        pre = rng.integers(-1, n, n).astype(np.int32)
        dL = rng.normal(0, 1, (ksteps, 2)).astype(np.float32)
        fresh = Sim()
        fresh.load_model_from_spec(build_config(1, 1, 10.0))
        assert fresh.set_dense_blocks_f32(blocks) == 3
        out = []
        for g in (kept, fresh):
            dw, dx = np.zeros(n, np.float32), np.zeros((2, ksteps), np.float32)
            rc = g.replay_compute_dw_dx_from_signals_into(it, dv, dp, dL, np.array([0, n - 1], np.int32),
                                                          np.array([1, 2], np.int32), pre, dw, dx, 0.1, percise, eps=4.0,
                                                          grad_l2norm_threshold=0.05)
            assert rc == 0, g.last_error()
            out.append((dw, dx))
        assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1]), (n, ksteps, percise)
        assert np.any(out[0][0])

"""The tree solve by substructuring (k_solve_split) against the round-by-round solve and the
oracle, at the sizes where it could go wrong: cells of a single node, of one chunk and one
more, packs of several cells, a level wider than a wavefront, more chunks than 512 threads
and more than the kernel takes, cells of unequal size; with the voltage and with the change
as the unknown; the pivots and the solution read after a step, through a handle, and after a
coefficient changed."""
import dataclasses

import numpy as np
import pytest

import oracle
from heliox_amd import Sim, build_config
from heliox_amd.spec import MechSpec, ModelSpec
from parity_util import V_TOL

pytestmark = pytest.mark.gpu

# Rounding alone separates the two orders of elimination: a step leaves a few ulp of v
# (1.4e-14 mV at 65 mV) times the matrix' condition (couplings of at most 4 a node over the
# capacitive 0.04: 100), and the cells are passive, so 40 steps stay below 1e-10 mV.
TOL = 1e-10


def chain(n):
    return [-1] + list(range(n - 1))


def star(n):
    return [-1] + [0] * (n - 1)


def bushy(n):
    rng = np.random.default_rng(n)
    return [-1] + [int(rng.integers(max(0, i - 6), i)) for i in range(1, n)]


def passive(parents, ncell, clamp):
    """`ncell` copies of one tree (see forest)."""
    return forest([parents] * ncell, clamp)


def forest(trees, clamp):
    """Cells of these trees with unequal couplings, pas everywhere; `clamp` adds a current
    injection, which leaves the change as the unknown."""
    ncell, n = len(trees), sum(len(t) for t in trees)
    par, free = np.full(n, -1, np.int32), ncell
    for c, t in enumerate(trees):
        node = np.concatenate([[c], free + np.arange(len(t) - 1)]).astype(np.int64)
        free += len(t) - 1
        par[node[1:]] = node[np.asarray(t[1:], np.int64)]
    rng = np.random.default_rng(31 * len(trees[0]) + ncell)
    a, b = -rng.uniform(0.05, 2.0, n), -rng.uniform(0.05, 2.0, n)
    deg = np.bincount(par[ncell:], minlength=n) if n > ncell else np.zeros(n)
    a[ncell:] /= np.maximum(1.0, deg[par[ncell:]])
    a[:ncell] = b[:ncell] = 0.0
    mechs = {"pas": MechSpec(np.arange(n, dtype=np.int32),
                             {"g_pas": rng.uniform(1e-4, 1e-3, n), "e_pas": rng.uniform(-75.0, -60.0, n)})}
    if clamp:
        mechs["IClamp"] = MechSpec(np.arange(ncell, dtype=np.int32),
                                   {"delay": np.full(ncell, 0.2), "dur": np.full(ncell, 5.0), "amp": np.full(ncell, 0.1)})
    return ModelSpec(ncell=ncell, parent=par, a=a, b=b, area=rng.uniform(50.0, 500.0, n), cm=np.ones(n), mechs=mechs)


def run(spec, split, tstop=1.0, groups=1, unit_cells=0, handle=None):
    g = Sim()
    g.set_cell_groups(groups)
    g.set_solve_unit_cells(unit_cells)
    g.set_solve_split(split)
    g.load_model_from_spec(dataclasses.replace(spec, monitors=[("global", "v", c) for c in range(spec.ncell)]))
    if handle:
        g.get_variable_handle(*handle)
    g.finitialize(-65.0)
    for _ in range(2):
        g.continue_run(tstop / 2)
    return g


@pytest.mark.parametrize("clamp", [False, True])
@pytest.mark.parametrize("shape,size,ncell,takes", [
    (chain, 1, 3, 1), (chain, 16, 5, 1), (chain, 17, 5, 1), (chain, 101, 9, 1), (star, 71, 2, 1), (bushy, 40, 30, 1),
    (bushy, 260, 3, 1), (bushy, 1000, 2, 1), (bushy, 1600, 1, 0)])
def test_split_solve_matches_the_rounds(gpu_lib, shape, size, ncell, takes, clamp):
    print(f"case split {shape.__name__} {size} x {ncell} clamp={clamp}", flush=True)
    spec = passive(shape(size), ncell, clamp)
    s, r = run(spec, True), run(spec, False)
    print("chunks", s.info("nchunk_total"), flush=True)
    assert s.info("solve_split") == takes and r.info("solve_split") == 0
    assert s.info("solve_voltage") == int(not clamp)
    assert float(np.max(np.abs(s.traces() - r.traces()))) < TOL
    for k in ("v", "rhs"):
        assert float(np.max(np.abs(s.get_array("global", k) - r.get_array("global", k)))) < TOL, k
    np.testing.assert_allclose(s.get_array("global", "d"), r.get_array("global", "d"), rtol=TOL)
    o = oracle.OracleSim(spec, monitors=[("global", "v", c) for c in range(ncell)])
    o.finitialize(-65.0)
    for _ in range(2):
        o.continue_run(0.5)
    assert float(np.max(np.abs(o.traces() - s.traces()))) < V_TOL


@pytest.mark.parametrize("unit_cells,groups", [(1, 1), (7, 1), (3, 2)])
def test_packs_change_no_bit(gpu_lib, unit_cells, groups):
    print(f"case split packs unit_cells={unit_cells} groups={groups}", flush=True)
    spec = build_config(5, 20, 5.0)
    base, g = run(spec, True, 5.0), run(spec, True, 5.0, groups, unit_cells)
    assert g.info("solve_split") == 1
    assert np.array_equal(base.traces(), g.traces())
    assert np.array_equal(base.get_array("global", "v"), g.get_array("global", "v"))


# cells of about 3, 200, 400 and 620 chunks: a workgroup size each
MIXED = [bushy(1000), bushy(330), bushy(640)] + [bushy(5), chain(3), bushy(330), chain(1), chain(20)]


@pytest.mark.parametrize("clamp", [False, True])
@pytest.mark.parametrize("small,unit_cells,launches", [(20, 1, 1), (600, 1, 4), (600, 3, 1), (2000, 3, 4)])
def test_cells_of_unequal_size(gpu_lib, small, unit_cells, launches, clamp):
    """One launch for all packs, padded to the largest, or one for each workgroup size."""
    print(f"case split unequal small={small} unit_cells={unit_cells} clamp={clamp}", flush=True)
    spec = forest(MIXED + [bushy(9)] * small, clamp)
    s, r = run(spec, True, unit_cells=unit_cells), run(spec, False, unit_cells=unit_cells)
    assert s.info("solve_split") == 1 and r.info("solve_split") == 0
    assert s.info("solve_split_launches") == launches
    assert float(np.max(np.abs(s.traces() - r.traces()))) < TOL
    for k in ("v", "rhs"):
        assert float(np.max(np.abs(s.get_array("global", k) - r.get_array("global", k)))) < TOL, k
    np.testing.assert_allclose(s.get_array("global", "d"), r.get_array("global", "d"), rtol=TOL)
    if unit_cells == 3:         # packs and classes change no bit
        one = run(spec, True, unit_cells=1, groups=1 if clamp else 2)
        assert np.array_equal(s.traces(), one.traces())
        assert np.array_equal(s.get_array("global", "v"), one.get_array("global", "v"))
    if small == 20:
        o = oracle.OracleSim(spec, monitors=[("global", "v", c) for c in range(spec.ncell)])
        o.finitialize(-65.0)
        for _ in range(2):
            o.continue_run(0.5)
        assert float(np.max(np.abs(o.traces() - s.traces()))) < V_TOL


def test_adjoint_of_cells_of_unequal_size(gpu_lib):
    """The transposed solve, launch by launch, against the rounds; a gradient is a sum over
    40 steps of terms that carry the solve's rounding (TOL, relative to the largest)."""
    print("case split unequal adjoint", flush=True)
    spec = forest(MIXED + [bushy(9)] * 600, True)
    out = []
    for split in (True, False):
        g = Sim()
        g.set_solve_unit_cells(1)
        g.set_solve_split(split)
        g.load_model_from_spec(spec, add_monitors=False)
        g.tape_begin(40)
        g.finitialize(-65.0)
        g.run(40.25 * spec.dt)
        assert g.info("solve_split_launches") == (4 if split else 0)
        loss = g.adjoint(np.arange(spec.ncell), np.full((40, spec.ncell), -60.0))
        out.append((loss, g.gradient("pas", "g_pas")))
    assert abs(out[0][0] - out[1][0]) <= 1e-12 * abs(out[1][0])
    scale = float(np.max(np.abs(out[1][1])))
    assert scale > 0 and float(np.max(np.abs(out[0][1] - out[1][1]))) < TOL * scale


def test_pivots_and_solution_on_demand(gpu_lib):
    spec = passive(bushy(60), 4, False)
    print("case split on demand", flush=True)
    plain, held = run(spec, True), run(spec, True, handle=("global", "rhs", 5))
    assert np.array_equal(plain.traces(), held.traces())        # a reader of rhs changes no voltage
    late = run(spec, True)
    late.set_variable_value(-1.5, "global", "a", 50)            # after the step that d and rhs belong to
    for k in ("d", "rhs"):
        want = plain.get_array("global", k)
        assert np.array_equal(held.get_array("global", k), want), k
        assert np.array_equal(late.get_array("global", k), want), k
    assert held.get_variables_by_handles([0])[0] == plain.get_variable_value("global", "rhs", 5)


def test_handles_and_monitors_of_the_solution(gpu_lib):
    """Handles of d and rhs read after every step, one written, and a monitor of rhs: the
    values of the arrays after the same steps."""
    spec = passive(bushy(60), 4, False)
    print("case split handles", flush=True)
    names = [("global", "rhs", 5), ("global", "d", 70)]
    held, plain, watched, rounds = run(spec, True), run(spec, True), run(spec, True), run(spec, False)
    hs = [held.get_variable_handle(*n) for n in names]
    m = [g.add_monitor(*names[0]) for g in (watched, rounds)]
    for _ in range(3):
        for g in (held, plain, watched, rounds):
            g.fadvance()
        got = held.get_variables_by_handles(hs)
        want = [plain.get_array("global", "rhs")[5], plain.get_array("global", "d")[70]]
        assert list(got) == want
        assert watched.get_variable_value(*names[0]) == want[0]
    a, b = watched.monitor_array(m[0]), rounds.monitor_array(m[1])
    assert a.size == b.size > 0 and float(np.max(np.abs(a - b))) < TOL and np.any(b != 0)
    held.fadvance()
    plain.fadvance()
    held.set_variable_by_handle(hs[0], 2.5)
    rhs = plain.get_array("global", "rhs")
    rhs[5] = 2.5
    assert np.array_equal(held.get_array("global", "rhs"), rhs)
    assert np.array_equal(held.get_array("global", "d"), plain.get_array("global", "d"))


def test_outputs_on_demand_after_a_reader_left(gpu_lib):
    """A transfer that named rhs and is gone leaves the solution made on every step; the
    outputs made later from the old voltages are the same run's without it."""
    spec = build_config(3, 2, 2.0)
    print("case split outputs after a transfer", flush=True)
    out = []
    for reader in (False, True):
        g = Sim()
        g.load_model_from_spec(spec)
        if reader:
            sid = g.add_gap_source(-1, "global", "rhs", 3)
            assert sid >= 0 and g.add_gap_target(sid, "capacitance", "cm", 3) == 0
            assert g.clear_all_gap_junctions() == 0
        g.finitialize(-65.0)
        g.continue_run(2.0)
        assert g.info("solve_split") == 1 and g.info("outputs_pending") == 1
        out.append([g.get_array(*k) for k in (("hh", "ina"), ("Ca_HVA", "ica"), ("pas", "i"), ("global", "v"))])
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_vecplay_into_the_solution(gpu_lib):
    """VecPlay writes its rhs entry after each solve; the other entries stay the solution's."""
    spec = passive(bushy(60), 4, False)
    print("case split vecplay into rhs", flush=True)
    out = []
    for split in (True, False):
        for late in (False, True):
            g = Sim()
            g.set_solve_split(split)
            g.load_model_from_spec(spec, add_monitors=False)
            g.finitialize(-65.0)
            if late:
                g.continue_run(0.5)
            assert g.add_vecplay("global", "rhs", 7, [0.0, 100.0], [3.0, 3.0]) == 0
            g.continue_run(0.5 if late else 1.0)
            out.append((g.get_array("global", "d"), g.get_array("global", "rhs")))
    for d, rhs in out:
        assert rhs[7] == 3.0
        np.testing.assert_allclose(d, out[2][0], rtol=TOL)
        assert float(np.max(np.abs(rhs - out[2][1]))) < TOL

"""GPU lanes against the oracle, through the C ABI.

The LU boundary must be bitwise the oracle's replay; operating points must be
bitwise the oracle's Newton on the same points, pivot tape and start (the
device physics, exp/log and the LU all round identically); and the golden
ngspice cases must match to the fixtures' own tolerances.
"""
import sys

import numpy as np
import pytest

import golden_cases as G
from espice_amd import circuits
from test_oracle_lu import random_system

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


@pytest.fixture(scope="module")
def lanes():
    from espice_amd import lanes as L
    L.load()
    return L


def test_tape_replay_bitwise_random_systems(lanes, oracle):
    rng = np.random.default_rng(11)
    checked = 0
    for t in range(48):
        n = int(rng.integers(2, 64))
        cp, ri, vals = random_system(rng, n, rng.random() * 0.3)
        q = rng.permutation(n).astype(np.uint32)
        if oracle.lu_factor(cp, ri, vals, q) is None:
            continue
        say(f"tape replay case {t} n={n} nnz={len(ri)}")
        lanes_n = 64
        a = vals[None, :] * (0.8 + 0.4 * rng.random((lanes_n, len(vals))))
        a[5] = vals
        a[7, 0] = np.nan
        a[9] = 0.0
        rhs = 2 * rng.random((lanes_n, n)) - 1
        tape = lanes.Tape(cp, ri, vals, q)
        ref = oracle.lu_replay(cp, ri, vals, q, a, rhs)
        tx = tape.export()
        t0 = ref["tape"]
        for k in ["pinv", "lp", "li", "up", "ui", "prow"]:
            assert np.array_equal(tx[k], t0[k]), k
        got = tape.replay(a, rhs)
        assert np.array_equal(got["fail"], ref["fail"])
        ok = ref["fail"] == 0
        for k in ["lx", "ux", "udiag", "dx"]:
            assert np.array_equal(bits(got[k][ok]), bits(ref[k][ok])), (t, k)
        tape.close()
        checked += 1
    assert checked >= 24


@pytest.mark.parametrize("tiling", [1, 2])
@pytest.mark.parametrize("name", sorted(G.load()))
def test_golden_cases_on_gpu(lanes, oracle, name, tiling):
    case = G.load()[name]
    deck, live, reader = G.build(case)
    say(f"golden {name} rows={live.shape[0]} tiling={tiling}")
    eng = lanes.Engine(deck.arrays())
    cp, ri, q = eng.pattern()
    c = oracle.Circuit(deck.arrays())
    ocp, ori, _, _ = c.pattern()
    assert np.array_equal(cp, ocp) and np.array_equal(ri, ori)
    got = eng.solve_op(live, tiling=tiling)
    assert (got["reasons"] == 0).all()
    misses, worst = G.check(case, got["x"], reader)
    assert misses == 0, worst
    ref = c.op(live, q, threads=4)
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    eng.close()


@pytest.mark.parametrize("tiling", [1, 2])
@pytest.mark.parametrize("family,lanes_n", [("inverter_chain", 256), ("ota_array", 256)])
def test_family_bitwise_against_oracle(lanes, oracle, family, lanes_n, tiling):
    fam = circuits.FAMILIES[family]()
    vals = fam.sample(2026, lanes_n)
    say(f"family {family} lanes={lanes_n} tiling={tiling}")
    eng = lanes.Engine(fam.deck.arrays())
    _, _, q = eng.pattern()
    got = eng.solve_op(vals, tiling=tiling)
    ref = oracle.Circuit(fam.deck.arrays()).op(vals, q, threads=8)
    assert np.array_equal(got["reasons"], ref["reasons"])
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    say(f"  converged {(got['reasons'] == 0).sum()}/{lanes_n} mean iters {got['iterations'].mean():.2f} "
        f"repivots {eng.timing().repivots}")
    eng.close()


@pytest.mark.parametrize("stages", [16, 64])
def test_device_and_host_repivots_give_the_oracles_bits(lanes, oracle, stages):
    """Long inverter chains change pivot order many times on their way from
    a cold start: the lanes' own factors on the device and the host's
    re-pivot tapes must both reproduce the oracle (its replay, then a full
    factor whenever a peel test fails) bit for bit."""
    fam = circuits.inverter_chain(stages)
    vals = fam.sample(77, 96)
    eng = lanes.Engine(fam.deck.arrays())
    _, _, q = eng.pattern()
    t = lanes.default_options().tol
    t.max_iter = 400
    dev = eng.solve_op(vals, tiling=lanes.TILING_WAVE, tol=t)
    dev_rep = eng.timing().repivots
    host = eng.solve_op(vals, tiling=lanes.TILING_WAVE, tol=t, host_repivot=True)
    host_rep = eng.timing().repivots
    ref = oracle.Circuit(fam.deck.arrays()).op(vals, q, threads=8,
                                                tol=oracle.Tol(t.reltol, t.abstol, t.vntol, t.residual_tol, 400, 0))
    say(f"  {stages} stages: host re-pivots {host_rep}, device run's host re-pivots {dev_rep}, "
        f"oracle re-pivots {int(ref['repivots'].sum())}, converged {(ref['reasons'] == 0).sum()}/96")
    assert ref["repivots"].sum() > 0 and host_rep > 0 and dev_rep == 0
    for got in (dev, host):
        assert np.array_equal(got["reasons"], ref["reasons"])
        assert np.array_equal(got["iterations"], ref["iterations"])
        assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    eng.close()


@pytest.mark.parametrize("tiling", [1, 2])
def test_warm_start_bitwise_against_oracle(lanes, oracle, tiling):
    fam = circuits.ota_array()
    vals = fam.sample(5, 128)
    eng = lanes.Engine(fam.deck.arrays())
    _, _, q = eng.pattern()
    c = oracle.Circuit(fam.deck.arrays())
    nom = c.op(fam.nominal()[None, :], q)
    x0 = np.repeat(nom["x"], 128, 0)
    say("warm start from the nominal operating point, 128 lanes")
    got = eng.solve_op(vals, x0=x0, tiling=tiling)
    ref = c.op(vals, q, start_x=x0, threads=8)
    assert np.array_equal(got["reasons"], ref["reasons"])
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    assert got["iterations"].mean() < 6
    eng.close()


def test_replicas_are_identical(lanes):
    # tools/gpu_lane_parity.py:1-19: replicas of one point agree bitwise.
    fam = circuits.ota_array()
    vals = np.repeat(fam.sample(9, 1), 200, 0)
    eng = lanes.Engine(fam.deck.arrays())
    got = eng.solve_op(vals)
    assert (got["x"] == got["x"][0]).all()
    assert (got["iterations"] == got["iterations"][0]).all()
    eng.close()


@pytest.mark.parametrize("tiling", [0, 1, 2])
def test_full_size_ota_converges_and_satisfies_kcl(lanes, oracle, tiling):
    """16,384 lanes of the OTA array: every lane converges, the published
    points satisfy the residual gate when re-assembled by the oracle, and a
    sample of lanes is bitwise the oracle."""
    fam = circuits.ota_array()
    n_lanes = 16384
    vals = fam.sample(4, n_lanes)
    say(f"ota_array full size {n_lanes} tiling={tiling}")
    eng = lanes.Engine(fam.deck.arrays())
    _, _, q = eng.pattern()
    got = eng.solve_op(vals, tiling=tiling)
    assert (got["reasons"] == 0).all()
    c = oracle.Circuit(fam.deck.arrays())
    pick = np.arange(0, n_lanes, 1021)
    ref = c.op(vals[pick], q, threads=8)
    # both runs take their lead tape from point 0, so every lane is bitwise
    assert np.array_equal(got["iterations"][pick], ref["iterations"])
    assert np.array_equal(bits(got["x"][pick]), bits(ref["x"]))
    for l in pick[:8]:
        g, f = c.assemble_at(vals[l], got["x"][l])
        assert np.abs(f).max() < 1e-5
    eng.close()


# ---- FP32 factors with FP64 refinement ----

@pytest.mark.parametrize("family,lanes_n", [("inverter_chain", 256), ("ota_array", 256), ("diffpair_array", 256)])
def test_fp32_refined_bitwise_against_oracle(lanes, oracle, family, lanes_n):
    """The FP32 mode is bitwise the oracle's FP32 mode: FP32 replay, FP32
    solves, FP64 residual and refinement, re-pivots and FP64 fallbacks."""
    fam = circuits.FAMILIES[family]()
    vals = fam.sample(2027, lanes_n)
    say(f"fp32 refined {family} lanes={lanes_n}")
    eng = lanes.Engine(fam.deck.arrays())
    _, _, q = eng.pattern()
    got = eng.solve_op(vals, precision=lanes.FP32_REFINED)
    ref = oracle.Circuit(fam.deck.arrays()).op(vals, q, threads=8, precision=1)
    assert np.array_equal(got["reasons"], ref["reasons"])
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    assert eng.timing().fp64_lanes == int(ref["fp64_lanes"].sum())
    say(f"  converged {(got['reasons'] == 0).sum()}/{lanes_n} fp64 fallbacks {eng.timing().fp64_lanes} "
        f"repivots {eng.timing().repivots}")
    eng.close()


def test_fp32_refinement_never_succeeding_is_the_fp64_newton(lanes):
    """refine_tol 0 with one step: every lane stalls in its first solve,
    redoes that iteration in FP64 and finishes in FP64, so the results are
    bitwise the FP64 lanes'."""
    fam = circuits.ota_array()
    vals = fam.sample(8, 256)
    eng = lanes.Engine(fam.deck.arrays())
    a = eng.solve_op(vals, tiling=lanes.TILING_WAVE)
    b = eng.solve_op(vals, precision=lanes.FP32_REFINED, refine_tol=0.0, refine_max=1)
    assert eng.timing().fp64_lanes == 256
    assert np.array_equal(a["iterations"], b["iterations"])
    assert np.array_equal(bits(a["x"]), bits(b["x"]))
    eng.close()


def test_fp32_full_size_ota_error_against_fp64(lanes, oracle):
    """16,384 OTA lanes from a cold start on the benchmark's seed: FP32
    factors + FP64 refinement against plain FP64, per node value |x32 - x64|
    <= 1e-7 max(|x64|, 1e-6) (relative, floored at vntol). Scope of the
    contract at the default refinement target (relative residual 1e-12):
    every lane whose FP64 Newton takes fewer than 30 iterations; the few
    longer runs (their limiting paths split over 30+ iterations) stay within
    the Newton tolerance's 1e-6. With the target at 1e-15 every lane meets
    1e-7. A sample is bitwise the oracle's FP32 mode."""
    fam = circuits.ota_array()
    n_lanes = 16384
    vals = fam.sample(2026, n_lanes)
    say(f"fp32 refined ota_array full size {n_lanes}")
    eng = lanes.Engine(fam.deck.arrays())
    _, _, q = eng.pattern()
    a = eng.solve_op(vals, tiling=lanes.TILING_WAVE)
    b = eng.solve_op(vals, precision=lanes.FP32_REFINED)
    conv = a["reasons"] == 0
    assert conv.mean() > 0.999 and np.array_equal(b["reasons"], a["reasons"])
    err = (np.abs(a["x"] - b["x"]) / np.maximum(np.abs(a["x"]), 1e-6)).max(1)[conv]
    short = a["iterations"][conv] < 30
    say(f"  max relative error {err.max():.3e} ({err[short].max():.3e} on the {short.sum()} lanes under 30 "
        f"iterations), fp64 fallbacks {eng.timing().fp64_lanes}")
    assert err[short].max() <= 1e-7
    assert err.max() <= 1e-6
    c = eng.solve_op(vals, precision=lanes.FP32_REFINED, refine_tol=1e-15, refine_max=16)
    err15 = (np.abs(a["x"] - c["x"]) / np.maximum(np.abs(a["x"]), 1e-6)).max(1)[conv]
    say(f"  refinement to 1e-15: max relative error {err15.max():.3e}")
    assert err15.max() <= 1e-7
    pick = np.arange(0, n_lanes, 2039)
    ref = oracle.Circuit(fam.deck.arrays()).op(vals[pick], q, threads=8, precision=1)
    assert np.array_equal(b["iterations"][pick], ref["iterations"])
    assert np.array_equal(bits(b["x"][pick]), bits(ref["x"]))
    eng.close()


def test_probes_return_the_selected_unknowns(lanes):
    fam = circuits.ota_array()
    vals = fam.sample(12, 300)
    eng = lanes.Engine(fam.deck.arrays())
    probes = np.array([fam.deck.node_index(f"out{k}") for k in range(64)] + [0, eng.n - 1], np.uint32)
    full = eng.solve_op(vals)
    got = eng.solve_op(vals, probes=probes)
    assert got["x"].shape == (300, len(probes))
    assert np.array_equal(bits(got["x"]), bits(full["x"][:, probes]))
    assert np.array_equal(got["iterations"], full["iterations"])
    eng.close()


def test_diffpair_array_fp64_and_fp32_bitwise_and_within_contract(lanes, oracle):
    """The Gummel-Poon workload: 2048 points of 64 differential pairs, FP64
    lanes bitwise the oracle, FP32 factors + FP64 refinement bitwise the
    oracle's FP32 mode and within 1e-7 relative of FP64 (floored at 1 uV /
    1 nA)."""
    fam = circuits.diffpair_array()
    vals = fam.sample(2032, 2048)
    say("diffpair_array 2048 points")
    eng = lanes.Engine(fam.deck.arrays())
    _, _, q = eng.pattern()
    a = eng.solve_op(vals)
    b = eng.solve_op(vals, precision=lanes.FP32_REFINED)
    assert (a["reasons"] == 0).all() and (b["reasons"] == 0).all()
    err = np.abs(a["x"] - b["x"]) / np.maximum(np.abs(a["x"]), 1e-6)
    say(f"  FP32 refined vs FP64 max relative {err.max():.3e}, fallbacks {eng.timing().fp64_lanes}")
    assert err.max() <= 1e-7
    c = oracle.Circuit(fam.deck.arrays())
    pick = np.arange(0, 2048, 97)
    r64 = c.op(vals[pick], q, threads=8)
    r32 = c.op(vals[pick], q, threads=8, precision=1)
    assert np.array_equal(bits(a["x"][pick]), bits(r64["x"]))
    assert np.array_equal(bits(b["x"][pick]), bits(r32["x"]))
    eng.close()


@pytest.mark.parametrize("stages,host_repivot", [(64, False), (128, False), (128, True)])
def test_ladder_matches_oracle_bitwise(lanes, oracle, stages, host_repivot):
    """Long inverter chains that plain Newton leaves unconverged climb the
    .op ladder (the gmin rung, then source stepping and a final run): every
    run and the rung control on the device; the oracle's op_ladder must
    give the same bits, iterations (summed over the runs) and reasons. Some
    points of each case go past the gmin rung (the oracle without its source
    rung ends them differently), so both rungs are compared."""
    fam = circuits.inverter_chain(stages)
    eng = lanes.Engine(fam.deck.arrays())
    _, _, q = eng.pattern()
    vals = fam.sample(5, 32)
    plain = eng.solve_op(vals, tiling=lanes.TILING_WAVE, host_repivot=host_repivot)
    got = eng.solve_op(vals, tiling=lanes.TILING_WAVE, host_repivot=host_repivot, ladder=True)
    c = oracle.Circuit(fam.deck.arrays())
    ref = c.op(vals, q, threads=8, tol=oracle.Tol(1e-3, 1e-12, 1e-6, 1e-9, 100, 1))
    gmin_only = c.op(vals, q, threads=8, tol=oracle.Tol(1e-3, 1e-12, 1e-6, 1e-9, 100, 1 | 8))
    past_gmin = ref["iterations"] != gmin_only["iterations"]
    tm = eng.timing()
    say(f"  chain {stages}: plain {int((plain['reasons'] == 0).sum())}/32, ladder {int((got['reasons'] == 0).sum())}/32, "
        f"past the gmin rung {int(past_gmin.sum())}, launches {tm.launches}")
    assert past_gmin.any()
    same_x = [bool(np.array_equal(bits(a), bits(b))) for a, b in zip(got["x"], ref["x"])]
    for l in np.nonzero((got["iterations"] != ref["iterations"]) | ~np.array(same_x))[0]:
        say(f"  lane {l}: reasons {got['reasons'][l]}/{ref['reasons'][l]} iterations {got['iterations'][l]}/"
            f"{ref['iterations'][l]} plain {plain['iterations'][l]} same x {same_x[l]}")
    assert (got["reasons"] == 0).sum() > (plain["reasons"] == 0).sum()
    assert np.array_equal(got["reasons"], ref["reasons"])
    assert all(same_x)
    assert np.array_equal(got["iterations"], ref["iterations"])
    eng.close()


def elimination_order(cp, ri, n, shallow):
    """Minimum degree on the pattern of A + A^T as a scan of every vertex at
    every step (ties to the lowest index); shallow: least 2 * degree +
    level. Returns the order, its longest path and its fill."""
    adj = [set() for _ in range(n)]
    for j in range(n):
        for i in ri[cp[j]:cp[j + 1]]:
            if i != j:
                adj[i].add(j)
                adj[j].add(int(i))
    level, gone, q, fill = [0] * n, [False] * n, [], 0
    for _ in range(n):
        v = min((v for v in range(n) if not gone[v]),
                key=lambda v: (2 * len(adj[v]) + level[v] if shallow else len(adj[v]), v))
        q.append(v)
        gone[v] = True
        nb, adj[v] = adj[v], set()
        fill += len(nb)
        for u in nb:
            level[u] = max(level[u], level[v] + 1)
            adj[u] = (adj[u] | nb) - {u, v}
    return q, max(level), fill


@pytest.mark.parametrize("fam,shallow", [
    (circuits.rc_ladder(2), False), (circuits.diode_stack(3), True), (circuits.diode_stack(24), True),
    (circuits.rc_ladder(97), True), (circuits.rc_mesh(9), False), (circuits.rc_mesh(14), False),
    (circuits.inverter_chain(7), False), (circuits.ota_array(3), False), (circuits.diffpair_array(5), False),
    (circuits.rc_ladder(780), True), (circuits.rc_ladder(900), False)], ids=lambda f: getattr(f, "name", f))
def test_column_order_is_the_stated_one(lanes, fam, shallow):
    """The engine's column order against a plain statement of it: minimum
    degree, or for decks without transistors the shallow order where it at
    least halves the longest path and leaves a lane half of a workgroup's
    LDS (10,240 doubles for n + 2 fill + 8 n)."""
    eng = lanes.Engine(fam.deck.arrays())
    cp, ri, q = eng.pattern()
    want, depth, _ = elimination_order(cp, ri, eng.n, False)
    if not any(k in (5, 6) for k in fam.deck.kind) and 8 * depth >= eng.n:
        q1, d1, f1 = elimination_order(cp, ri, eng.n, True)
        took = 2 * d1 <= depth and 9 * eng.n + 2 * f1 <= 10240
        assert took == shallow
        want = q1 if took else want
    else:
        assert not shallow
    assert list(q) == want
    eng.close()


def chain_with_floats(stages, floats):
    """An inverter chain and `floats` nodes that only capacitors touch: void
    unknowns of its operating point."""
    fam = circuits.inverter_chain(stages)
    for k in range(floats):
        fam.deck.capacitor(f"cf{k}", f"f{k}", 0, 1e-14)
    return fam


@pytest.mark.parametrize("stages,floats", [(2, 0), (58, 0), (59, 0), (60, 0), (20, 3), (56, 3)])
def test_own_lu_of_small_lanes_bitwise(lanes, oracle, stages, floats):
    """Lanes that re-pivot hold their own factors dense in LDS up to 64
    unknowns where it has room (a few lanes), and sparse beyond (65
    unknowns), with void unknowns, and where many lanes leave no room: the
    same bits on every path, the oracle's."""
    fam = chain_with_floats(stages, floats)
    eng = lanes.Engine(fam.deck.arrays())
    assert eng.n == stages + 5 + floats
    vals = fam.sample(78, 4500)
    _, _, q = eng.pattern()
    t = lanes.default_options().tol
    t.max_iter = 150
    few = eng.solve_op(vals[:48], tiling=lanes.TILING_WAVE, tol=t)
    own = eng.timing().device_repivot_lanes
    ref = oracle.Circuit(fam.deck.arrays()).op(vals[:48], q, threads=8,
                                               tol=oracle.Tol(t.reltol, t.abstol, t.vntol, t.residual_tol, 150, 0))
    say(f"  n {eng.n}: {own} of 48 lanes on their own LU, converged {(ref['reasons'] == 0).sum()}/48")
    assert stages < 16 or own > 0
    many = eng.solve_op(vals, tiling=lanes.TILING_WAVE, tol=t)
    assert stages < 16 or eng.timing().device_repivot_lanes > 2048   # eight and more a CU
    for got in (few, many):
        assert np.array_equal(got["reasons"][:48], ref["reasons"])
        assert np.array_equal(got["iterations"][:48], ref["iterations"])
        assert np.array_equal(bits(got["x"][:48]), bits(ref["x"]))
    eng.close()


@pytest.mark.parametrize("stages,count,tuned", [(43, 1024, True), (43, 1023, False), (44, 1024, False)])
def test_the_tilings_are_tried_up_to_48_unknowns(lanes, stages, count, tuned):
    """48 and 49 unknowns: a first batch of 1,024 points times both tilings
    up to 48 unknowns and runs one wavefront a lane beyond; the results are
    the wavefront tiling's either way."""
    fam = circuits.inverter_chain(stages)
    eng = lanes.Engine(fam.deck.arrays())
    assert eng.n == stages + 5
    vals = fam.sample(79, count)
    got = eng.solve_op(vals)
    assert (eng.info().tiling != 0) == tuned
    ref = eng.solve_op(vals, tiling=lanes.TILING_WAVE)
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    eng.close()


@pytest.mark.parametrize("stages", [12, 24, 40])
def test_fp32_lanes_that_stall_on_a_later_tape_go_on_in_fp64(lanes, stages):
    """Lanes whose refinement stalls go on in FP64 on the tape they stand on.
    Here the engine's first tape has fewer factor slots than this solve's
    lead: the launch must have room for the lead's, and the results are the
    FP64 lanes' bit for bit."""
    fam = circuits.inverter_chain(stages)
    vals = fam.sample(3, 4)
    eng = lanes.Engine(fam.deck.arrays())
    eng.solve_op(vals)
    first = eng.info().lds_bytes
    x0 = np.random.default_rng(5).uniform(-0.2, 1.2, (4, eng.n))
    x0[:, 0] = 0
    t = lanes.default_options().tol
    t.max_iter = 400
    got = eng.solve_op(vals, x0=x0, precision=lanes.FP32_REFINED, refine_tol=0.0, refine_max=1, tol=t)
    assert eng.timing().fp64_lanes == 4 and eng.info().lds_bytes > first
    ref = eng.solve_op(vals, x0=x0, tiling=lanes.TILING_WAVE, tol=t)
    assert (ref["reasons"] == 0).all()
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    eng.close()

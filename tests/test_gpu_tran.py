"""Diode operating points and transient lanes on the GPU against the oracle.

Bitwise: the device runs the oracle's operations in the oracle's order
(device physics, companion, LU on shared tapes), so node voltages, probe
rows, iteration counts and reasons agree bit for bit; the hipGraph replay
and plain launches, and any number of steps per launch, give the same bits.
"""
import sys

import numpy as np
import pytest

from espice_amd import circuits
from test_oracle_tran import rc_deck, trapezoid_reference

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


@pytest.mark.parametrize("precision", [0, 1])
def test_diode_stack_operating_points_bitwise(lanes, oracle, precision):
    fam = circuits.diode_stack(8)
    vals = fam.sample(21, 256)
    say(f"diode stack .op precision={precision}")
    eng = lanes.Engine(fam.deck.arrays())
    _, _, q = eng.pattern()
    got = eng.solve_op(vals, precision=precision, tiling=lanes.TILING_AUTO if precision == 0 else lanes.TILING_WAVE)
    ref = oracle.Circuit(fam.deck.arrays()).op(vals, q, threads=8, precision=precision)
    assert (got["reasons"] == 0).all()
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    eng.close()


def test_rc_ladder_transient_matches_the_recurrence(lanes):
    R, C, dt, steps, stages = 1e3, 1e-12, 1e-10, 40, 6
    d = rc_deck(R, C, stages)
    eng = lanes.Engine(d.arrays())
    probes = [d.node_index(f"n{k}") for k in range(stages)]
    r = eng.solve_tran(np.zeros((4, 0)), dt, steps, probes=probes, steps_per_launch=7)
    assert (r["reasons"] == 0).all()
    ref = trapezoid_reference(R, C, stages, dt, steps)
    assert np.allclose(r["probes"][0], ref, rtol=1e-9, atol=1e-12)
    assert (r["iterations"] == 2 * steps).all()
    eng.close()


@pytest.mark.parametrize("k,lanes_n,steps", [(6, 64, 40), (12, 128, 30)])
def test_rc_mesh_transient_bitwise_against_oracle(lanes, oracle, k, lanes_n, steps):
    fam = circuits.rc_mesh(k, diode_frac=0.1)
    vals = fam.sample(2031, lanes_n)
    d = fam.deck
    probes = [d.node_index("n0_0"), d.node_index(f"n{k - 1}_{k - 1}"), d.node_index(f"n{k // 2}_{k // 2}")]
    say(f"rc mesh {k}x{k}, {lanes_n} lanes, {steps} steps")
    eng = lanes.Engine(d.arrays())
    _, _, q = eng.pattern()
    got = eng.solve_tran(vals, 1e-12, steps, probes=probes, steps_per_launch=10)
    tm = eng.timing()
    ref = oracle.tran(oracle.Circuit(d.arrays()), vals, q, 1e-12, steps, probes=probes, threads=8)
    say(f"  reasons ok {(got['reasons'] == 0).sum()}, iterations/lane {got['iterations'].mean():.1f}, "
        f"repivots {tm.repivots}, launches {tm.launches}")
    assert np.array_equal(got["reasons"], ref["reasons"])
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["probes"]), bits(ref["probes"]))
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    eng.close()


def test_graph_and_launch_blocking_do_not_change_bits(lanes):
    fam = circuits.rc_mesh(8, diode_frac=0.1)
    vals = fam.sample(77, 64)
    probes = [fam.deck.node_index("n7_7")]
    eng = lanes.Engine(fam.deck.arrays())
    a = eng.solve_tran(vals, 1e-12, 25, probes=probes, steps_per_launch=10, use_graph=True)
    b = eng.solve_tran(vals, 1e-12, 25, probes=probes, steps_per_launch=10, use_graph=False)
    c = eng.solve_tran(vals, 1e-12, 25, probes=probes, steps_per_launch=1, use_graph=True)
    d = eng.solve_tran(vals, 1e-12, 25, probes=probes, steps_per_launch=25, use_graph=True)
    for r in (b, c, d):
        assert np.array_equal(bits(a["probes"]), bits(r["probes"]))
        assert np.array_equal(a["iterations"], r["iterations"])
    eng.close()


def test_switching_transient_repivots_on_the_device_bitwise(lanes, oracle):
    """Inverter chains switching under a step input change pivot order
    during the transient: lanes whose replay fails factor their own
    Jacobian on the device and must still match the oracle (replay, then a
    full factor when a peel test fails) bit for bit, probes included."""
    fam = circuits.inverter_chain_tran(16)
    eng = lanes.Engine(fam.deck.arrays())
    _, _, q = eng.pattern()
    vals = fam.sample(8, 48)
    dt, steps = 2e-12, 60
    probes = [eng.n - 1, 3]
    r = eng.solve_tran(vals, dt, steps, probes=probes, steps_per_launch=13)
    tm = eng.timing()
    ref = oracle.tran(oracle.Circuit(fam.deck.arrays()), vals, q, dt, steps, probes=probes, threads=8)
    say(f"  lanes on their own LU {tm.device_repivot_lanes}, host re-pivots {tm.repivots}")
    assert (ref["reasons"] == 0).mean() > 0.9
    assert np.array_equal(r["reasons"], ref["reasons"])
    assert np.array_equal(r["iterations"], ref["iterations"])
    ok = r["reasons"] == 0
    assert np.array_equal(bits(r["x"][ok]), bits(ref["x"][ok]))
    assert np.array_equal(bits(r["probes"][ok]), bits(ref["probes"][ok]))
    eng.close()


def test_progress_groups_and_cancellation(lanes):
    """The progress callback sees each group of steps; grouping the launches
    (one graph per group) leaves the bits unchanged; a true return cancels."""
    fam = circuits.rc_mesh(8, diode_frac=0.1)
    vals = fam.sample(77, 32)
    probes = [fam.deck.node_index("n7_7")]
    eng = lanes.Engine(fam.deck.arrays())
    ref = eng.solve_tran(vals, 1e-12, 25, probes=probes, steps_per_launch=5)
    seen = []
    got = eng.solve_tran(vals, 1e-12, 25, probes=probes, steps_per_launch=5,
                         progress=lambda done, total: seen.append((done, total)), progress_steps=10)
    assert seen == [(10, 25), (20, 25), (25, 25)]
    assert np.array_equal(bits(got["probes"]), bits(ref["probes"]))
    assert np.array_equal(got["iterations"], ref["iterations"])
    with pytest.raises(lanes.EslError) as ex:
        eng.solve_tran(vals, 1e-12, 25, probes=probes, steps_per_launch=5,
                       progress=lambda done, total: done >= 10, progress_steps=10)
    assert "cancelled" in str(ex.value)
    again = eng.solve_tran(vals, 1e-12, 25, probes=probes, steps_per_launch=5)
    assert np.array_equal(bits(again["probes"]), bits(ref["probes"]))
    eng.close()


def adaptive_cases():
    """(family, points, t_stop, t_step, dt_max, probes of the deck)"""
    mesh = circuits.rc_mesh(8, diode_frac=0.15)
    chain = circuits.inverter_chain_tran(12)
    ladder = circuits.rc_ladder(40, tran=True, clamp_every=8)
    pairs = circuits.diffpair_array_tran(4)
    return [
        ("rc_mesh_8", mesh, 48, 200e-12, 2e-12, 50e-12, ["n0_0", "n7_7", "n4_4"]),
        ("inverter_chain_tran_12", chain, 40, 300e-12, 5e-12, 75e-12, None),
        ("rc_ladder_tran_40", ladder, 40, 2e-9, 20e-12, 0.5e-9, None),
        ("diffpair_array_tran_4", pairs, 24, 1e-9, 20e-12, 0.25e-9, None),
    ]


@pytest.mark.parametrize("case", [c[0] for c in adaptive_cases()])
def test_adaptive_transient_bitwise_against_oracle(lanes, oracle, case):
    """Per-lane step control on the device (esl_tran_adaptive_solve): every
    lane's accepted times, probe rows, final state, accepted and rejected
    steps, Newton iterations and reasons are bitwise the oracle's
    (orc_tran_adaptive) on the same points, with several attempts per
    launch so lanes stop and resume between launches."""
    name, fam, count, t_stop, t_step, dt_max, pnames = [c for c in adaptive_cases() if c[0] == case][0]
    d = fam.deck
    eng = lanes.Engine(d.arrays())
    _, _, q = eng.pattern()
    probes = [d.node_index(p) for p in pnames] if pnames else [eng.n - 1, 1]
    vals = fam.sample(77, count)
    say(f"adaptive {name}: {count} points, t_stop {t_stop:g}")
    got = eng.solve_tran_adaptive(vals, t_stop, t_step, probes=probes, dt_max=dt_max, max_steps=3000,
                                  attempts_per_launch=16)
    ref = oracle.tran_adaptive(oracle.Circuit(d.arrays()), vals, q, t_stop, t_step,
                               dt_max=(dt_max if dt_max > 0 else None), max_steps=3000, probes=probes, threads=8)
    say(f"  accepted {got['accepted'].mean():.1f} rejected {got['rejected'].mean():.2f} its "
        f"{got['iterations'].mean():.1f} ok {(got['reasons'] == 0).sum()}; launches {eng.timing().launches}")
    assert (ref["reasons"] == 0).mean() > 0.9
    for k in ("reasons", "accepted", "rejected", "iterations"):
        assert np.array_equal(got[k], ref[k]), k
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    for l in range(count):
        a = int(ref["accepted"][l])
        assert np.array_equal(bits(got["times"][l, :a]), bits(ref["times"][l, :a])), l
        assert np.array_equal(bits(got["probes"][l, :a]), bits(ref["probes"][l, :a])), l
    eng.close()


def test_adaptive_breakpoint_landing_bitwise_against_oracle(lanes, oracle):
    """A step source at td > 0: the lanes land on the edge, drop to order 1
    and restart with a tenth of the step, bitwise as the oracle."""
    from test_oracle_adaptive import one_rc
    d = one_rc(td=2.5e-9)
    eng = lanes.Engine(d.arrays())
    _, _, q = eng.pattern()
    probes = [d.node_index("n0")]
    got = eng.solve_tran_adaptive(np.zeros((3, 0)), 8e-9, 1e-10, probes=probes, dt_max=1e-9, attempts_per_launch=5)
    ref = oracle.tran_adaptive(oracle.Circuit(d.arrays()), np.zeros((3, 0)), q, 8e-9, 1e-10, dt_max=1e-9,
                               max_steps=1000, probes=probes)
    for k in ("reasons", "accepted", "rejected", "iterations"):
        assert np.array_equal(got[k], ref[k]), k
    a = int(ref["accepted"][0])
    assert np.array_equal(bits(got["times"][:, :a]), bits(ref["times"][:, :a]))
    assert np.array_equal(bits(got["probes"][:, :a]), bits(ref["probes"][:, :a]))
    assert np.min(np.abs(got["times"][0, :a] - 2.5e-9)) <= 1e-19
    eng.close()


def test_adaptive_rows_past_the_accepted_ones_stay_the_callers(lanes):
    """A short adaptive run after a longer one on the same engine leaves the
    rows past its accepted steps as the caller had them (zeros here)."""
    fam = circuits.rc_ladder(16, tran=True)
    vals = fam.sample(5, 9)
    eng = lanes.Engine(fam.deck.arrays())
    long = eng.solve_tran_adaptive(vals, 1e-9, 1e-11, probes=[2, 3], max_steps=300)
    short = eng.solve_tran_adaptive(vals, 2e-10, 1e-11, probes=[2, 3], max_steps=300, dt_max=2e-11)
    assert (short["reasons"] == 0).all() and (short["accepted"] < long["accepted"]).all()
    for l, a in enumerate(short["accepted"]):
        assert (short["times"][l, :a] > 0).all()
        assert (short["times"][l, a:] == 0).all() and (short["probes"][l, a:] == 0).all()
    eng.close()


@pytest.mark.parametrize("nodes,shallow", [(5, None), (63, True), (64, True), (700, True), (1384, False)])
def test_lines_take_the_shallow_order_bitwise_against_oracle(lanes, oracle, nodes, shallow):
    """Lines of resistors take the shallow column order while its lane fits
    half of a workgroup's LDS; operating points and steps stay bitwise the
    oracle's in that order."""
    fam = circuits.rc_ladder(nodes, tran=True)
    vals = fam.sample(11, 5)
    eng = lanes.Engine(fam.deck.arrays())
    _, _, q = eng.pattern()
    got = eng.solve_tran(vals, 10e-12, 6, probes=[2, 3])
    if shallow is not None:   # the plain order of a line has about two levels a node
        assert (eng.info().levels < nodes) == shallow
    ref = oracle.tran(oracle.Circuit(fam.deck.arrays()), vals, q, 10e-12, 6, probes=[2, 3], threads=5)
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["probes"]), bits(ref["probes"]))
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    eng.close()


@pytest.mark.parametrize("points,probes,steps", [(3, 1, 40), (6000, 160, 40), (2, 4000, 40)])
def test_adaptive_rows_come_back_by_slabs(lanes, points, probes, steps):
    """The accepted rows come back packed in slabs of lanes (several of them
    for 6,000 lanes of 160 probes), or lane by lane where one lane's rows are
    long; either way each lane's rows are those of a solve of its own, and
    what lies past them stays the caller's."""
    fam = circuits.rc_ladder(16, tran=True)
    vals = fam.sample(21, points)
    eng = lanes.Engine(fam.deck.arrays())
    ids = [2 + k % 16 for k in range(probes)]
    got = eng.solve_tran_adaptive(vals, steps * 1e-11, 1e-11, probes=ids, max_steps=200)
    assert (got["reasons"] == 0).all()
    assert got["accepted"].min() >= 10 and got["accepted"].max() < 200
    words = int(got["accepted"].max()) * probes
    assert points < 6000 or points * words > 8 << 20   # several slabs
    assert probes < 4000 or words > 32 << 10           # long rows
    for l in {0, 1, points // 2, points - 1}:
        one = eng.solve_tran_adaptive(vals[l:l + 1], steps * 1e-11, 1e-11, probes=ids[:16], max_steps=200)
        a = int(got["accepted"][l])
        assert one["accepted"][0] == a
        assert np.array_equal(bits(got["times"][l]), bits(one["times"][0]))
        assert np.array_equal(bits(got["probes"][l][:, :16]), bits(one["probes"][0][:, :probes]))
        assert (got["times"][l, a:] == 0).all() and (got["probes"][l, a:] == 0).all()
    for k in range(16, probes, 16):   # the further probes repeat the first 16
        assert np.array_equal(got["probes"][:, :, k:k + 16], got["probes"][:, :, :16])
    eng.close()


def test_adaptive_rows_take_no_second_copy_on_the_device(lanes):
    """A run whose lanes fill max_steps holds its rows once on the device:
    the slabs they come back through are of a fixed size."""
    import ctypes

    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert lanes.load().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    fam = circuits.rc_ladder(16, tran=True)
    eng = lanes.Engine(fam.deck.arrays())
    ids = [2 + k % 16 for k in range(128)]
    steps = int(eng.solve_tran_adaptive(fam.sample(22, 1), 4e-10, 1e-11, probes=ids, max_steps=200)["accepted"][0])
    vals = np.repeat(fam.sample(22, 1), 16 * 1024, axis=0)   # 16 MB a step
    free0 = free()
    got = eng.solve_tran_adaptive(vals, 4e-10, 1e-11, probes=ids, max_steps=steps)
    used = free0 - free()
    rows = vals.shape[0] * steps * len(ids) * 8
    say(f"  {steps} steps, rows {rows / 2**20:.0f} MB, device memory taken {used / 2**20:.0f} MB")
    assert (got["accepted"] == steps).all()
    assert used < 1.5 * rows
    eng.close()


def test_a_lane_that_just_fills_a_workgroups_lds_runs(lanes, oracle):
    """A transient lane's working set is its factor slots, the larger of two
    n-vectors and the staging cells, three n-vectors and the charge cells,
    and nothing beside: the lane that takes the last double of a workgroup's
    LDS runs, bitwise the oracle's, and one double more is refused."""
    import ctypes

    static = ctypes.c_uint32()
    assert lanes.load().esl_kernel_static_lds(ctypes.byref(static)) == 0
    limit = (160 * 1024 - (static.value + 255) // 256 * 256) // 8

    def line(nodes, caps):
        """A line of resistors with `caps` of its nodes capacitive to ground."""
        d = circuits.Deck(f"line_{nodes}_{caps}")
        d.vsource("vs", "src", 0, 0.0, step_to=1.0, step_at=0.0)
        prev = "src"
        for k in range(nodes):
            d.resistor(f"r{k}", prev, f"n{k}", 1e3)
            d.bind(f"r{k}", 0, f"r{k}")
            if k < caps:
                d.capacitor(f"c{k}", f"n{k}", 0, 30e-15)
            prev = f"n{k}"
        return d

    def doubles(eng, caps):
        eng.solve_op(np.full((1, eng.n_live), 1e3))
        n = eng.n
        n_tv = eng.info().lds_bytes // 8 - max(3 * n, 1024) - 2 * n - 2
        return n_tv + max(2 * n, 1024) + 3 * n + caps   # (a charge cell for each capacitor to ground)

    # the longest line that fits, and as many capacitors as then fit
    nodes = 2540
    while True:
        eng = lanes.Engine(line(nodes, 0).arrays())
        caps = limit - doubles(eng, 0)
        eng.close()
        if caps > 0:
            break
        nodes -= 1
    say(f"  limit {limit} doubles, line of {nodes} with {caps} capacitors")
    assert caps < nodes
    for extra in (0, 1):
        d = line(nodes, caps + extra)
        eng = lanes.Engine(d.arrays())
        assert doubles(eng, caps + extra) == limit + extra
        vals = 1e3 * (1 + 0.05 * np.random.default_rng(3).standard_normal((2, eng.n_live)))
        if extra:
            with pytest.raises(lanes.EslError):
                eng.solve_tran(vals, 1e-12, 3, probes=[2, 3])
        else:
            _, _, q = eng.pattern()
            got = eng.solve_tran(vals, 1e-12, 3, probes=[2, 3])
            ref = oracle.tran(oracle.Circuit(d.arrays()), vals, q, 1e-12, 3, probes=[2, 3], threads=2)
            assert np.array_equal(got["iterations"], ref["iterations"])
            assert np.array_equal(bits(got["x"]), bits(ref["x"]))
        eng.close()


@pytest.mark.parametrize("kind,count", [("r", 16), ("r", 17), ("r", 63), ("r", 64), ("r", 65), ("r", 200), ("c", 64),
                                        ("d", 40), ("d", 64), ("m", 33), ("m", 64), ("q", 17), ("q", 64)])
def test_rails_of_many_devices_step_bitwise(lanes, oracle, kind, count):
    """A rail that every device of a kind hangs from: its Jacobian entry,
    residual row and charge collect up to 64 cells a chunk, as chains where
    they are long (slots and residuals of more than 16 cells) and as rows of
    three cells a word otherwise. The sums keep the device order: operating
    points and steps are bitwise the oracle's."""
    d = circuits.Deck(f"rail_{kind}_{count}")
    d.vsource("vs", "src", 0, 0.6, step_to=0.7, step_at=0.0)
    d.resistor("rs", "src", "rail", 10.0)
    for k in range(count):
        a = f"a{k % 7}"   # a few nodes share many devices too
        if kind == "r":
            d.resistor(f"x{k}", "rail", a, 1e3 * (1 + 0.01 * k))
        elif kind == "c":
            d.capacitor(f"x{k}", "rail", a, 1e-14 * (1 + 0.01 * k))
        elif kind == "d":
            d.diode(f"x{k}", "rail", a, {"is": 1e-15 * (1 + 0.01 * k), "cjo": 1e-14})
        elif kind == "m":
            d.mos1(f"x{k}", "rail", "rail", a, 0, {"type": 1, "vto": 0.2 + 0.001 * k, "kp": 2e-4, "cgso": 1e-10}, w=1e-6, l=1e-7)
        else:
            d.bjt(f"x{k}", "rail", "rail", a, 0, {"type": 1, "is": 1e-16 * (1 + 0.01 * k), "bf": 100.0})
    for k in range(7):
        d.resistor(f"g{k}", f"a{k}", 0, 500.0)
        d.bind(f"g{k}", 0, f"g{k}")
        d.capacitor(f"h{k}", f"a{k}", 0, 1e-14)
    d.capacitor("cr", "rail", 0, 1e-14)
    vals = 500.0 * (1 + 0.1 * np.random.default_rng(4).standard_normal((9, 7)))
    eng = lanes.Engine(d.arrays())
    _, _, q = eng.pattern()
    c = oracle.Circuit(d.arrays())
    op = eng.solve_op(vals)
    ref = c.op(vals, q, threads=8)
    assert (op["reasons"] == 0).all()
    assert np.array_equal(op["iterations"], ref["iterations"]) and np.array_equal(bits(op["x"]), bits(ref["x"]))
    got = eng.solve_tran(vals, 1e-12, 5, probes=[2, 3])
    ref = oracle.tran(c, vals, q, 1e-12, 5, probes=[2, 3], threads=8)
    assert np.array_equal(got["reasons"], ref["reasons"]) and np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["probes"]), bits(ref["probes"]))
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    eng.close()

"""Lanes beyond a workgroup's LDS: the 64 x 64 RC mesh with diode clamps
(4,099 unknowns; its factors hold about 140,000 slots per lane) and others,
one workgroup per lane (eight wavefronts, or one where the elimination is
narrow) with the factors in HBM. The arithmetic is the
wavefront kernels' (same stamps, same column replay, same gates), so the
lanes must equal the oracle bit for bit, operating points and transient
probes alike.
"""
import sys

import numpy as np
import pytest

from espice_amd import circuits

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


@pytest.fixture(scope="module")
def mesh(lanes):
    fam = circuits.rc_mesh(64)
    eng = lanes.Engine(fam.deck.arrays())
    yield fam, eng
    eng.close()


def test_mesh_operating_points_bitwise(lanes, oracle, mesh):
    fam, eng = mesh
    vals = fam.sample(41, 8)
    _, _, q = eng.pattern()
    say(f"rc mesh 64x64 .op, n {eng.n}, 8 lanes")
    got = eng.solve_op(vals)
    tm = eng.timing()
    assert tm.tiling == lanes.TILING_WAVE   # (no LDS kernel fits the mesh)
    ref = oracle.Circuit(fam.deck.arrays()).op(vals, q, threads=8)
    say(f"  iterations {got['iterations']}, kernel {tm.kernel_ms:.1f} ms")
    assert (got["reasons"] == 0).all()
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))


@pytest.mark.parametrize("graph", [True, False])
def test_mesh_transient_bitwise(lanes, oracle, mesh, graph):
    fam, eng = mesh
    d = fam.deck
    vals = fam.sample(2031, 6)
    _, _, q = eng.pattern()
    probes = [d.node_index("n0_0"), d.node_index("n63_63"), d.node_index("n32_32")]
    steps = 16
    say(f"rc mesh 64x64 transient, 6 lanes, {steps} steps, graph {graph}")
    got = eng.solve_tran(vals, 1e-12, steps, probes=probes, steps_per_launch=5, use_graph=graph)
    tm = eng.timing()
    ref = oracle.tran(oracle.Circuit(d.arrays()), vals, q, 1e-12, steps, probes=probes, threads=8)
    say(f"  iterations/lane {got['iterations'].mean():.1f}, repivots {tm.repivots}, kernel {tm.kernel_ms:.1f} ms")
    assert (ref["reasons"] == 0).all()
    assert np.array_equal(got["reasons"], ref["reasons"])
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["probes"]), bits(ref["probes"]))
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))


def test_mesh_rejects_fp32_and_batches(lanes, mesh):
    fam, eng = mesh
    vals = fam.sample(3, 2)
    with pytest.raises(lanes.EslError):
        eng.solve_op(vals, precision=lanes.FP32_REFINED)
    with pytest.raises(lanes.EslError):
        lanes.solve_batch([{"engine": eng, "values": vals}])


def test_void_unknowns_of_a_big_lane_bitwise(lanes, oracle):
    """Nodes that only capacitors touch are void in the operating point:
    their columns and rows hold zeros and their pivots are set to 1 after
    the replay has found those zeros. 200 of them, so that the slots are
    read by other wavefronts than set them: every lane keeps its first
    pivots, bitwise the oracle's, and steps on from there."""
    fam = circuits.rc_mesh(40)
    d = fam.deck
    for k in range(200):
        d.capacitor(f"cv{k}", f"v{k}", f"v{k + 1}" if k % 3 else 0, 1e-14)
    vals = fam.sample(17, 5)
    eng = lanes.Engine(d.arrays())
    _, _, q = eng.pattern()
    say(f"mesh 40x40 and 200 void unknowns, n {eng.n}, 5 lanes")
    got = eng.solve_op(vals)
    tm = eng.timing()
    c = oracle.Circuit(d.arrays())
    ref = c.op(vals, q, threads=5)
    assert tm.repivots == 0
    assert (got["reasons"] == 0).all()
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(bits(got["x"]), bits(ref["x"]))
    eng.close()


def strip(rows, cols):
    """`rows` x `cols` RC strip driven by a step in one corner: the longest
    path of its elimination holds few columns a node, so its width grows
    with `rows`."""
    d = circuits.Deck(f"strip_{rows}x{cols}")
    d.vsource("vs", "src", 0, 0.0, step_to=1.0, step_at=0.0)
    d.resistor("rs", "src", "n0_0", 50.0)
    draws = []
    for j in range(cols):
        for i in range(rows):
            for nm, to in ((f"rh{i}_{j}", (i, j + 1)), (f"rv{i}_{j}", (i + 1, j))):
                if to[0] < rows and to[1] < cols:
                    d.resistor(nm, f"n{i}_{j}", f"n{to[0]}_{to[1]}", 1e3)
                    d.bind(nm, 0, nm)
                    draws.append((nm, "log_uniform", 100.0, 1e4))
            d.capacitor(f"c{i}_{j}", f"n{i}_{j}", 0, 1e-14)
    return circuits.Family(d.title, d, draws)


def all_kinds(fam, node):
    """The family's deck with every kind of device on it: followers and
    diodes on some of its nodes, a current source into another."""
    d = fam.deck
    d.vsource("vdd", "vdd", 0, 1.2)
    d.isource("ib", 0, node(0), 1e-5)
    for k in range(70):   # more than a chunk of each
        a = node(3 * k + 1)
        d.bjt(f"q{k}", "vdd", a, f"qe{k}", 0, {"type": 1, "is": 1e-16, "bf": 100.0, "vaf": 100.0})
        d.resistor(f"rq{k}", f"qe{k}", 0, 1e4)
        d.mos1(f"m{k}", "vdd", a, f"ms{k}", 0, {"type": 1, "vto": 0.3, "kp": 2e-4, "lambda": 0.05}, w=1e-6, l=1e-7)
        d.resistor(f"rm{k}", f"ms{k}", 0, 1e4)
        d.diode(f"dd{k}", a, f"ms{k}", {"is": 1e-15})
    return fam


def against_oracle(lanes, oracle, fam, eng, vals, pick, dt, steps, op=None, tran=None):
    """Operating points and a transient of the picked rows of vals, solved
    in one batch, against the oracle's."""
    _, _, q = eng.pattern()
    c = oracle.Circuit(fam.deck.arrays())
    op = op or eng.solve_op(vals)
    ref = c.op(vals[pick], q, threads=8)
    assert np.array_equal(op["reasons"][pick], ref["reasons"])
    assert np.array_equal(op["iterations"][pick], ref["iterations"])
    assert np.array_equal(bits(op["x"][pick]), bits(ref["x"]))
    got = tran or eng.solve_tran(vals, dt, steps, probes=[2, 3, 5])
    ref = oracle.tran(c, vals[pick], q, dt, steps, probes=[2, 3, 5], threads=8)
    assert np.array_equal(got["reasons"][pick], ref["reasons"])
    assert np.array_equal(got["iterations"][pick], ref["iterations"])
    assert np.array_equal(bits(got["probes"][pick]), bits(ref["probes"]))
    assert np.array_equal(bits(got["x"][pick]), bits(ref["x"]))
    return op, got


BIG = {
    "ota_array": lambda: circuits.ota_array(640),                                   # MOS, wide
    "diffpair_array": lambda: circuits.diffpair_array_tran(500),                    # BJT, wide
    "line": lambda: circuits.rc_ladder(2900, tran=True),                            # narrow
    "all_on_line": lambda: all_kinds(circuits.rc_ladder(2700, tran=True), lambda k: f"n{k}"),
    "all_on_strip": lambda: all_kinds(strip(24, 110), lambda k: f"n{k % 24}_{k // 24}"),
}


@pytest.mark.parametrize("name", list(BIG))
def test_big_decks_bitwise(lanes, oracle, name):
    fam = BIG[name]()
    eng = lanes.Engine(fam.deck.arrays())
    vals = fam.sample(5, 6)
    say(f"{fam.name} {name}, n {eng.n}, 6 lanes")
    with pytest.raises(lanes.EslError):   # (beyond a workgroup's LDS)
        eng.solve_op(vals, precision=lanes.FP32_REFINED)
    op, _ = against_oracle(lanes, oracle, fam, eng, vals, np.arange(6), 10e-12, 4)
    given = eng.solve_op(vals, x0=op["x"])
    assert (given["iterations"] <= op["iterations"]).all()
    eng.close()


@pytest.mark.parametrize("fam,few,many", [(strip(8, 450), 12, 300), (circuits.mirror_tree(10, tran=True), 12, 1100)],
                         ids=["strip", "mirror_tree"])
def test_a_big_decks_lanes_change_their_team_with_the_batch(lanes, oracle, fam, few, many):
    """Elimination widths of about 141 and 880: eight wavefronts a lane for
    a few points, one for many, back and forth on one engine. The lanes'
    numbers are the same, bitwise the oracle's."""
    eng = lanes.Engine(fam.deck.arrays())
    vals = fam.sample(9, many)
    say(f"{fam.name}, n {eng.n}, {few} and {many} lanes")
    pick = np.arange(0, few)
    a, at = against_oracle(lanes, oracle, fam, eng, vals[:few], pick, 10e-12, 3)
    first = eng.info().tapes
    b, bt = against_oracle(lanes, oracle, fam, eng, vals, pick, 10e-12, 3)
    assert eng.info().tapes > first      # the other team has programs of its own
    last = np.arange(many - few, many)
    against_oracle(lanes, oracle, fam, eng, vals, last, 10e-12, 3, b, bt)
    tapes = eng.info().tapes
    c = eng.solve_op(vals[:few])
    d = eng.solve_tran(vals, 10e-12, 3, probes=[2, 3, 5])
    assert eng.info().tapes == tapes   # each team's programs are kept
    assert np.array_equal(bits(c["x"]), bits(a["x"])) and np.array_equal(bits(d["x"]), bits(bt["x"]))
    assert np.array_equal(bits(at["x"]), bits(bt["x"][:few]))
    eng.close()

"""GPU parity of context-sensitive, multi-phase derivation (Collider,
IfCollides; MultiPhaseEvaluator, GPUEvaluator.cuh:395-456): the interpreting
kernels through the C ABI against the oracle, bit-exact instance multisets
and equal collider counts, and the refusals of the paths that do not run
such programs."""
import sys

import numpy as np
import pytest

from operatorgraph_amd import abi, axioms, grammars
from tests.helpers import assert_same_multiset
from tests.test_context import lot_4x4, yard_program

pytestmark = pytest.mark.gpu

B, Q = abi.BOX, abi.QUAD
TECHNIQUES = [abi.KERNELS, abi.MEGAKERNEL]


def _note(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def E():
    from operatorgraph_amd import engine
    return engine


def run(E, program, ax, n_terms, technique=abi.MEGAKERNEL, params=None, cap=1 << 20, **cfg):
    eng = E.Engine(technique=technique, **cfg)
    try:
        eng.load(program).set_axioms(ax)
        if params is not None:
            eng.set_axiom_params(params)
        for t in range(n_terms):
            eng.bind(t, cap)
        eng.execute()
        return [eng.instances(t) for t in range(n_terms)], eng.colliders()
    finally:
        eng.close()


def check(E, program, ax, n_terms, technique=abi.MEGAKERNEL, params=None, **cfg):
    from oracle import oracle as O
    ref = O.derive(program, ax, params=params)
    got, (ncoll, phases) = run(E, program, ax, n_terms, technique, params=params, **cfg)
    for t in range(n_terms):
        assert_same_multiset(got[t], ref.instances(t), f"{program.name} terminal {t}")
    assert ncoll == ref.colliders
    return got, ref, phases


@pytest.mark.parametrize("technique", TECHNIQUES)
@pytest.mark.parametrize("variant", ["two_phases", "same_phase", "other_tag", "dropped", "three_phases",
                                     "three_phases_tag1", "three_phases_tag5", "unassigned"])
def test_yard_programs(E, technique, variant):
    _note(f"yard {variant} technique={technique}")
    kw = {"two_phases": {}, "same_phase": {"yard_phase": 0}, "other_tag": {"tag": 3},
          "dropped": {"late_generate_phase": 0}, "three_phases": {"lamps": True},
          "three_phases_tag1": {"lamps": True, "lamp_tag": 1}, "three_phases_tag5": {"lamps": True, "lamp_tag": 5},
          "unassigned": {"yard_phase": -1}}[variant]
    got, ref, phases = check(E, yard_program(**kw), lot_4x4(), 5, technique)
    assert phases == 3          # the lamp entries name phase 2 even where unreachable
    if variant == "two_phases":
        assert [len(g) for g in got] == [1, 12, 4, 0, 0]


@pytest.mark.parametrize("quad_depth", [0.0, 0.7])
def test_collision_pairs(E, quad_depth):
    """Every pairing of Box and Quad, random sizes, rotations and offsets:
    the device's decision for each pair is the oracle's."""
    _note(f"collision pairs quad_depth={quad_depth}")
    rng = np.random.default_rng(11 + int(quad_depth * 10))
    kinds = [(ta, tb) for ta in (B, Q) for tb in (B, Q)] * 256
    ax, p = axioms.collision_pair_axioms(kinds, rng, quad_depth=quad_depth)
    got, ref, phases = check(E, grammars.collision_pairs(), ax, 3, params=p)
    assert phases == 2
    assert len(got[0]) == len(kinds) and len(got[1]) + len(got[2]) == len(kinds)
    assert 0.2 * len(kinds) < len(got[1]) < 0.8 * len(kinds)


@pytest.mark.parametrize("pairs", [32, 33, 65, 9001])
def test_collision_walk_of_overlapping_colliders(E, pairs):
    """Colliders that lie on each other, on either side of the count that is
    scanned and with more of them than a walk's stack can hold the subtrees
    of; every other question asks for a tag that differs from its collider's
    in the bits above the low 16 only, and no shape meets it."""
    _note(f"collision walk pairs={pairs}")
    rng = np.random.default_rng(29)
    ax, p = axioms.collision_pair_axioms([(B, B)] * pairs, rng, spread=0.3)
    p[1::4, 9] += 65536.0
    got, ref, phases = check(E, grammars.collision_pairs(), ax, 3, params=p)
    assert phases == 2 and len(got[0]) == pairs
    assert len(got[1]) <= pairs // 2 and len(got[2]) >= (pairs + 1) // 2


def _trail(pairs, outliers):
    """Colliders in a cluster at the scene's high corner, a chain of twins
    trailing away from it along each axis at doubling distances (`outliers`),
    all of one tag. The questions are upright sheets that lie across the scene,
    clear of every collider: their boxes hold all outliers and the cluster's
    low corner."""
    rng = np.random.default_rng(5)
    ax, p = axioms.collision_pair_axioms([(B, B)] * pairs, rng)
    a, b = p[0::2], p[1::2]
    a[:, 0:6] = (0.01, 0.01, 0.01, 0.0, 0.0, 0.0)
    a[:, 6:9] = rng.uniform(0.0, 32.0, (pairs, 3))
    if outliers:
        for k in range(30):
            a[k, 6:9] = 0.0
            a[k, 6 + k // 2 % 3] = 32.0 - 768.0 / 2 ** (k // 6)
    reach, w = 1100.0, -1100.0 / 2 + 1.0
    b[:] = (0.01, reach, 2 ** 0.5 * reach, 0.0, -45.0, 0.0, 2 ** 0.5 * w, w, 0.0, 7.0)
    a[:, 9] = 7.0
    return ax, p


def test_collision_walk_of_a_trail(E):
    """A walk whose stack is full of outliers when it comes to the cluster:
    the same answers as the oracle, questions that do collide among them."""
    _note("collision walk over a trail")
    ax, p = _trail(1500, True)
    rng = np.random.default_rng(6)
    p[1::4, 0:3] = rng.uniform(0.5, 4.0, (750, 3))
    p[1::4, 3:6] = rng.uniform(0.0, 360.0, (750, 3))
    p[1::4, 6:9] = rng.uniform(-30.0, 30.0, (750, 3))
    got, ref, phases = check(E, grammars.collision_pairs(), ax, 3, params=p)
    assert phases == 2 and len(got[1]) > 0 and len(got[2]) > 750


def test_collision_walk_is_not_a_scan(E):
    """The trail costs little beside the cluster alone (305 and 265 us for
    16,384 pairs; 14.6 ms when the walk, its stack full, scanned the cluster
    leaf by leaf). The bound lies between."""
    _note("collision walk over a trail, time")
    best = {}
    for outliers in (False, True):
        ax, p = _trail(16384, outliers)
        eng = E.Engine()
        try:
            eng.load(grammars.collision_pairs()).set_axioms(ax).set_axiom_params(p)
            for t in range(3):
                eng.bind(t, 16384)
            times = []
            for _ in range(6):
                eng.execute()
                times.append(eng.kernel_seconds())
            assert [int(c) for c in eng.counts(3)] == [16384, 0, 16384]
            best[outliers] = min(times)
        finally:
            eng.close()
    assert best[True] < 5.0 * best[False], best


@pytest.mark.parametrize("technique", TECHNIQUES)
@pytest.mark.parametrize("walls", [False, True])
def test_context_city(E, technique, walls):
    _note(f"context city walls={walls} technique={technique}")
    lots = axioms.city_lots(64)
    got, ref, phases = check(E, grammars.context_city(walls=walls), lots, 4, technique)
    cells = sum(int(np.floor(a["size"][0])) * int(np.floor(a["size"][2])) for a in lots)
    assert len(got[1]) + len(got[2]) == cells and len(got[2]) > 0


@pytest.mark.parametrize("block_size", [256, 768, 1024])
def test_context_city_block_sizes(E, block_size):
    _note(f"context city block_size={block_size}")
    check(E, grammars.context_city(walls=True), axioms.city_lots(256), 4, block_size=block_size)


def test_repeated_and_appended_executes(E):
    """Colliders start empty at every execute; an appending execute adds the
    same instances again."""
    _note("context city execute twice, then append")
    from oracle import oracle as O
    lots = axioms.city_lots(32)
    prog = grammars.context_city()
    ref = O.derive(prog, lots)
    eng = E.Engine()
    try:
        eng.load(prog).set_axioms(lots)
        for t in range(4):
            eng.bind(t, 1 << 18)
        for _ in range(2):
            eng.execute()
            for t in range(3):
                assert_same_multiset(eng.instances(t), ref.instances(t), f"terminal {t}")
            assert eng.colliders() == (ref.colliders, 2)
        eng.execute(append=True)
        for t in range(3):
            assert_same_multiset(eng.instances(t), np.concatenate([ref.instances(t)] * 2), f"appended {t}")
        assert eng.colliders() == (ref.colliders, 2)
    finally:
        eng.close()


def test_collider_capacity_overflow(E):
    _note("collider capacity 4 with 13 colliders")
    eng = E.Engine()
    try:
        eng.load(yard_program()).set_axioms(lot_4x4())
        for t in range(5):
            eng.bind(t, 1024)
        eng.set_collider_capacity(4)
        with pytest.raises(E.PGAError) as e:
            eng.execute()
        assert e.value.status == abi.ERR_OVERFLOW_QUEUE
        eng.set_collider_capacity(0)
        eng.execute()
        assert [int(c) for c in eng.counts(5)] == [1, 12, 4, 0, 0]
    finally:
        eng.close()


@pytest.mark.parametrize("technique", TECHNIQUES)
@pytest.mark.parametrize("capacity", [1, 2, 32, 33, 2000])
def test_collider_capacity_lowered(E, technique, capacity):
    """A store made smaller than the one before, down to a single collider
    (for which no tree is built), with more colliders than it holds, then as
    many as it holds, and the default again."""
    from oracle import oracle as O
    _note(f"collider capacity lowered to {capacity}, technique={technique}")
    lots = axioms.city_lots(3000)
    prog = grammars.context_city()
    few = lots[:min(capacity, 48)]
    ref_few = O.derive(prog, few)
    eng = E.Engine(technique=technique)
    try:
        eng.load(prog).set_axioms(lots)
        for t in range(3):
            eng.bind(t, 1 << 18)
        eng.execute()
        counts = [int(c) for c in eng.counts(3)]
        assert eng.colliders()[0] == len(lots)
        eng.set_collider_capacity(capacity)
        with pytest.raises(E.PGAError) as e:
            eng.execute()
        assert e.value.status == abi.ERR_OVERFLOW_QUEUE
        eng.set_axioms(few)
        eng.execute()
        for t in range(3):
            assert_same_multiset(eng.instances(t), ref_few.instances(t), f"terminal {t}")
        assert eng.colliders()[0] == len(few)
        eng.set_collider_capacity(0)
        eng.set_axioms(lots)
        eng.execute()
        assert [int(c) for c in eng.counts(3)] == counts
    finally:
        eng.close()


def test_refusals(E):
    _note("context-sensitive programs: specialise, tape and capture refused; phase 16 rejected")
    eng = E.Engine()
    try:
        eng.load(grammars.context_city()).set_axioms(axioms.city_lots(4))
        for t in range(4):
            eng.bind(t, 4096)
        with pytest.raises(E.PGAError) as e:
            eng.specialize()
        assert e.value.status == abi.ERR_UNSUPPORTED
        eng.tape_reserve(1 << 16, 1 << 16)
        with pytest.raises(E.PGAError) as e:
            eng.forward_tape()
        assert e.value.status == abi.ERR_UNSUPPORTED
        with pytest.raises(E.PGAError) as e:
            with eng.capture():
                eng.execute_async()
        assert e.value.status == abi.ERR_UNSUPPORTED
        eng.execute()                       # still runs eagerly
        assert eng.colliders()[0] == 4
        bad = yard_program()
        bad.table.entries[0].successors[1].phase_index = 16
        with pytest.raises(E.PGAError) as e:
            eng.load(bad)
        assert e.value.status == abi.ERR_BAD_PROGRAM
    finally:
        eng.close()


def test_depth_limit_of_multi_phase_programs(E):
    """Depth shares the instance meta with the phase: a multi-phase program
    stops at depth 4096 with PGA_ERR_MAX_DEPTH, as the oracle does."""
    _note("multi-phase depth limit")
    from oracle import oracle as O
    from operatorgraph_amd.grammars import CONTEXT_PROCEDURES, _cop
    from operatorgraph_amd.program import DispatchTable, Entry, Program, Scalar
    # Lot = Replicate { Loop (phase 1) }; Loop = Translate(0, 0, 0) Loop
    prog = Program(CONTEXT_PROCEDURES, DispatchTable([
        Entry(_cop(abi.REPLICATE, B), [], [(1, 1)]),
        Entry(_cop(abi.TRANSLATE, B), [Scalar(0.0), Scalar(0.0), Scalar(0.0)], [(1, 1)]),
    ]), "loop")
    with pytest.raises(O.OracleError) as e:
        O.derive(prog, lot_4x4())
    assert e.value.status == abi.ERR_MAX_DEPTH
    eng = E.Engine()
    try:
        eng.load(prog).set_axioms(lot_4x4())
        eng.bind(0, 16)
        with pytest.raises(E.PGAError) as e:
            eng.execute()
        assert e.value.status == abi.ERR_MAX_DEPTH
    finally:
        eng.close()

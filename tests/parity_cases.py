"""Parity cases of the sampler against the CPU oracle, shared by backends.

Each case takes the sampler class under test (the HIP library on an MI355X,
or the host build of the same engine source) and the oracle module.  Both
consume the same random stream (Philox keyed by seed and replica, one
sub-stream per MC step; or a recorded reference-RNG tape), so every
acceptance decision, lattice configuration, FP64 energy and move counter
must agree exactly.  Energies are compared with a 1e-12 relative tolerance
written out below; in practice they agree to the last bit.
"""
import sys

import pytest

from latticednaorigami_amd import abi, systems

ENERGY_RTOL = 1e-12
EXACT_KEYS = ["num_staples", "num_domains", "num_bound_domain_pairs",
              "num_fully_bound_domain_pairs", "num_misbound_domain_pairs",
              "num_stacked_domain_pairs", "num_unassigned_domains", "step", "status",
              "last_move", "last_accepted"]


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def assert_same(gpu, ref, r):
    a, b = gpu.observables(r), ref.observables(r)
    for k in EXACT_KEYS:
        assert a[k] == b[k], (r, k, a[k], b[k])
    for k in ("energy", "enthalpy", "entropy", "stacking_energy"):
        assert a[k] == pytest.approx(b[k], rel=ENERGY_RTOL, abs=1e-12), (r, k, a[k], b[k])
    assert gpu.config(r) == ref.config(r), r


def assert_counters(gpu, ref):
    ca, cb = gpu.counters(), ref.counters()
    assert list(ca.attempts) == list(cb.attempts)
    assert list(ca.accepts) == list(cb.accepts)
    assert (ca.site_empty, ca.site_bind, ca.commits) == (cb.site_empty, cb.site_bind, cb.commits)


def case_four_domain_constant_t_bit_exact(sampler_cls, oracle_mod):
    say("case: four-domain system, 330 K, 5 x 10000 steps, lanes_per_replica=64")
    s = systems.four_domain_system()
    gpu = sampler_cls(s, temps=[330.0])
    ref = oracle_mod.Oracle(s, temps=[330.0])
    for _ in range(5):
        gpu.sweep(10000)
        ref.sweep(10000)
        assert_same(gpu, ref, 0)
    assert_counters(gpu, ref)
    # the per-move tracking behind the .moves summary
    tr = gpu.move_tracking(0)
    assert tr == ref.move_tracking(0)
    assert sum(tr["met_insert_attempts"]) + sum(tr["met_delete_attempts"]) == \
        gpu.counters().attempts[1]
    assert sum(tr["ctcb_length_attempts"]) == sum(tr["ctcb_staples_attempts"]) == \
        gpu.counters().attempts[3]


def case_lane_mappings_agree(sampler_cls, oracle_mod):
    say("case: four-domain system, 40 replicas at 310-350 K, lanes_per_replica=1 vs 64")
    s = systems.four_domain_system()
    temps = [310.0 + i for i in range(40)]
    a = sampler_cls(s, temps=temps, lanes_per_replica=1)
    b = sampler_cls(s, temps=temps, lanes_per_replica=64)
    ref = oracle_mod.Oracle(s, temps=temps)
    for x in (a, b):
        x.sweep(3000)
    ref.sweep(3000)
    for r in range(0, 40, 7):
        assert_same(a, ref, r)
        assert_same(b, ref, r)


def case_raster_nearest_neighbour_bit_exact(sampler_cls, oracle_mod):
    say("case: 64-domain raster, NN energies, 300 K and 360 K, 4 x 5000 steps")
    s = systems.raster_system(replicas=2)
    gpu = sampler_cls(s, temps=s.temps)
    ref = oracle_mod.Oracle(s, temps=s.temps)
    for _ in range(4):
        gpu.sweep(5000)
        ref.sweep(5000)
        for r in range(2):
            assert_same(gpu, ref, r)
    assert_counters(gpu, ref)
    for r in range(2):
        assert gpu.move_tracking(r) == ref.move_tracking(r)


def case_sweep_kernels_agree(sampler_cls, oracle_mod):
    say("case: 64-domain raster, 2 replicas, sweep with blocks in LDS and in device memory, "
        "3 x 2000 steps")
    import os
    s = systems.raster_system(replicas=2)
    os.environ["LDO_SWEEP_KERNEL"] = "global"
    try:
        glob = sampler_cls(s, temps=s.temps)
    finally:
        del os.environ["LDO_SWEEP_KERNEL"]
    lds = sampler_cls(s, temps=s.temps)
    ref = oracle_mod.Oracle(s, temps=s.temps)
    for _ in range(3):
        glob.sweep(2000)
        lds.sweep(2000)
        ref.sweep(2000)
        for r in range(2):
            assert_same(glob, ref, r)
            assert_same(lds, ref, r)
    assert_counters(glob, ref)
    assert_counters(lds, ref)


def case_ptmc_exchange_matches_oracle(sampler_cls, oracle_mod):
    say("case: 64-domain raster, 8-replica PTMC ladder 300-360 K, 12 swaps x 250 steps")
    s = systems.raster_system(replicas=8)
    gpu = sampler_cls(s, temps=s.temps, exchange_mode=abi.EXCHANGE_TEMPERATURE)
    ref = oracle_mod.Oracle(s, temps=s.temps)
    for _ in range(3):
        gpu.run(4, 250)
        ref.run(4, 250)
        assert gpu.permutation() == ref.permutation()
        for r in range(8):
            assert_same(gpu, ref, r)
    cg, cr = gpu.counters(), ref.counters()
    assert cg.exchange_attempts == cr.exchange_attempts
    assert cg.exchange_accepts == cr.exchange_accepts


PT_LADDER = dict(temps=[320.0, 326.0, 326.0, 332.0, 338.0, 344.0],
                 u=[1.0, 1.1, 0.9, 1.05, 1.0, 0.95],
                 b=[1.0, 0.9, 1.1, 1.0, 1.2, 1.0],
                 s=[1.0, 1.1, 0.9, 1.2, 1.0, 0.8])


def _pt_pair(sampler_cls, oracle_mod, mode, system):
    gpu = sampler_cls(system, temps=PT_LADDER["temps"], exchange_mode=mode)
    ref = oracle_mod.Oracle(system, temps=PT_LADDER["temps"], exchange_mode=mode)
    return gpu, ref


def _pt_compare(gpu, ref, n, rounds, steps):
    for _ in range(rounds):
        gpu.run(1, steps)
        ref.run(1, steps)
        assert gpu.permutation() == ref.permutation()
    for r in range(n):
        assert_same(gpu, ref, r)
    cg, cr = gpu.counters(), ref.counters()
    assert (cg.exchange_attempts, cg.exchange_accepts) == (cr.exchange_attempts,
                                                           cr.exchange_accepts)
    ag, bg = gpu.exchange_counts()
    ar, br = ref.exchange_counts()
    assert ag.tolist() == ar.tolist() and bg.tolist() == br.tolist()
    assert int(ag.sum()) == cg.exchange_attempts and int(bg.sum()) == cg.exchange_accepts
    return cg


def case_pt_variants_match_oracle(sampler_cls, oracle_mod):
    """t/ut/hut/st_parallel_tempering on one ladder whose chemical-potential,
    bias and stacking multipliers all differ from 1 (two slots share a
    temperature), then 2d_parallel_tempering on a 2 x 3 grid."""
    s = systems.four_domain_system()
    L = PT_LADDER
    for mode in (abi.EXCHANGE_T, abi.EXCHANGE_TEMPERATURE, abi.EXCHANGE_HUT, abi.EXCHANGE_ST):
        say(f"case: four-domain system, 6-slot ladder, exchange mode {mode}, "
            "12 swaps x 150 steps")
        gpu, ref = _pt_pair(sampler_cls, oracle_mod, mode, s)
        for x in (gpu, ref):
            x.set_ladder(L["temps"], L["u"], L["b"], L["s"])
        c = _pt_compare(gpu, ref, 6, 12, 150)
        assert c.exchange_attempts == 6 * 2 + 6 * 3
    say("case: four-domain system, 2D ladder 2 temperatures x 3 stacking multipliers, "
        "12 swaps x 150 steps")
    gpu, ref = _pt_pair(sampler_cls, oracle_mod, abi.EXCHANGE_2D, s)
    for x in (gpu, ref):
        x.set_ladder_2d([326.0, 334.0], [1.0, 1.15, 0.85], 1.0)
    c = _pt_compare(gpu, ref, 6, 12, 150)
    # sets 0/2 try 3 and 0 temperature pairs, sets 1/3 try 2 and 2 stacking pairs
    assert c.exchange_attempts == 3 * (3 + 0 + 2 + 2)
    with pytest.raises(abi.LdoError):
        gpu.set_ladder_2d([320.0, 330.0], [1.0, 1.15], 1.0)
    one = sampler_cls(s, temps=L["temps"], exchange_mode=abi.EXCHANGE_T)
    with pytest.raises(abi.LdoError):
        one.set_ladder_2d([320.0, 330.0], [1.0, 1.15, 0.85], 1.0)


def _raster_windows(n):
    """One numstaples window per replica: nested LinearStepWell restraints
    [0, 2 + w] (the raster holds 0-4 staples over these runs, so every pair
    of windows overlaps and swaps are tried) and a seeded grid bias of 41
    points per window, so swap acceptance is not trivially one."""
    import random
    rnd = random.Random(4242)
    wins, grid = [], []
    for w in range(n):
        wins.append(abi.Window(abi.OP_NUMSTAPLES, 0, 2 + w, 0, 0.0, 2.0, 1.5, 0.0, 1.0))
        grid += [rnd.uniform(-1.0, 1.0) for _ in range(41)]
    return wins, grid, 41


def case_windows_exchange_matches_oracle(sampler_cls, oracle_mod):
    say("case: 64-domain raster, 8 numstaples windows at 330 K, 2 x 2000 biased steps, "
        "then 12 window swaps x 250 steps")
    s = systems.raster_system(replicas=8)
    temps = [330.0] * 8
    wins, grid, glen = _raster_windows(8)
    us = sampler_cls(s, temps=temps)
    ref = oracle_mod.Oracle(s, temps=temps)
    us.set_windows(wins, grid, glen)
    ref.set_windows(wins, grid, glen)
    for _ in range(2):
        us.sweep(2000)
        ref.sweep(2000)
        for r in range(8):
            assert_same(us, ref, r)
            assert us.observables(r)["bias"] == ref.observables(r)["bias"], r
    assert_counters(us, ref)
    gpu = sampler_cls(s, temps=temps, exchange_mode=abi.EXCHANGE_WINDOWS)
    ref = oracle_mod.Oracle(s, temps=temps, exchange_mode=abi.EXCHANGE_WINDOWS)
    gpu.set_windows(wins, grid, glen)
    ref.set_windows(wins, grid, glen)
    for _ in range(3):
        gpu.run(4, 250)
        ref.run(4, 250)
        assert gpu.permutation() == ref.permutation()
        for r in range(8):
            assert_same(gpu, ref, r)
            assert gpu.observables(r)["bias"] == ref.observables(r)["bias"], r
    cg, cr = gpu.counters(), ref.counters()
    assert cg.exchange_attempts == cr.exchange_attempts
    assert cg.exchange_accepts == cr.exchange_accepts
    assert 0 < cg.exchange_accepts < cg.exchange_attempts
    assert_counters(gpu, ref)
    with pytest.raises(abi.LdoError) as e:
        gpu.set_windows(wins[:4], grid[:4 * glen], glen)
    assert e.value.code == abi.LDO_E_ARG


def case_window_histogram_and_grid_replacement(sampler_cls, oracle_mod):
    say("case: 64-domain raster, 8 numstaples windows at 330 K with a 3-point grid "
        "(visits at 3-4 staples fall off it), per-step histograms over 2 x 2000 steps "
        "with the grid replaced in between, then 8 window swaps x 250 steps")
    import numpy as np
    s = systems.raster_system(replicas=8)
    temps = [330.0] * 8
    wins, grid, _ = _raster_windows(8)
    glen = 3
    grid = [g for w in range(8) for g in grid[41 * w:41 * w + glen]]
    grid2 = [0.7 * g - 0.3 for g in grid]
    for mode in (None, abi.EXCHANGE_WINDOWS):
        kw = {} if mode is None else {"exchange_mode": mode}
        gpu = sampler_cls(s, temps=temps, **kw)
        ref = oracle_mod.Oracle(s, temps=temps, **kw)
        for x in (gpu, ref):
            x.set_windows(wins, grid, glen)
            x.set_histogram(True)
        if mode is None:
            for g in (grid, grid2):
                for x in (gpu, ref):
                    x.set_window_grid(g)
                    x.sweep(2000)
                hg, hr = gpu.histogram(reset=True), ref.histogram(reset=True)
                assert np.array_equal(hg, hr)
                assert (hg.sum(axis=1) == 2000).all()
                assert hg[:, glen].sum() > 0  # some steps ended off the grid
                for r in range(8):
                    assert_same(gpu, ref, r)
                    assert gpu.observables(r)["bias"] == ref.observables(r)["bias"], r
            assert not gpu.histogram().any()
        else:
            for x in (gpu, ref):
                x.run(8, 250)
            hg, hr = gpu.histogram(), ref.histogram()
            assert np.array_equal(hg, hr)
            assert (hg.sum(axis=1) == 2000).all()
            assert gpu.permutation() == ref.permutation()
        assert_counters(gpu, ref)
        gpu.set_histogram(False)
        with pytest.raises(abi.LdoError) as e:
            gpu.histogram()
        assert e.value.code == abi.LDO_E_ARG


def case_three_quarter_turn_and_three_domain_staples(sampler_cls, oracle_mod):
    say("case: ThreeQuarterTurn four-domain system (8 replicas, 340-354 K) and the "
        "three-domain staple system with both CTCB endpoint rules (8 replicas, 345-352 K), "
        "3 x 5000 steps")
    tq = systems.four_domain_system(seed=17)
    tq.domain_type = abi.THREEQUARTERTURN
    cases = [(tq, [340.0 + 2 * i for i in range(8)])]
    for flags in (0, abi.FLAG_CTCB_SCAFFOLD_ENDPOINTS):
        for dt in (abi.HALFTURN, abi.THREEQUARTERTURN):
            s = systems.three_domain_system(domain_type=dt, max_total_staples=2, flags=flags)
            cases.append((s, [345.0 + i for i in range(8)]))
    for s, temps in cases:
        gpu = sampler_cls(s, temps=temps)
        ref = oracle_mod.Oracle(s, temps=temps)
        for _ in range(3):
            gpu.sweep(5000)
            ref.sweep(5000)
            for r in range(len(temps)):
                assert_same(gpu, ref, r)
        assert_counters(gpu, ref)


def case_mwus3d_window_ladders_by_temperature(sampler_cls, oracle_mod):
    say("case: 200-domain ThreeQuarterTurn 5x5x8 scaffold, 3-domain staples, NN; "
        "numfulldomains windows: 3 at 318 K, 2 at 322 K, 3 at 326 K (three ladders), "
        "6 window swaps x 500 steps")
    s, wins, grid, glen = systems.mwus3d_system(windows=64, temps=(318.0,))
    pick = [0, 1, 2, 0, 1, 0, 1, 2]
    temps = [318.0] * 3 + [322.0] * 2 + [326.0] * 3
    wins = [wins[i] for i in pick]
    for i, w in enumerate(wins):  # wide wells so that the bare scaffold swaps
        wins[i] = abi.Window(w.op, 0, w.max_op + 4 * i, 0, 0.0, 0.0, 1.0, 0.0, 1.0)
    s.temps = temps
    gpu = sampler_cls(s, temps=temps, exchange_mode=abi.EXCHANGE_WINDOWS)
    ref = oracle_mod.Oracle(s, temps=temps, exchange_mode=abi.EXCHANGE_WINDOWS)
    gpu.set_windows(wins, grid, glen)
    ref.set_windows(wins, grid, glen)
    groups = [range(0, 3), range(3, 5), range(5, 8)]
    for _ in range(3):
        gpu.run(2, 500)
        ref.run(2, 500)
        perm = gpu.permutation()
        assert perm == ref.permutation()
        for g in groups:
            assert sorted(perm[q] for q in g) == list(g)  # swaps stay in their ladder
        for r in range(8):
            assert_same(gpu, ref, r)
            assert gpu.observables(r)["bias"] == ref.observables(r)["bias"], r
    cg, cr = gpu.counters(), ref.counters()
    # even rounds pair (0,1), (3,4), (5,6); odd rounds (1,2), (6,7)
    assert cg.exchange_attempts == cr.exchange_attempts == 3 * 3 + 3 * 2
    assert cg.exchange_accepts == cr.exchange_accepts > 0
    assert_counters(gpu, ref)


def case_window_temperature_swaps(sampler_cls, oracle_mod):
    """LDO_FLAG_WINDOW_TEMPERATURE_SWAPS: three ladders of the same three
    windows at 318, 320 and 322 K, each slot with its own seeded grid bias;
    every round swaps windows within the ladders, then window w between
    neighbouring ladders."""
    import random
    say("case: 200-domain 3D scaffold, 3 windows x 3 temperatures with temperature-direction "
        "swaps, 6 rounds x 500 steps")
    s, wins, grid, glen = systems.mwus3d_system(windows=64, temps=(318.0,))
    temps = [318.0] * 3 + [320.0] * 3 + [322.0] * 3
    wins = [abi.Window(wins[i].op, 0, wins[i].max_op + 4 * i, 0, 0.0, 0.0, 1.0, 0.0, 1.0)
            for i in (0, 1, 2)] * 3
    rnd = random.Random(77)
    grid = [rnd.uniform(-0.5, 0.5) for _ in range(9 * glen)]
    s.temps = temps
    s.flags = abi.FLAG_WINDOW_TEMPERATURE_SWAPS
    gpu = sampler_cls(s, temps=temps, exchange_mode=abi.EXCHANGE_WINDOWS)
    ref = oracle_mod.Oracle(s, temps=temps, exchange_mode=abi.EXCHANGE_WINDOWS)
    gpu.set_windows(wins, grid, glen)
    ref.set_windows(wins, grid, glen)
    crossed = False
    for _ in range(3):
        gpu.run(2, 500)
        ref.run(2, 500)
        perm = gpu.permutation()
        assert perm == ref.permutation()
        crossed |= any(perm[q] // 3 != q // 3 for q in range(9))
        for r in range(9):
            assert_same(gpu, ref, r)
            assert gpu.observables(r)["bias"] == ref.observables(r)["bias"], r
    assert_counters(gpu, ref)
    ag, bg = gpu.exchange_counts()
    ar, br = ref.exchange_counts()
    assert ag.tolist() == ar.tolist() and bg.tolist() == br.tolist()
    # odd rounds pair ladders 1, 2 and even rounds 0, 1, window by window
    assert ag[1].tolist() == [3, 3, 3, 3, 3, 3, 0, 0, 0]
    assert bg[1].sum() > 0 and crossed
    # the flag needs equal ladders: a different window in the last ladder
    bad = list(wins)
    bad[8] = abi.Window(wins[2].op, 0, wins[2].max_op + 1, 0, 0.0, 0.0, 1.0, 0.0, 1.0)
    for x in (gpu, ref):
        with pytest.raises(abi.LdoError):
            x.set_windows(bad, grid, glen)


LONG_LADDERS = {
    "50_50_50": [50] * 3, "70_70": [70] * 2, "131": [131], "63_2_64_65": [63, 2, 64, 65]}


def case_window_ladders_past_64_slots(sampler_cls, oracle_mod, name):
    """Window ladders that do not fit the exchange's 64 lanes: ladders that end within a
    set of 64 slots, pairs across its edge, more than 64 temperature-direction pairs,
    draws numbered on from set to set, in odd and even rounds."""
    import random
    sizes = LONG_LADDERS[name]
    say(f"case: four-domain system, window ladders of {sizes}, 6 rounds x 40 steps")
    s = systems.four_domain_system(max_total_staples=8)
    n = sum(sizes)
    temps = [330.0 + 2.0 * k for k, size in enumerate(sizes) for _ in range(size)]
    equal = len(sizes) > 1 and len(set(sizes)) == 1
    if equal:
        s.flags = abi.FLAG_WINDOW_TEMPERATURE_SWAPS
    s.temps = temps
    glen = 5
    wins = [abi.Window(abi.OP_NUMFULLDOMAINS, 0, 2 + i % 3, 0, 0.0, 0.0, 1.0, 0.0, 1.0)
            for size in sizes for i in range(size)]
    rnd = random.Random(n)
    grid = [rnd.uniform(-1.0, 1.0) for _ in range(n * glen)]
    gpu = sampler_cls(s, temps=temps, exchange_mode=abi.EXCHANGE_WINDOWS)
    ref = oracle_mod.Oracle(s, temps=temps, exchange_mode=abi.EXCHANGE_WINDOWS)
    for x in (gpu, ref):
        x.set_windows(wins, grid, glen)
    for rounds in (1, 1, 2, 1, 1):
        gpu.run(rounds, 40)
        ref.run(rounds, 40)
        assert gpu.permutation() == ref.permutation()
        ag, bg = gpu.exchange_counts()
        ar, br = ref.exchange_counts()
        assert ag.tolist() == ar.tolist() and bg.tolist() == br.tolist()
    for r in range(n):
        assert_same(gpu, ref, r)
    # swaps at every ladder, and not at every try
    at = 0
    for size in sizes:
        assert size < 3 or 0 < bg[0][at:at + size].sum() < ag[0][at:at + size].sum()
        at += size
    assert not equal or 0 < bg[1].sum() < ag[1].sum()


def case_mwus3d_full_size_exchanges(sampler_cls, oracle_mod):
    """The 3D umbrella workload at its full size: 64 windows x 4 temperatures
    (256 replicas of the 200-domain scaffold), exchanges every 500 steps,
    window swaps within each temperature and temperature-direction swaps.
    The windows are widened to start at 0 fully bound pairs, so that the
    replicas, still near the bare scaffold, lie inside their neighbours'
    windows and the swaps are decided by seeded grid biases."""
    import random
    say("case: mwus3d full size, 256 replicas (64 windows x 4 T), 4 rounds x 500 steps")
    s, wins, grid, glen = systems.mwus3d_system()
    s.flags |= abi.FLAG_WINDOW_TEMPERATURE_SWAPS
    glen = 8
    wins = [abi.Window(w.op, 0, w.max_op, 0, 0.0, 0.0, 1.0, 0.0, 1.0) for w in wins]
    rnd = random.Random(4711)
    grid = [rnd.uniform(-1.0, 1.0) for _ in range(256 * glen)]
    gpu = sampler_cls(s, temps=s.temps, exchange_mode=abi.EXCHANGE_WINDOWS)
    ref = oracle_mod.Oracle(s, temps=s.temps, exchange_mode=abi.EXCHANGE_WINDOWS)
    gpu.set_windows(wins, grid, glen)
    ref.set_windows(wins, grid, glen)
    for _ in range(2):
        gpu.run(2, 500)
        ref.run(2, 500)
        assert gpu.permutation() == ref.permutation()
    for r in range(256):
        assert_same(gpu, ref, r)
    assert_counters(gpu, ref)
    ag, bg = gpu.exchange_counts()
    ar, br = ref.exchange_counts()
    assert ag.tolist() == ar.tolist() and bg.tolist() == br.tolist()
    # both kinds of swap were tried and taken
    assert bg[0].sum() > 0 and bg[1].sum() > 0
    assert ag[1].sum() == 2 * 64 + 2 * 128


def case_exchange_and_site_eval(sampler_cls, oracle_mod):
    """ldo_exchange between ldo_run intervals with chosen pair sets, and
    ldo_site_eval: trial placements of every domain of a four-domain
    configuration with staples bound, at the sites around its chain
    neighbour in every orientation, at its own site and at an empty one."""
    say("case: explicit exchange rounds between PTMC intervals, 6-replica raster ladder")
    s = systems.raster_system(replicas=6)
    gpu = sampler_cls(s, temps=s.temps, exchange_mode=abi.EXCHANGE_TEMPERATURE)
    ref = oracle_mod.Oracle(s, temps=s.temps, exchange_mode=abi.EXCHANGE_TEMPERATURE)
    for k, sw in enumerate([2, 2, 1, 4, 3, 3]):
        for x in (gpu, ref):
            x.run(1, 200)
            x.exchange(sw)
        assert gpu.permutation() == ref.permutation(), k
    for r in range(6):
        assert_same(gpu, ref, r)
    cg, cr = gpu.counters(), ref.counters()
    assert (cg.exchange_attempts, cg.exchange_accepts) == (cr.exchange_attempts,
                                                           cr.exchange_accepts)
    # the runs' own rounds are 1, 3, ..., 11 (odd: pairs (1,2), (3,4)); the
    # explicit ones pair 3, 3, 2, 3, 2, 2 neighbours
    assert cg.exchange_attempts == 6 * 2 + (3 + 3 + 2 + 3 + 2 + 2)
    with pytest.raises(abi.LdoError):
        gpu.exchange(-1)

    say("case: site evaluations on the four-domain system at 345 K")
    s = systems.four_domain_system(max_total_staples=2)
    gpu = sampler_cls(s, temps=[345.0] * 2)
    ref = oracle_mod.Oracle(s, temps=[345.0] * 2)
    for x in (gpu, ref):
        x.sweep(3000)
    for r in range(2):
        assert_same(gpu, ref, r)
    units = [(1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)]
    queries = []
    for r in range(2):
        cfg = gpu.config(r)
        for c in cfg:
            n = len(c.positions)
            for d in range(n):
                queries.append((r, c.index, d, c.positions[d], c.orientations[d]))
                queries.append((r, c.index, d, (40 + d, 40, 40), (0, 0, 1)))
                a = c.positions[d - 1] if d > 0 else c.positions[(d + 1) % n]
                for u in units:
                    site = tuple(a[i] + u[i] for i in range(3))
                    for o in units:
                        queries.append((r, c.index, d, site, o))
    before = [(gpu.observables(r)["energy"], gpu.config(r)) for r in range(2)]
    got = gpu.site_eval(queries)
    want = ref.site_eval(queries)
    assert len(got) == len(want) == len(queries)
    for k, (g, w) in enumerate(zip(got, want)):
        assert g[2] == w[2], (k, queries[k], g, w)
        if not g[2]:
            assert g[1] == pytest.approx(w[1], rel=ENERGY_RTOL, abs=1e-12), (k, queries[k])
        assert g[0] == pytest.approx(w[0], rel=ENERGY_RTOL, abs=1e-12), (k, queries[k])
    # a domain put back where it was restores the energy; an empty far site
    # costs nothing
    for k in range(0, len(queries), 38):
        own, far = got[k], got[k + 1]
        assert not own[2] and own[0] + own[1] == pytest.approx(0.0, abs=1e-9), queries[k]
        assert far == (own[0], 0.0, 0), queries[k + 1]
    assert any(g[2] for g in got) and any(not g[2] and g[1] < 0 for g in got)
    # the replicas are unchanged and keep replaying the oracle
    for r in range(2):
        assert gpu.observables(r)["energy"] == before[r][0] and gpu.config(r) == before[r][1]
    for x in (gpu, ref):
        x.sweep(2000)
    for r in range(2):
        assert_same(gpu, ref, r)
    with pytest.raises(abi.LdoError):
        gpu.site_eval([(0, 99, 0, (0, 0, 0), (1, 0, 0))])
    with pytest.raises(abi.LdoError):
        gpu.site_eval([(0, 0, 0, (0, 0, 0), (1, 1, 0))])


def random_network(n_ident, seed, out_scale=3.0):
    """Seeded network parameters in the ldo_mlp.h layout; the output layer is
    scaled by `out_scale` (3: a proposal far from uniform)."""
    import numpy as np
    rng = np.random.default_rng(seed)
    H, F, E, O = 256, 4459, 16, 36
    parts = [rng.uniform(-1, 1, F * H) * np.sqrt(6 / 343), rng.uniform(-1, 1, n_ident * E),
             rng.uniform(-1, 1, E * H) * np.sqrt(6 / E), rng.uniform(-0.1, 0.1, H),
             rng.uniform(-1, 1, H * H) * np.sqrt(6 / H), rng.uniform(-0.1, 0.1, H),
             rng.uniform(-1, 1, H * H) * np.sqrt(6 / H), rng.uniform(-0.1, 0.1, H),
             rng.uniform(-1, 1, H * O) * np.sqrt(6 / H) * out_scale,
             rng.uniform(-0.5, 0.5, O) * out_scale / 3]
    return np.concatenate(parts).astype(np.float32)


def case_learned_move_matches_oracle(sampler_cls, oracle_mod):
    say("case: learned moves (domain regrowth and staple exchange, random network, CB "
        "fallback 0.1) on the 64-domain raster at 330 K and 345 K: 3 x (150 learned attempts "
        "+ 500 steps), samples")
    import numpy as np
    s = systems.raster_system(replicas=2)
    temps = [330.0, 345.0]
    gpu = sampler_cls(s, temps=temps)
    ref = oracle_mod.Oracle(s, temps=temps)
    gpu.sweep(3000)
    ref.sweep(3000)
    net = random_network(64, 11)
    gpu.learned_set_network(64, net, 0.1)
    ref.learned_set_network(64, net, 0.1)
    for _ in range(3):
        gpu.learned_sweep(150)
        ref.learned_sweep(150)
        for r in range(2):
            assert_same(gpu, ref, r)
        gpu.sweep(500)
        ref.sweep(500)
    assert_counters(gpu, ref)
    c = gpu.counters()
    # slots 5, 6, 7: learned staple exchange, CB fallback, learned domain regrowth
    assert c.attempts[5] + c.attempts[6] + c.attempts[7] == 2 * 450
    assert min(c.attempts[5], c.attempts[6], c.attempts[7]) > 0
    assert 0 < c.accepts[7] < c.attempts[7] and 0 < c.accepts[5] < c.attempts[5]
    a, b = gpu.learned_samples(4096), ref.learned_samples(4096)
    assert len(a[0]) > 0
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


def case_learned_moves_in_3d_umbrella_windows(sampler_cls, oracle_mod):
    say("case: learned moves (random network over 200 identities, CB fallback 0.1) in the "
        "200-domain 3/4-turn 5x5x8 umbrella run with three-domain staples: 8 numfulldomains "
        "windows at 318 K, 3 x (100 learned attempts + 2 window swaps x 500 steps)")
    s, wins, grid, glen = systems.mwus3d_system(windows=64, temps=(318.0,))
    wins = [abi.Window(w.op, 0, w.max_op + 4 * i, 0, 0.0, 0.0, 1.0, 0.0, 1.0)
            for i, w in enumerate(wins[:8])]
    temps = [318.0] * 8
    s.temps = temps
    gpu = sampler_cls(s, temps=temps, exchange_mode=abi.EXCHANGE_WINDOWS)
    ref = oracle_mod.Oracle(s, temps=temps, exchange_mode=abi.EXCHANGE_WINDOWS)
    net = random_network(200, 23)
    for x in (gpu, ref):
        x.set_windows(wins, grid[:8 * glen], glen)
        x.run(2, 500)
        x.learned_set_network(200, net, 0.1)
    for _ in range(3):
        for x in (gpu, ref):
            x.learned_sweep(100)
            x.run(2, 500)
        assert gpu.permutation() == ref.permutation()
        for r in range(8):
            assert_same(gpu, ref, r)
            assert gpu.observables(r)["bias"] == ref.observables(r)["bias"], r
    assert_counters(gpu, ref)
    c = gpu.counters()
    assert c.attempts[5] + c.attempts[6] + c.attempts[7] == 8 * 300
    assert c.accepts[7] > 0


def case_batch_matches_oracle(batch_cls, oracle_mod):
    say("case: batch of 12 chains (8-40 domains, 310-350 K), 3 x 500 steps, each segment on "
        "a different sweep kernel (LDS, wavefront, lane, wavefront run by its first lane)")
    ss, ts = systems.batch_systems(12, len_lo=8, len_hi=40)
    b = batch_cls(ss, ts)
    refs = [oracle_mod.Oracle(s, temps=[t]) for s, t in zip(ss, ts)]
    for kernel in (abi.BATCH_LDS, abi.BATCH_WAVE, abi.BATCH_LANE, abi.BATCH_WAVE_SOLO):
        b.set_kernel(kernel)
        b.sweep(500)
        obs = b.observables()
        for k, ref in enumerate(refs):
            ref.sweep(500)
            a, r = obs[k], ref.observables(0)
            for key in EXACT_KEYS:
                assert a[key] == r[key], (kernel, k, key, a[key], r[key])
            for key in ("energy", "enthalpy", "entropy", "stacking_energy"):
                assert a[key] == pytest.approx(r[key], rel=ENERGY_RTOL, abs=1e-12), (kernel, k, key)
            assert b.config(k) == ref.config(0), (kernel, k)
    tot = b.counters()
    sums = [ref.counters() for ref in refs]
    assert list(tot.attempts) == [sum(c.attempts[i] for c in sums) for i in range(len(tot.attempts))]
    assert list(tot.accepts) == [sum(c.accepts[i] for c in sums) for i in range(len(tot.accepts))]
    for key in ("site_empty", "site_bind", "commits"):
        assert getattr(tot, key) == sum(getattr(c, key) for c in sums), key
    chosen, ms = b.tune(20)
    assert chosen in ms and ms[chosen] is not None


def case_reference_rng_tape_replay(sampler_cls, oracle_mod):
    say("case: four-domain system, mt19937_64 tape recorded by the oracle, 30000 steps")
    s = systems.four_domain_system()
    ref = oracle_mod.Oracle(s, temps=[330.0], rng_kind=1)
    ref.record_tape(0)
    ref.sweep(30000)
    gpu = sampler_cls(s, temps=[330.0], rng_mode=abi.RNG_TAPE)
    gpu.set_tape(0, ref.tape(0))
    gpu.sweep(30000)
    assert_same(gpu, ref, 0)


def case_config_roundtrip_and_errors(sampler_cls, oracle_mod):
    say("case: set_config/get_config round trip at another temperature, argument errors")
    s = systems.four_domain_system()
    gpu = sampler_cls(s, temps=[330.0, 340.0])
    ref = oracle_mod.Oracle(s, temps=[330.0, 340.0])
    ref.sweep(20000)
    chains = ref.config(0)
    gpu.set_config(1, chains)
    ref.set_config(1, chains)
    assert gpu.config(1) == chains
    assert ref.config(1) == chains
    a, b = gpu.observables(1), ref.observables(1)
    for k in EXACT_KEYS:
        if k not in ("step", "last_move", "last_accepted"):
            # the oracle's sweep also stepped its replica 1
            assert a[k] == b[k], (k, a[k], b[k])
    for k in ("energy", "enthalpy", "entropy", "stacking_energy"):
        assert a[k] == pytest.approx(b[k], rel=ENERGY_RTOL, abs=1e-12), (k, a[k], b[k])
    assert gpu.observables(1)["energy"] == pytest.approx(ref.recompute_energy(1), rel=1e-12)
    with pytest.raises(abi.LdoError) as e:
        gpu.set_config(5, chains)
    assert e.value.code == abi.LDO_E_ARG
    bad = [systems.Chain(0, 0, [(0, 0, 0), (1, 0, 0), (3, 0, 0), (4, 0, 0)], [(0, 0, 1)] * 4)]
    with pytest.raises(abi.LdoError) as e:
        gpu.set_config(0, bad)
    assert e.value.code == abi.LDO_E_CONSTRAINT


# ------------------------------------------------ hand-built pins (pin_cases)
def case_hand_built_fourbody_configurations(sampler_cls, oracle_mod):
    """Every hand-built FourBody configuration gives the oracle's result
    (which test_oracle_pins.py holds to the hand-derived stacked-pair count
    and energy): the same observables, or the same constraint error."""
    import pin_cases as pin
    say("case: hand-built FourBody configurations (set_config)")
    for name, (pos, ore, dtype, n_stack, why) in sorted(pin.FOURBODY.items()):
        s = pin.fourbody_system(dtype)
        gpu = sampler_cls(s, temps=[330.0])
        ref = oracle_mod.Oracle(s, temps=[330.0])
        if n_stack is None:
            for x in (gpu, ref):
                with pytest.raises(abi.LdoError) as e:
                    x.set_config(0, pin.fourbody_chains(name))
                assert e.value.code == abi.LDO_E_CONSTRAINT, (name, why)
            continue
        gpu.set_config(0, pin.fourbody_chains(name))
        ref.set_config(0, pin.fourbody_chains(name))
        assert_same(gpu, ref, 0)
        ob = gpu.observables(0)
        assert ob["num_stacked_domain_pairs"] == n_stack, (name, why)
        assert ob["energy"] == pytest.approx(pin.uniform_energy(s, 330.0, 4, 2, n_stack),
                                             rel=ENERGY_RTOL, abs=1e-12), name
    for name, (pos, n_stack, why) in sorted(pin.THREE_DOMAIN.items()):
        s = systems.three_domain_system()
        gpu = sampler_cls(s, temps=[349.0])
        ref = oracle_mod.Oracle(s, temps=[349.0])
        if n_stack is None:
            for x in (gpu, ref):
                with pytest.raises(abi.LdoError) as e:
                    x.set_config(0, pin.three_domain_chains(name))
                assert e.value.code == abi.LDO_E_CONSTRAINT, (name, why)
            continue
        gpu.set_config(0, pin.three_domain_chains(name))
        ref.set_config(0, pin.three_domain_chains(name))
        assert_same(gpu, ref, 0)
        assert gpu.observables(0)["num_stacked_domain_pairs"] == n_stack, name


def case_folded_crossover_networks(sampler_cls, oracle_mod, steps=3000):
    """The raster's designed fold (64 bound pairs joined by crossover
    staples), seeded subsets of its staples and proper rotations of them:
    the device's FourBody evaluation gives the oracle's observables for each
    configuration, and the moveset started from the full fold replays the
    oracle's chain bit for bit over dense crossover networks."""
    import random
    import pin_cases as pin
    say("case: folded raster crossover networks (set_config, rotations, replay)")
    s = systems.raster_system(replicas=1)
    gpu = sampler_cls(s, temps=[330.0])
    ref = oracle_mod.Oracle(s, temps=[330.0])
    rng = random.Random(20261203)
    rot = lambda p: (p[2], p[0], p[1])  # noqa: E731
    for case in range(6):
        keep = (lambda t: True) if case == 0 else set(
            rng.sample(range(1, len(s.identities)), rng.randint(8, 28))).__contains__
        cfg = pin.folded_raster(s, keep)
        for c in (cfg, pin.rotate_chains(cfg, rot)):
            gpu.set_config(0, c)
            ref.set_config(0, c)
            assert_same(gpu, ref, 0)
    full = pin.folded_raster(s, lambda t: True)
    gpu.set_config(0, full)
    ref.set_config(0, full)
    assert gpu.observables(0)["num_stacked_domain_pairs"] == 24
    gpu.sweep(steps)
    ref.sweep(steps)
    assert_same(gpu, ref, 0)
    assert gpu.observables(0)["num_fully_bound_domain_pairs"] > 32


def case_fixed_configuration_exchange_chains(sampler_cls, oracle_mod, rounds=2000):
    """PTMC and window exchange over fixed configurations (0 MC steps per
    round): the device exchange kernel makes the oracle's decisions round by
    round, and its visit frequencies approach the exact stationary
    distribution that test_oracle_pins.py holds the oracle to."""
    import pin_cases as pin
    s = pin.exchange_system()
    cfgs, energies = pin.straight_configs()
    for mode in (abi.EXCHANGE_TEMPERATURE, abi.EXCHANGE_WINDOWS):
        say(f"case: fixed-configuration exchange chain, mode {mode}, {rounds} rounds")
        temps = pin.PT_TEMPS if mode == abi.EXCHANGE_TEMPERATURE else [pin.WIN_TEMP] * 4
        gpu = sampler_cls(s, temps=temps, exchange_mode=mode)
        ref = oracle_mod.Oracle(s, temps=temps, exchange_mode=mode)
        if mode == abi.EXCHANGE_WINDOWS:
            for x in (gpu, ref):
                x.set_windows(pin.windows(), sum(pin.WIN_GRIDS, []), len(pin.WIN_GRIDS[0]))
        for r, c in enumerate(cfgs):
            gpu.set_config(r, c)
            ref.set_config(r, c)
        if mode == abi.EXCHANGE_TEMPERATURE:
            exact = pin.ptmc_stationary(s, energies)
        else:
            exact = pin.window_stationary([e[0] for e in energies], ref.permutation())
        counts = {}
        for _ in range(rounds):
            gpu.run(1, 0)
            ref.run(1, 0)
            p = gpu.permutation()
            assert p == ref.permutation()
            counts[tuple(p)] = counts.get(tuple(p), 0) + 1
        assert set(counts) <= set(exact)
        # a loose bound at this length: the stationary law itself is pinned
        # on the oracle with 60 000 rounds
        for p, q in exact.items():
            assert abs(counts.get(p, 0) / rounds - q) < 0.08, (mode, p, q)
        for r in range(4):
            assert_same(gpu, ref, r)


def case_met_known_answer_tapes(sampler_cls, oracle_mod):
    """Met staple insertion and deletion replayed from hand-written tapes of
    the reference's draws, with the acceptance uniform just below and just
    above the hand-computed ratio (test_oracle_pins.py)."""
    import pin_cases as pin
    say("case: Met insertion/deletion known-answer tapes")
    p = 0.4
    for kind in ("insert", "delete"):
        for below in (True, False):
            u = p * (1 - 1e-9) if below else p * (1 + 1e-9)
            if kind == "insert":
                s = pin.met_system(pin.met_insert_concentration(p))
                tape = pin.met_insert_tape(u)
            else:
                s = pin.met_system(pin.met_delete_concentration(p))
                tape = pin.met_delete_tape(u)
            gpu = sampler_cls(s, temps=[pin.MET_TEMP], rng_mode=abi.RNG_TAPE)
            ref = oracle_mod.Oracle(s, temps=[pin.MET_TEMP])
            if kind == "delete":
                gpu.set_config(0, pin.met_full_chains())
                ref.set_config(0, pin.met_full_chains())
            gpu.set_tape(0, tape)
            ref.set_tape(0, tape)
            gpu.sweep(1)
            ref.sweep(1)
            assert_same(gpu, ref, 0)
            assert_counters(gpu, ref)
            staples = gpu.observables(0)["num_staples"]
            expect = (1 if below else 0) if kind == "insert" else (0 if below else 1)
            assert staples == expect, (kind, below)


# ------------------------------------------------ batches at the workload size
BATCH_LENGTHS = [8, 9, 16, 24, 31, 40, 48, 57, 64, 72, 85, 96, 101, 113, 128, 128]


def _batch_systems(lengths, t_lo=310.0, t_hi=350.0, seed=20261202):
    import dataclasses
    cache = {}
    ss, ts = [], []
    for k, L in enumerate(lengths):
        if L not in cache:
            cache[L] = systems.batch_chain_system(L)
        t = t_lo + (t_hi - t_lo) * k / max(1, len(lengths) - 1)
        ss.append(dataclasses.replace(cache[L], seed=seed + 7 * k, temps=[t]))
        ts.append(t)
    return ss, ts


def _assert_chain(obs, ref, chain, ref_cfg, k, tag):
    r = ref.observables(0)
    for key in EXACT_KEYS:
        assert obs[key] == r[key], (tag, k, key, obs[key], r[key])
    for key in ("energy", "enthalpy", "entropy", "stacking_energy"):
        assert obs[key] == pytest.approx(r[key], rel=ENERGY_RTOL, abs=1e-12), (tag, k, key)
    assert chain == ref_cfg, (tag, k)


def case_batch_lengths_8_to_128(batch_cls, oracle_mod, steps=2000):
    """Chains across the workload's length range, two of them at L = 128 (the
    LDS kernel then gives every workgroup the largest block of the
    batch), each sweep kernel for `steps` steps against per-chain oracles."""
    say(f"case: batch of {len(BATCH_LENGTHS)} chains, L = 8..128, {steps} steps on each of the "
        "LDS, wavefront, lane and first-lane kernels")
    ss, ts = _batch_systems(BATCH_LENGTHS)
    b = batch_cls(ss, ts)
    refs = [oracle_mod.Oracle(s, temps=[t]) for s, t in zip(ss, ts)]
    for kernel in (abi.BATCH_LDS, abi.BATCH_WAVE, abi.BATCH_LANE, abi.BATCH_WAVE_SOLO):
        say(f"  kernel {kernel}")
        b.set_kernel(kernel)
        b.sweep(steps)
        obs = b.observables()
        for k, ref in enumerate(refs):
            ref.sweep(steps)
            _assert_chain(obs[k], ref, b.config(k), ref.config(0), k, kernel)
    tot = b.counters()
    sums = [ref.counters() for ref in refs]
    assert list(tot.accepts) == [sum(c.accepts[i] for c in sums) for i in range(len(tot.accepts))]
    for key in ("site_empty", "site_bind", "commits"):
        assert getattr(tot, key) == sum(getattr(c, key) for c in sums), key


def case_batch_full_workload(batch_cls, oracle_mod, steps=1000):
    """The batching workload at its size: 4096 chains, L ~ U{8..128},
    T ~ U(310, 350) K, autotuned kernel.  Every chain ends OK with the
    moveset's attempt count; 16 chains spread over the batch (the longest
    among them) are replayed on the oracle and must agree bit for bit."""
    say(f"case: batch workload, 4096 chains, tune + {steps} steps, 16 chains replayed on the oracle")
    ss, ts = systems.batch_systems()
    b = batch_cls(ss, ts)
    chosen, ms = b.tune(20)
    say(f"  tuned kernel {chosen}: {ms}")
    b.sweep(steps)
    obs = b.observables()
    assert all(o["status"] == 0 for o in obs)
    n_steps = [o["step"] for o in obs]
    assert min(n_steps) == max(n_steps) and n_steps[0] >= steps
    tot = b.counters()
    assert sum(tot.attempts) == sum(n_steps)
    for o, s in zip(obs, ss):
        assert 0 <= o["num_staples"] <= s.max_total_staples
        assert o["num_fully_bound_domain_pairs"] + o["num_misbound_domain_pairs"] == \
            o["num_bound_domain_pairs"]
    longest = max(range(len(ss)), key=lambda k: len(ss[k].identities[0]))
    sample = sorted(set(list(range(0, 4096, 273)) + [longest]))[:16]
    for k in sample:
        ref = oracle_mod.Oracle(ss[k], temps=[ts[k]])
        ref.sweep(n_steps[k])
        _assert_chain(obs[k], ref, b.config(k), ref.config(0), k, "batch4096")


def case_learned_rejects_single_domain_staples(sampler_cls, oracle_mod):
    """The learned moves place a staple end next to its chain neighbour; a
    staple type of one domain has none, so both learned entry points refuse
    such a system instead of reading another chain's slot."""
    say("case: learned moves refuse single-domain staple types")
    s = systems.four_domain_system()
    s.identities = [[-1, -2, -3, -4], [1], [2, 3]]
    gpu = sampler_cls(s, temps=[330.0])
    with pytest.raises(abi.LdoError) as e:
        gpu.learned_set_network(4, random_network(4, 1))
    assert e.value.code == abi.LDO_E_NOTIMPL
    with pytest.raises(abi.LdoError) as e:
        gpu.learned_samples(16)
    assert e.value.code == abi.LDO_E_NOTIMPL


def _ctrg_chain(sampler_cls, oracle_mod, s, temps, rounds, steps):
    gpu = sampler_cls(s, temps=temps)
    ref = oracle_mod.Oracle(s, temps=temps)
    for _ in range(rounds):
        gpu.sweep(steps)
        ref.sweep(steps)
        for r in range(len(temps)):
            assert_same(gpu, ref, r)
    assert_counters(gpu, ref)
    for r in range(len(temps)):
        tr = gpu.move_tracking(r)
        assert tr == ref.move_tracking(r)
        kinds = [m.kind for m in s.moves]
        if abi.MOVE_CTRG_SCAFFOLD_REGROWTH in kinds:
            slot = kinds.index(abi.MOVE_CTRG_SCAFFOLD_REGROWTH)
            assert sum(tr["ctrg_length_attempts"]) <= gpu.counters().attempts[slot]
    return gpu


def case_ctrg_scaffold_regrowth_bit_exact(sampler_cls, oracle_mod):
    """CTRG recoil regrowth (rg_movetypes.cpp) with the reference's example
    limits (max_num_recoils 1, max_c_attempts 36): the four-domain system,
    whose segments reach both scaffold ends, and the 64-domain raster, where
    staples bound to the segment are regrown with it (stem domains, inactive
    endpoints) and networks bound outside it pin their scaffold domains."""
    say("case: CTRG scaffold regrowth, four-domain at 330/345 K (3 x 5000 steps) and "
        "64-domain raster at 300/360 K (3 x 5000 steps)")
    four = systems.four_domain_system()
    four.moves = systems.ctrg_moveset(4)
    _ctrg_chain(sampler_cls, oracle_mod, four, [330.0, 345.0], 3, 5000)
    raster = systems.raster_system(replicas=2)
    raster.moves = systems.ctrg_moveset(12)
    g = _ctrg_chain(sampler_cls, oracle_mod, raster, raster.temps, 3, 5000)
    assert g.observables(0)["num_staples"] >= 3  # staples bound at 300 K


def case_ctrg_recoil_and_attempt_limits(sampler_cls, oracle_mod):
    """Recoil growth without recoils and with one trial configuration per
    domain, with two recoils (feeler growth two levels deep), and with three
    recoils and six trial configurations, on the raster at 300 K with staples
    bound."""
    say("case: CTRG (recoils, attempts) = (0, 1), (2, 36), (3, 6) on the 64-domain raster "
        "at 300 K, 2 x 8000 steps")
    for rec, att in ((0, 1), (2, 36), (3, 6)):
        s = systems.raster_system(replicas=1)
        s.moves = systems.ctrg_moveset(12, rec, att)
        _ctrg_chain(sampler_cls, oracle_mod, s, [300.0], 2, 8000)


def case_ctrg_three_domain_staples(sampler_cls, oracle_mod):
    """CTRG through networks of three-domain staples (growth from the middle
    domain, both endpoint rules) and ThreeQuarterTurn domains."""
    say("case: CTRG on the three-domain staple system (both endpoint rules, HalfTurn and "
        "ThreeQuarterTurn, 4 replicas at 345-348 K, 3 x 4000 steps)")
    for flags in (0, abi.FLAG_CTCB_SCAFFOLD_ENDPOINTS):
        for dt in (abi.HALFTURN, abi.THREEQUARTERTURN):
            s = systems.three_domain_system(domain_type=dt, max_total_staples=2, flags=flags)
            s.moves = systems.ctrg_moveset(3, 2, 12)
            _ctrg_chain(sampler_cls, oracle_mod, s, [345.0 + i for i in range(4)], 3, 4000)


def case_ctrg_rejects_bad_limits(sampler_cls, oracle_mod):
    """max_c_attempts outside 1..36 (the trial configurations are the 36
    (site, orientation) pairs, drawn without replacement), negative
    max_num_recoils, max_regrowth below 2, and for the non-contiguous move
    max_seg_regrowth below 1 (its first segment's length is drawn from
    [2, max_seg_regrowth + 1]) or max_regrowth above 60 are refused at
    creation."""
    say("case: CTRG limits outside their ranges are refused")
    bad = [systems.ctrg_moveset(maxreg, rec, att)
           for maxreg, rec, att in ((12, 1, 37), (12, 1, 0), (12, -1, 36), (1, 1, 36))]
    bad += [systems.jump_moveset(12, 1, 36, 0), systems.jump_moveset(61, 1, 36, 2)]
    for moves in bad:
        s = systems.raster_system(replicas=1)
        s.moves = moves
        with pytest.raises(abi.LdoError) as e:
            sampler_cls(s, temps=[300.0])
        assert e.value.code == abi.LDO_E_ARG


def case_ctrg_jump_bit_exact(sampler_cls, oracle_mod):
    """Non-contiguous CTRG (select_noncontig_segs, movetypes.cpp:512-721;
    rg_movetypes.cpp:791-853) in the reference's example moveset: hairpin
    scaffolds of 4 and 6 domains whose crossover staples give stem domains
    (segment pairs grown from a staple domain, walk checks over both), and
    the 64-domain raster, whose selections are mostly single segments."""
    say("case: CTRG jump, hairpins of 4 and 6 domains at 330/345 K (3 x 5000 steps), "
        "64-domain raster at 300 K (3 x 5000 steps)")
    for n in (4, 6):
        s = systems.hairpin_system(n)
        s.moves = systems.jump_moveset(n)
        g = _ctrg_chain(sampler_cls, oracle_mod, s, [330.0, 345.0], 3, 5000)
        assert g.move_tracking(0)["ctrg_jump_attempts"][0] > 1000
    s = systems.raster_system(replicas=1)
    s.moves = systems.jump_moveset(12)
    _ctrg_chain(sampler_cls, oracle_mod, s, [300.0], 3, 5000)


def case_ctrg_jump_limits(sampler_cls, oracle_mod):
    """Non-contiguous CTRG with other limits: (recoils, attempts,
    max_seg_regrowth) = (0, 36, 1), (2, 6, 3), (3, 12, 4) on the six-domain
    hairpin at 330 K."""
    say("case: CTRG jump limits (0, 36, 1), (2, 6, 3), (3, 12, 4) on the 6-domain hairpin, "
        "2 x 6000 steps")
    for rec, att, sreg in ((0, 36, 1), (2, 6, 3), (3, 12, 4)):
        s = systems.hairpin_system(6)
        s.moves = systems.jump_moveset(6, rec, att, sreg)
        _ctrg_chain(sampler_cls, oracle_mod, s, [330.0, 340.0], 2, 6000)


def case_ctcb_jump_bit_exact(sampler_cls, oracle_mod):
    """Non-contiguous CTCB (cb_movetypes.cpp:872-983): the jump selection
    grown by configurational bias, stems bound by set_first_seg_domain, on
    the 4- and 6-domain hairpins and the 64-domain raster, with the
    reference's limits and with (max_seg_regrowth 1, 4)."""
    say("case: CTCB jump, hairpins of 4 and 6 domains at 330/345 K and the 64-domain raster "
        "at 300 K, 3 x 5000 steps")
    for n, sreg in ((4, 2), (6, 1), (6, 4)):
        s = systems.hairpin_system(n)
        s.moves = systems.ctrg_moveset(n)[:3] + [
            systems.Move(abi.MOVE_CTCB_JUMP_SCAFFOLD_REGROWTH, 2 / 6, n, 0, 0, sreg)]
        g = _ctrg_chain(sampler_cls, oracle_mod, s, [330.0, 345.0], 3, 5000)
        assert sum(g.move_tracking(0)["ctcb_jump_staples_attempts"]) > 1000
    s = systems.raster_system(replicas=1)
    s.moves = systems.ctrg_moveset(12)[:3] + [
        systems.Move(abi.MOVE_CTCB_JUMP_SCAFFOLD_REGROWTH, 2 / 6, 12, 0, 0, 2)]
    _ctrg_chain(sampler_cls, oracle_mod, s, [300.0], 3, 5000)

"""The wavefront sweep engine at the forms where it leaves the general one:
rings (segments and stacked pairs across the scaffold's ends), sequence
specific stacking (energies that differ from pair to pair), disallowed
misbinding, more staples than a wavefront has lanes, staples of up to eight
domains in strides with unused slots, centring and constraint checks every few
steps, and more active endpoints than a wavefront reads at once.  Each runs step
for step against the CPU oracle, on the host build of the engine and on the GPU,
and the general engine runs beside it."""
import ctypes as C
import dataclasses
import os
import subprocess
import time

import pytest

import parity_cases as pc
from test_engine_host_parity import HOST_DIR, HOST_LIB, sampler_cls as host_sampler  # noqa: F401
from latticednaorigami_amd import abi, systems

RING = [(0, 0, 0), (1, 0, 0), (2, 0, 0), (3, 0, 0), (3, 1, 0), (2, 1, 0), (1, 1, 0), (0, 1, 0)]


def ring(domain_type, moves):
    s = systems.four_domain_system(max_total_staples=8)
    n = len(RING)
    return dataclasses.replace(
        s, identities=[[-(i + 1) for i in range(n)], [1, 2], [3, 6], [4, 5], [7, 8], [8, 1]],
        chains=[systems.Chain(0, 0, RING, [(0, 0, 1)] * n)], cyclic=True,
        domain_type=domain_type, moves=moves(n), temps=[335.0, 348.0])


def raster(**kw):
    s = systems.raster_system(n_domains=20, width=5, replicas=2, t_lo=325.0, t_hi=345.0)
    return dataclasses.replace(s, **kw)


def crowded():
    """A concentration at which more than 64 staples hang on four domains
    (without scaffold regrowth, whose growth stack holds 32 levels)."""
    s = systems.four_domain_system(max_total_staples=160)
    moves = [systems.Move(abi.MOVE_ORIENTATION_ROTATION, 0.1),
             systems.Move(abi.MOVE_MET_STAPLE_EXCHANGE, 0.7),
             systems.Move(abi.MOVE_CB_STAPLE_REGROWTH, 0.2)]
    return dataclasses.replace(s, staple_M=3000.0, max_type_staples=160, moves=moves,
                               temps=[320.0, 350.0])


def long_staples(moves):
    s = systems.four_domain_system(max_total_staples=6)
    n = 12
    return dataclasses.replace(
        s, identities=[[-(i + 1) for i in range(n)], [1, 2, 3, 4, 5, 6, 7, 8], [9, 10, 11],
                       [12, 11, 3], [5]],
        chains=[systems.Chain(0, 0, [(i, 0, 0) for i in range(n)], [(0, 0, 1)] * n)],
        max_staple_size=8, staple_M=1e-3, moves=moves(n), temps=[340.0, 360.0],
        flags=abi.FLAG_CTCB_SCAFFOLD_ENDPOINTS)


def crossings(regrowth):
    """Two rows of 200 domains joined by a staple at every column: a regrown segment
    begins with an endpoint for each of its domains, up to 180, where a wavefront
    reads 64 at a time and holds 64 in LDS.  Binding is weak at these temperatures,
    so that the product of 180 weights stays a double (the oracle's has 64 bits and
    a wider exponent)."""
    w = 200
    s = systems.batch_chain_system(8)
    sites = [(i, 0, 0) for i in range(w)] + [(i, 1, 0) for i in range(w - 1, -1, -1)]
    ores = [(0, 0, (-1) ** i) for i in range(2 * w)]
    staples = [[i + 1, 2 * w - i] for i in range(w)]
    chains = [systems.Chain(0, 0, sites, ores)]
    for t, ids in enumerate(staples, start=1):
        at = [v - 1 for v in ids]
        chains.append(systems.Chain(t, t, [sites[i] for i in at],
                                    [tuple(-x for x in ores[i]) for i in at]))
    moves = [systems.Move(abi.MOVE_ORIENTATION_ROTATION, 0.1),
             systems.Move(abi.MOVE_MET_STAPLE_EXCHANGE, 0.1),
             systems.Move(abi.MOVE_CB_STAPLE_REGROWTH, 0.1),
             dataclasses.replace(regrowth, freq=0.7)]
    return dataclasses.replace(
        s, identities=[[-(i + 1) for i in range(2 * w)]] + staples, chains=chains, moves=moves,
        max_total_staples=w, max_type_staples=2, temps=[354.0, 358.0],
        flags=abi.FLAG_CTCB_SCAFFOLD_ENDPOINTS)


FORMS = {
    "ring": lambda: ring(abi.HALFTURN, systems.standard_moveset),
    "ring_three_quarter": lambda: ring(abi.THREEQUARTERTURN, systems.standard_moveset),
    "ring_ctrg": lambda: ring(abi.HALFTURN, systems.ctrg_moveset),
    "ring_jump": lambda: ring(abi.THREEQUARTERTURN, systems.jump_moveset),
    "sequence_stacking": lambda: raster(stacking_pot=abi.STACK_SEQUENCESPECIFIC),
    "sequence_stacking_ctrg": lambda: raster(stacking_pot=abi.STACK_SEQUENCESPECIFIC,
                                             moves=systems.ctrg_moveset(12)),
    "misbinding_disallowed": lambda: raster(misbinding_pot=abi.MISBIND_DISALLOWED),
    "crowded": crowded,
    "long_staples": lambda: long_staples(systems.standard_moveset),
    "long_staples_ctrg": lambda: long_staples(systems.ctrg_moveset),
    "crossings": lambda: crossings(
        systems.Move(abi.MOVE_CTCB_SCAFFOLD_REGROWTH, 1.0, 180)),
    "crossings_ctrg": lambda: crossings(
        systems.Move(abi.MOVE_CTRG_SCAFFOLD_REGROWTH, 1.0, 180, 1, 36)),
    "centred": lambda: raster(centering_freq=7, constraint_check_freq=11),
}


def check(make, oracle_mod, name):
    s = FORMS[name]()
    print("form", name, flush=True)
    slow = any(k in name for k in ("ctrg", "jump", "crossings"))
    steps = 4000 if name == "crowded" else 150 if slow else 1500
    os.environ["LDO_SWEEP_KERNEL"] = "global"
    try:
        general = make(s, temps=s.temps)
        general.sweep(steps)
    finally:
        del os.environ["LDO_SWEEP_KERNEL"]
    wave = make(s, temps=s.temps)
    ref = oracle_mod.Oracle(s, temps=s.temps)
    for k in range(3):
        wave.sweep(steps)
        ref.sweep(steps)
        for r in range(len(s.temps)):
            pc.assert_same(wave, ref, r)
            if k == 0:
                pc.assert_same(general, ref, r)
                assert wave.move_tracking(r) == general.move_tracking(r)
    pc.assert_counters(wave, ref)
    return wave


@pytest.mark.parametrize("name", sorted(FORMS))
def test_forms_on_the_host_build(host_sampler, oracle_mod, name):  # noqa: F811
    wave = check(host_sampler, oracle_mod, name)
    if name == "crowded":
        assert max(wave.observables(r)["num_staples"] for r in range(2)) > 64
    if name.startswith("crossings"):
        host = C.CDLL(HOST_LIB)
        host.eh_active_endpoints.argtypes = [C.c_void_p, C.c_int32]
        host.eh_wave_lds_bytes.argtypes = [C.c_void_p]
        host.eh_wave_lds_bytes.restype = C.c_int64
        assert host.eh_wave_lds_bytes(wave.h) <= 160 * 1024  # the GPU takes this engine too
        began = set()
        for _ in range(60):
            wave.sweep(1)
            began.update(host.eh_active_endpoints(wave.h, r) for r in range(2))
        assert any(64 < n <= 128 for n in began) and max(began) > 128


@pytest.mark.parametrize("target", ["alias", "fold"])
def test_sanitized_parts(target):
    """alias: records written by field and read whole are accessed in a way the compiler
    may not reorder, the type sanitizer finds nothing to name.  fold: networks of bound
    pairs score alike anywhere in the coordinate range, without undefined behaviour."""
    subprocess.run(["make", "-C", HOST_DIR, target], check=True, capture_output=True)
    r = subprocess.run([os.path.join(HOST_DIR, "_build", target + "_check")],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and not r.stderr, r.stdout + r.stderr


def test_default_lanes(host_sampler):  # noqa: F811
    """A wavefront per replica for every count where the block fits LDS, and up to
    40 000 where it does not."""
    lanes = C.CDLL(HOST_LIB).eh_default_lanes
    for n in (1, 2047, 2048, 40000, 40001, 65536):
        assert lanes(n, 1) == 64
        assert lanes(n, 0) == (64 if n <= 40000 else 1)


@pytest.mark.gpu
def test_replica_counts_around_2048_run_alike():
    """2048 replicas take the kernel that 2047 take: the same chains in about the same
    time (a lane per replica, the default there before, took 50 times as long)."""
    from latticednaorigami_amd.sampler import Sampler
    s = systems.four_domain_system(max_total_staples=8)
    temps = [320.0 + 0.01 * i for i in range(2048)]
    times, obs = {}, {}
    for n in (2047, 2048):
        print("replicas", n, flush=True)
        x = Sampler(s, temps=temps[:n])
        x.sweep(100)
        t0 = time.perf_counter()
        x.sweep(100)
        times[n] = time.perf_counter() - t0
        obs[n] = [x.observables(r) for r in (0, 1000, 2046)]
        x.close()
    assert obs[2047] == obs[2048]
    assert times[2048] < 10 * times[2047]


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(FORMS))
def test_forms_on_the_gpu(oracle_mod, name):
    from latticednaorigami_amd.sampler import Sampler
    check(Sampler, oracle_mod, name)

"""Day kernels where their waves' shares of work end (GPU), bit for bit
against the oracle."""
import ctypes

import numpy as np
import pytest

from arbo_gpu_fit_amd import abi, configs
from arbo_gpu_fit_amd.engine import Engine, SimSpec, climate_day
from tests.test_gpu_parity import _compare_series, _compare_state

pytestmark = pytest.mark.gpu


def _both(hip_lib, oracle_lib, specs, days, flags=0, checks=()):
    """Runs specs on the GPU and the oracle and compares census, series and
    kept outputs at the days in `checks` and at the end."""
    gpu, orc = Engine(hip_lib, flags=flags), Engine(oracle_lib, flags=flags & ~abi.F_GRAPH, threads=8)
    for e in (gpu, orc):
        e.init(specs, days)
    for day in sorted({*checks, days}):
        for e in (gpu, orc):
            e.step(day - e.day)
        for i in range(len(specs)):
            _compare_state(gpu.state(i), orc.state(i), f"day {day} sim {i}")
            _compare_series(gpu.series(i), orc.series(i), f"day {day} sim {i}")
            if flags & abi.F_AOI:
                assert np.array_equal(gpu.history(i), orc.history(i)), day
                assert np.array_equal(gpu.aoi(i), orc.aoi(i)), day
    gpu.close()
    orc.close()


@pytest.mark.parametrize("humans,per_day,serotypes", [(1, 3.0, 1), (40, 90.0, 2), (64, 1.5, 4), (700, 200.0, 3),
                                                      (5000, 700.5, 1)])
def test_introductions_use_their_tries_in_order(hip_lib, oracle_lib, humans, per_day, serotypes):
    """More introductions than the community has susceptible humans (every
    try is used and most repeat a human), and between one and several per
    wave's 64 tries."""
    print(f"[edges] introductions {humans} {per_day} {serotypes}", flush=True)
    p = configs.reference_params(n_serotypes=serotypes, external_infection=per_day, seed_frac_h=0.01, seed_frac_m=0.01)
    specs = [SimSpec(1, 1, np.array([humans], np.uint32), p, 5),
             SimSpec(2, 1, np.array([humans, humans + 3], np.uint32), p, 6)]
    _both(hip_lib, oracle_lib, specs, 40, flags=abi.F_AOI, checks=(1, 2, 15))


@pytest.mark.parametrize("grid,humans", [((1, 1), 3), ((16, 16), 40), ((257, 1), 30), ((23, 23), 30), ((2, 2), 9000)])
def test_age_of_infection_records_across_blocks(hip_lib, oracle_lib, grid, humans):
    """Communities below, at and above the rings' 256-community blocks, and
    communities of several waves' marks; rings that wrap; a resumed day of
    either parity."""
    print(f"[edges] rings {grid} {humans}", flush=True)
    p = configs.base_params(beta_hm=0.8, beta_mh=0.8, seed_frac_h=0.05, seed_frac_m=0.05, external_infection=3.0)
    small = configs.base_params(n_serotypes=2, beta_hm=0.8, beta_mh=0.8, seed_frac_h=0.05)
    specs = [SimSpec(3, 2, np.full(6, 50, np.uint32), small, 8),
             SimSpec(*grid, np.full(grid[0] * grid[1], humans, np.uint32), p, 9)]
    _both(hip_lib, oracle_lib, specs, 40, flags=abi.F_AOI, checks=(1, 5, 12, 25))
    gpu, orc = Engine(hip_lib, flags=abi.F_AOI), Engine(oracle_lib, flags=abi.F_AOI, threads=8)
    for e in (gpu, orc):
        e.init(specs, 40)
        e.step(11)
        st = [e.state(i) for i in range(2)]
        e.step(3)
        e.set_day(11)
        for i in range(2):
            e.write_state(i, st[i])
        e.step(6)
        e.set_day(20)
        e.step(5)
    for i in range(2):
        assert np.array_equal(gpu.aoi(i), orc.aoi(i)) and np.array_equal(gpu.history(i), orc.history(i))
    gpu.close()
    orc.close()


def test_lifetime_tables_shared_and_distinct(hip_lib, oracle_lib):
    """A batch whose simulations share lifespans, differ in one parameter of
    them, reach the last ages of the tables or follow climates: every table
    the device builds is read by births, rebirths and the t = 0 census."""
    T = 30
    base = dict(seed_frac_h=0.02, seed_frac_m=0.02)
    short = dict(h_scale=60.0, h_shape=1.0)       # rebirths every day
    specs = []

    def add(n, **over):
        climate = over.pop("climate", None)
        specs.append(SimSpec(3, 3, np.full(9, n, np.uint32), configs.base_params(**{**base, **over}), 50 + len(specs),
                             climate=climate))
    add(300)
    add(300, m_scale=10.5)
    add(200, **short)
    add(200, **short, h_infant_scale=1e-4)
    add(200, **short, h_loc=20.0)
    add(150, h_scale=3500.0, h_shape=1.0)          # exponential: draws up to the last tabulated age
    add(150, m_scale=100.0, m_shape=1.0)
    add(120, m_scale=1.0, m_shape=0.8)             # most die within a day or two
    add(100, climate=configs.seasonal_climate(T + 1))
    add(100, climate=configs.seasonal_climate(T + 1, t_amp=7.0, phase=2.0, scale_mle=2.0), m_shape=4.0)
    add(100, m_shape=4.0)
    add(300)
    print("[edges] lifetime tables", flush=True)
    _both(hip_lib, oracle_lib, specs, T, checks=(0, 1, 7))


def test_equal_climates_share_their_lifetime_rows(hip_lib, oracle_lib):
    """Simulations under one climate and lifespan share the rows of its
    lifetime table (a row a day): a batch of them takes the memory of a few,
    and one of them that differs still gets its own."""
    hip = ctypes.CDLL("libamdhip64.so.7")   # the runtime the engine is linked with

    def free():
        n, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(n), ctypes.byref(total)) == 0
        return n.value

    T, n = 3000, 48
    cl = configs.seasonal_climate(T + 1)
    other = configs.seasonal_climate(T + 1, scale_mle=2.0)
    spec = [SimSpec(1, 1, np.full(1, 50, np.uint32), configs.base_params(), 7 + i, climate=other if i == 3 else cl)
            for i in range(n)]
    print("[edges] shared climates", flush=True)
    gpu, used = Engine(hip_lib), []
    for k in (4, n):
        before = free()
        gpu.init(spec[:k], T)
        used.append(before - free())
    gpu.close()
    # a row has a guide of 256 words; a batch that replaces another returns its memory, so used[1] is the growth
    assert used[1] < (n - 4) * T * 256 * 4 // 4, used
    _both(hip_lib, oracle_lib, spec[:6], 20)


@pytest.mark.parametrize("humans,slots", [([1, 4095, 4096], [0, 4097, 4096]), ([4097, 8193, 30], [1, 12289, 8192]),
                                          ([65535, 1, 7], [100, 65535, 0])])
def test_first_census_across_workgroups(hip_lib, oracle_lib, humans, slots):
    """Communities below, at and above the members one workgroup of the t = 0
    census takes."""
    print(f"[edges] census {humans} {slots}", flush=True)
    p = configs.base_params(n_serotypes=3, immunity_mode=1, seed_frac_h=0.05, seed_frac_m=0.05)
    specs = [SimSpec(3, 1, np.array(humans, np.uint32), p, 77, mosq_slots=np.array(slots, np.uint32))]
    _both(hip_lib, oracle_lib, specs, 3, flags=abi.F_AOI | abi.F_SPATIAL, checks=(0,))


@pytest.mark.parametrize("grids,humans,omega", [([(32, 16)], 30, 0.3), ([(27, 19)], 30, 0.3), ([(8, 8)], 512, 1.0),
                                                ([(8, 8)], 513, 1.0), ([(32, 16)] * 8, 5, 0.1),
                                                ([(32, 16)] * 8 + [(1, 1)], 5, 0.1), ([(33, 1), (521, 1), (31, 1)], 25, 0.2)])
def test_small_batches_and_their_limits(hip_lib, oracle_lib, grids, humans, omega):
    """On both sides of the sizes up to which a batch's event kernel draws the
    long-distance events and sums the series itself, under both count laws,
    with staying events, and communities around the workgroups of 32."""
    print(f"[edges] small {grids[:2]} {humans} {omega}", flush=True)
    specs = []
    for i, (w, h) in enumerate(grids):
        over = dict(count_law=abi.COUNT_STOCH_ROUND) if i % 2 else {}
        if i % 3 == 1:
            over.update(no_distance=0.3, include_self=0)
        p = configs.base_params(beta_hm=0.7, beta_mh=0.7, seed_frac_h=0.05, seed_frac_m=0.05, long_distance=omega, **over)
        specs.append(SimSpec(w, h, np.full(w * h, humans, np.uint32), p, 90 + i))
    _both(hip_lib, oracle_lib, specs, 25, flags=abi.F_GRAPH, checks=(3, 9))


@pytest.mark.parametrize("grids", [[(32, 16), (16, 32)], [(32, 16), (16, 32), (1, 1)]])
def test_waves_per_community_of_an_unset_tuning(hip_lib, oracle_lib, grids):
    """1,024 communities, which the engine gives four waves each, and 1,025,
    which keep one; a tuning that was set holds for both, and reading one sets
    none."""
    print(f"[edges] waves {grids}", flush=True)
    p = configs.base_params(beta_hm=0.7, beta_mh=0.7, seed_frac_h=0.05, seed_frac_m=0.05)
    specs = [SimSpec(w, h, np.where(np.arange(w * h) % 7 == i, 600, 9).astype(np.uint32), p, 40 + i)
             for i, (w, h) in enumerate(grids)]
    orc = Engine(oracle_lib, threads=8)
    gpu = Engine(hip_lib, flags=abi.F_GRAPH)
    orc.init(specs, 12)
    orc.step(12)
    default = gpu.tuning()
    assert default["waves_per_comm"] == 1
    for knobs in ({}, default):
        gpu.init(specs, 12)
        if knobs:
            gpu.set_tuning(**knobs)
        gpu.step(12)
        assert gpu.tuning() == default
        for i in range(len(grids)):
            _compare_state(gpu.state(i), orc.state(i), f"sim {i}")
            _compare_series(gpu.series(i), orc.series(i), f"sim {i}")
    gpu.close()
    orc.close()


@pytest.mark.parametrize("humans,slots", [([30, 9000, 400, 5], [8193, 30000, 300, 1]),
                                          ([20000, 1, 65535, 700], [8192, 16385, 65535, 40000])])
@pytest.mark.parametrize("flags", [0, abi.F_AOI])
def test_large_communities_of_small_batches(hip_lib, oracle_lib, humans, slots, flags):
    """Several waves apply a community's events: bitmaps that end in the
    first, a middle and the last wave's words, days of one and of many
    chunks, introductions between the serotypes, long-distance arrivals."""
    print(f"[edges] large {humans} {slots} {flags}", flush=True)
    p = configs.base_params(beta_hm=0.8, beta_mh=0.8, seed_frac_h=0.05, seed_frac_m=0.05, external_infection=60.0,
                            long_distance=0.1)
    q = configs.base_params(n_serotypes=2, beta_hm=0.8, beta_mh=0.8, seed_frac_h=0.02, long_distance=0.05)
    specs = [SimSpec(2, 2, np.array(humans, np.uint32), c, 31, mosq_slots=np.array(slots, np.uint32)) for c in (p, q)]
    _both(hip_lib, oracle_lib, specs, 16, flags=flags, checks=(1, 6))


@pytest.mark.parametrize("grid", [(1024, 1024), (1025, 1024), (4096, 4096)])
def test_first_census_of_many_communities(hip_lib, oracle_lib, grid):
    """As many communities as one launch of the t = 0 census takes, one row
    more, and the most that a simulation may have; beyond 2^26 - 1 a batch is
    refused."""
    print(f"[edges] communities {grid}", flush=True)
    p = configs.base_params(n_serotypes=2, seed_frac_h=0.1, seed_frac_m=0.1, neighbourhood=4)
    spec = SimSpec(*grid, np.ones(grid[0] * grid[1], np.uint32), p, 5)
    gpu, orc = Engine(hip_lib), Engine(oracle_lib, threads=8)
    for e in (orc, gpu):
        e.init([spec], 1)
        e.step(1)
        print("[edges] stepped", flush=True)
    _compare_series(gpu.series(0), orc.series(0), "series")
    if grid != (4096, 4096):
        _compare_state(gpu.state(0), orc.state(0), "state")
    else:
        with pytest.raises(RuntimeError, match="communities"):
            gpu.init([spec] * 4, 1)
    gpu.close()
    orc.close()


@pytest.mark.parametrize("grids", [[(1277, 1), (1, 3)], [(1277, 1), (2, 2)], [(33, 77), (7, 1), (4, 3)], [(32, 80), (1, 1)],
                                   [(64, 79), (32, 1), (8, 4)], [(64, 79), (5, 13)], [(3, 1), (33, 1), (31, 9), (641, 19)]])
def test_event_counts_of_few_and_many_communities(hip_lib, oracle_lib, grids):
    """1,280, 2,560 and 5,120 communities, up to which a workgroup of the
    event counts takes 4, 8 and 16, and one more: blocks that end with a
    simulation, days without and with events in them."""
    print(f"[edges] counts {grids}", flush=True)
    specs = []
    for i, (w, h) in enumerate(grids):
        over = dict(count_law=abi.COUNT_STOCH_ROUND, no_distance=0.3) if i % 2 else {}
        p = configs.base_params(beta_hm=0.7, beta_mh=0.7, seed_frac_h=0.05 if i != 1 else 0.0, seed_frac_m=0.01,
                                long_distance=0.05, **over)
        specs.append(SimSpec(w, h, np.where(np.arange(w * h) % 5 == 3, 150, 6).astype(np.uint32), p, 70 + i))
    _both(hip_lib, oracle_lib, specs, 20, checks=(2, 9))


@pytest.mark.parametrize("grids,small", [([(1, 1)], True), ([(5, 3), (1, 2)], True), ([(23, 23)], False),
                                         ([(36, 36), (3, 2)], False), ([(51, 51)], False), ([(72, 72)], False)])
@pytest.mark.parametrize("serotypes,staying", [(1, 0.0), (4, 0.4)])
def test_event_counts_on_both_sides_of_the_inversion(hip_lib, oracle_lib, grids, small, serotypes, staying):
    """Mean event counts from below 1 to several hundred in one wave, so that
    from one to all of its lanes draw by rejection and share the others' lanes
    for their trials: in small batches, and in workgroups of 4, 8, 16 and 32
    communities."""
    print(f"[edges] rejection {grids} {serotypes} {staying}", flush=True)
    specs = []
    for i, (w, h) in enumerate(grids):
        humans = np.array([1, 3, 17, 60, 400, 9, 130], np.uint32)[(np.arange(w * h) + 4) % 7]
        p = configs.base_params(n_serotypes=serotypes, beta_hm=0.6, beta_mh=0.5, seed_frac_h=0.15, seed_frac_m=0.1,
                                long_distance=0.002, no_distance=staying)
        specs.append(SimSpec(w, h, humans, p, 90 + i))
    gpu = Engine(hip_lib)
    gpu.init(specs, 2)
    assert gpu.launch_shape()["small_batch"] == small
    gpu.close()
    _both(hip_lib, oracle_lib, specs, 8, checks=(1, 3))


@pytest.mark.parametrize("grids,humans,big", [([(10, 10)], 300, 0), ([(32, 16)], 40, 0), ([(32, 16)] * 5 + [(3, 1)], 9, 0),
                                              ([(2, 2)], 2000, 12000)])
@pytest.mark.parametrize("climate", [False, True])
def test_small_batches_by_what_they_send(hip_lib, oracle_lib, grids, humans, big, climate):
    """omega x slots x the transmission rates, times the waves per SIMD that
    draw the events or over the waves of a community that share them, up to
    24,000 and above it; with a climate the days' largest rates count."""
    T = 15
    cl = configs.seasonal_climate(T + 1, biting_rate=6.0) if climate else None
    n_comm = sum(w * h for w, h in grids)

    def specs(omega):
        out = []
        for i, (w, h) in enumerate(grids):
            n = np.full(w * h, humans, np.uint32)
            n[0] += big
            p = configs.base_params(beta_hm=2.0, beta_mh=1.5, seed_frac_h=0.05, seed_frac_m=0.05, long_distance=omega)
            out.append(SimSpec(w, h, n, p, 60 + i, climate=cl))
        return out
    gpu = Engine(hip_lib)
    gpu.init(specs(0.0), T)
    beta = 3.5
    if climate:
        beta = max(sum(climate_day(cl, r, oracle_lib)[:2]) for r in range(1, T + 1))
    waves = 8 if gpu.launch_shape()["waves_per_comm"] == 8 else 1
    assert waves == (8 if big else 1) and gpu.launch_shape()["small_batch"]
    slots = max(gpu.sizes(i)[2] for i in range(len(grids)))
    limit = 24000.0 * waves / (slots * beta * max(1.0, n_comm / 1024))
    print(f"[edges] sends {grids[:2]} {climate} omega {limit:.3f}", flush=True)
    assert limit * 1.01 < 1.0
    for omega, small in ((limit * 0.99, True), (limit * 1.01, False)):
        gpu.init(specs(omega), T)
        assert gpu.launch_shape()["small_batch"] == small
        _both(hip_lib, oracle_lib, specs(omega), T, checks=(4,))
    gpu.close()


@pytest.mark.parametrize("grids,law", [([(16, 16), (20, 13), (27, 19)], 0), ([(128, 256), (1, 1)], 0), ([(181, 183), (9, 9)], 1)])
def test_day_sums_of_many_workgroups(hip_lib, oracle_lib, grids, law):
    """Simulations of 64 and 65 workgroups of event counts (one record of the
    day's sums and two), and of 1,024 and more (the most records): the series
    and the first day's scan counts, and days of either parity done again."""
    print(f"[edges] sums {grids} {law}", flush=True)
    specs = [SimSpec(w, h, np.where(np.arange(w * h) % 3 == 1, 9, 4).astype(np.uint32),
                     configs.base_params(beta_hm=0.8, beta_mh=0.8, seed_frac_h=0.1, seed_frac_m=0.05, long_distance=0.1, count_law=law),
                     90 + i) for i, (w, h) in enumerate(grids)]
    gpu, orc = Engine(hip_lib), Engine(oracle_lib, threads=8)
    for e in (gpu, orc):
        e.init(specs, 12)
    assert not gpu.launch_shape()["small_batch"]
    for e in (gpu, orc):
        e.step(1)
    assert gpu.scan_counts() == orc.scan_counts()   # on day 0 both read everything
    for e in (gpu, orc):
        e.step(4)
    kept = [orc.state(i) for i in range(len(specs))]
    for e in (gpu, orc):
        e.step(4)
    for day in (5, 6):
        for e in (gpu, orc):
            for i, s in enumerate(kept):
                e.write_state(i, s)
            e.set_day(day)
            e.step(12 - day)
        for i in range(len(specs)):
            _compare_state(gpu.state(i), orc.state(i), f"sim {i}")
            _compare_series(gpu.series(i), orc.series(i), f"sim {i}")
    gpu.close()
    orc.close()

"""Launch tunings of the day kernels change no result (GPU).

Every candidate of arbo_tuning_candidates (census loads in flight, early
mosquito loads, XCD-contiguous community order, 8 waves per SIMD, several
waves per community) and the extremes of the
long-distance split give the oracle's census and series bit for bit, and an
autotuned run, graph replay included, equals an untuned one."""
import ctypes

import numpy as np
import pytest

from arbo_gpu_fit_amd import abi, configs
from arbo_gpu_fit_amd.engine import Engine, SimSpec
from tests.cases import CASES
from tests.test_gpu_parity import _compare_series, _compare_state

pytestmark = pytest.mark.gpu


def _reference(oracle_lib, specs, T):
    orc = Engine(oracle_lib, threads=8)
    orc.init(specs, T)
    orc.step(T)
    out = [(orc.state(i), orc.series(i)) for i in range(len(specs))]
    orc.close()
    return out


@pytest.mark.parametrize("case", ["ragged", "batch_pair", "climate", "burst"])
def test_every_tuning_is_bit_identical(case, hip_lib, oracle_lib):
    specs, T = CASES[case]()
    ref = _reference(oracle_lib, specs, T)
    gpu = Engine(hip_lib)
    cands = gpu.tuning_candidates()
    cands += [dict(cands[0], ld_split=1), dict(cands[1], ld_split=64)]
    for cand in cands:
        print(f"[tuning] case={case} tuning={cand}", flush=True)
        gpu.init(specs, T)
        gpu.set_tuning(**cand)
        assert gpu.tuning() == cand
        gpu.step(T)
        for i, (st, se) in enumerate(ref):
            _compare_state(gpu.state(i), st, f"{cand} sim {i}")
            _compare_series(gpu.series(i), se, f"{cand} sim {i}")
    gpu.close()


@pytest.mark.parametrize("flags", [0, abi.F_GRAPH])
def test_autotuned_run_equals_untuned(flags, hip_lib, oracle_lib):
    specs, T = CASES["lattice10"]()
    ref = _reference(oracle_lib, specs, T)
    gpu = Engine(hip_lib, flags=flags)
    gpu.init(specs, T)
    gpu.step(10)
    n = len(gpu.tuning_candidates())
    chosen, ms = gpu.autotune(days_each=2)
    print(f"[tuning] autotune flags={flags}: {chosen} {ms:.3f} ms/day", flush=True)
    assert gpu.day == 10 + 2 * n
    assert chosen == gpu.tuning() and ms > 0
    gpu.step(T - gpu.day)
    _compare_state(gpu.state(0), ref[0][0], "autotuned")
    _compare_series(gpu.series(0), ref[0][1], "autotuned")
    gpu.close()


def test_unsupported_tuning_is_rejected(hip_lib):
    gpu = Engine(hip_lib)
    with pytest.raises(RuntimeError):
        gpu.set_tuning(census_unroll=3)
    with pytest.raises(RuntimeError):
        gpu.set_tuning(ld_split=0)
    gpu.close()


def test_every_tuning_keeps_the_outputs(hip_lib, oracle_lib):
    """The instantiations that keep the infection history, the per-community
    series and the age-of-infection rings, under every launch tuning."""
    specs, T = CASES["reference_params"]()
    flags = abi.F_SPATIAL | abi.F_AOI
    orc = Engine(oracle_lib, flags=flags, threads=4)
    orc.init(specs, T)
    orc.step(T)
    ref = (orc.spatial(0), orc.history(0), orc.aoi(0), orc.state(0))
    orc.close()
    gpu = Engine(hip_lib, flags=flags)
    for cand in gpu.tuning_candidates():
        print(f"[tuning] outputs kept, tuning={cand}", flush=True)
        gpu.init(specs, T)
        gpu.set_tuning(**cand)
        gpu.step(T)
        assert np.array_equal(gpu.spatial(0), ref[0]), cand
        assert np.array_equal(gpu.history(0), ref[1]), cand
        assert np.array_equal(gpu.aoi(0), ref[2]), cand
        _compare_state(gpu.state(0), ref[3], f"{cand}")
    gpu.close()


@pytest.mark.parametrize("flags", [0, abi.F_SPATIAL | abi.F_AOI, abi.F_GRAPH])
def test_large_communities_under_every_tuning(hip_lib, oracle_lib, flags):
    """Communities above 8,192 slots (up to 65,535 humans and slots) take the
    eight-wave demography kernel and the eight-pass event kernel whatever
    the tuning asks for; census, series and kept outputs equal the
    oracle's."""
    specs, T = CASES["large"]()
    orc = Engine(oracle_lib, flags=flags & ~abi.F_GRAPH, threads=8)
    orc.init(specs, T)
    orc.step(T)
    ref = (orc.state(0), orc.series(0))
    kept = (orc.spatial(0), orc.history(0), orc.aoi(0)) if flags & abi.F_AOI else None
    orc.close()
    gpu = Engine(hip_lib, flags=flags)
    cands = gpu.tuning_candidates()
    for cand in (cands[0], cands[-1]):   # one wave per community, and four
        print(f"[tuning] large communities, flags={flags}, tuning={cand}", flush=True)
        gpu.init(specs, T)
        gpu.set_tuning(**cand)
        gpu.step(T)
        _compare_state(gpu.state(0), ref[0], f"large {cand}")
        _compare_series(gpu.series(0), ref[1], f"large {cand}")
        if kept:
            assert np.array_equal(gpu.spatial(0), kept[0])
            assert np.array_equal(gpu.history(0), kept[1])
            assert np.array_equal(gpu.aoi(0), kept[2])
    gpu.close()


def _lattice(grids, seed=40):
    p = configs.base_params(beta_hm=0.7, beta_mh=0.7, seed_frac_h=0.05, seed_frac_m=0.05)
    return [SimSpec(w, h, np.full(w * h, 9, np.uint32), p, seed + i) for i, (w, h) in enumerate(grids)]


SMALL, LARGE = [(32, 16)], [(27, 19)]   # 512 communities in a simulation, and one more


def test_waves_stay_the_engines_until_they_are_set(hip_lib):
    """A small batch's communities keep their four waves through a tuning
    that names other knobs, and through one found on a large batch; a named
    number of waves holds."""
    gpu = Engine(hip_lib, flags=abi.F_GRAPH)
    with pytest.raises(RuntimeError):
        gpu.launch_shape()   # no batch yet

    def shape(grids):
        gpu.init(_lattice(grids), 60)
        return gpu.launch_shape()
    four, one = ({"small_batch": True, "waves_per_comm": n} for n in (4, 1))
    assert shape(SMALL) == four
    gpu.set_tuning(ld_split=4, xcd_order=3)
    assert gpu.launch_shape() == four and gpu.tuning()["ld_split"] == 4
    assert shape(SMALL) == four
    assert shape(LARGE) == {"small_batch": False, "waves_per_comm": 1}
    chosen, _ = gpu.autotune(2)
    assert gpu.launch_shape()["waves_per_comm"] == chosen["waves_per_comm"]
    if chosen["waves_per_comm"] == 1:
        assert shape(SMALL) == four
    gpu.set_tuning(census_unroll=4, early_mosq=2, waves_per_simd=0, waves_per_comm=1)
    assert shape(SMALL) == one
    gpu.set_tuning(ld_split=8)
    assert shape(SMALL) == one
    assert shape([(32, 16), (32, 16), (1, 1)]) == one
    gpu.close()
    gpu = Engine(hip_lib)
    assert shape([(32, 16), (32, 16)]) == four
    assert shape([(32, 16), (32, 16), (1, 1)]) == one
    gpu.set_tuning(**gpu.tuning())   # all of them named
    assert shape(SMALL) == one
    with pytest.raises(RuntimeError):
        gpu.set_tuning(waves_per_comm=0)
    assert gpu.lib.arbo_update_tuning(gpu._h, ctypes.byref(abi.Tuning()), 64) == abi.E_INVALID
    gpu.close()


def test_autotuning_a_small_batch_compares_its_waves(hip_lib):
    """Candidates that are one kernel in a small batch leave the other knobs
    as they were; a batch whose bitmaps need eight waves has nothing to
    choose."""
    gpu = Engine(hip_lib)
    gpu.init(_lattice(SMALL), 60)
    gpu.set_tuning(ld_split=16, xcd_order=1)
    before = gpu.tuning()
    chosen, ms = gpu.autotune(2)
    assert chosen == gpu.tuning() and ms > 0 and gpu.day == 2 * len(gpu.tuning_candidates())
    assert gpu.launch_shape()["waves_per_comm"] == chosen["waves_per_comm"]
    assert chosen["waves_per_comm"] > 1 or chosen == before
    gpu.set_tuning(**before)
    gpu.init([SimSpec(1, 1, np.array([40000], np.uint32), configs.base_params(), 3, mosq_slots=np.array([65535], np.uint32))], 60)
    assert gpu.launch_shape() == {"small_batch": True, "waves_per_comm": 8}
    assert gpu.autotune(1)[0] == before
    gpu.close()

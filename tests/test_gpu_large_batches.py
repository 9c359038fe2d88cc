"""The day kernels of large batches (GPU), bit for bit against the oracle.

The parity cases are small batches, whose days run other kernels: each is
run here beside one more simulation of 513 communities of a few humans, one
above the most that a small batch's simulation may have, so that its days
take the demography kernel's tunings, the event counts, the long-distance
kernel and the event kernel of large batches."""
import numpy as np
import pytest

from arbo_gpu_fit_amd import abi, configs
from arbo_gpu_fit_amd.engine import Engine, SimSpec
from tests.cases import CASES
from tests.random_cases import N_RANDOM, random_case
from tests.test_gpu_parity import _compare_series, _compare_state

pytestmark = pytest.mark.gpu


def _enlarged(specs, days):
    p = configs.base_params(beta_hm=0.6, beta_mh=0.6, seed_frac_h=0.05, seed_frac_m=0.05, long_distance=0.1)
    return specs + [SimSpec(27, 19, np.full(513, 5, np.uint32), p, 99)], days


def _outputs(eng, n, flags):
    out = []
    for i in range(n):
        kept = (eng.spatial(i),) if flags & abi.F_SPATIAL else ()
        if flags & abi.F_AOI:
            kept += (eng.history(i), eng.aoi(i))
        out.append((eng.state(i), eng.series(i), kept))
    return out


def _reference(oracle_lib, specs, days, flags):
    orc = Engine(oracle_lib, flags=flags & ~abi.F_GRAPH, threads=8)
    orc.init(specs, days)
    orc.step(days)
    out = _outputs(orc, len(specs), flags)
    orc.close()
    return out


def _compare(gpu, ref, flags, tag):
    for i, ((st, se, kept), (st0, se0, kept0)) in enumerate(zip(_outputs(gpu, len(ref), flags), ref)):
        _compare_state(st, st0, f"{tag} sim {i}")
        _compare_series(se, se0, f"{tag} sim {i}")
        for a, b in zip(kept, kept0):
            assert np.array_equal(a, b), (tag, i)


@pytest.mark.parametrize("case,flags", [("ragged", 0), ("batch_pair", 0), ("climate", 0), ("burst", 0), ("burst", abi.F_AOI),
                                        ("reference_params", abi.F_SPATIAL | abi.F_AOI),
                                        ("climate", abi.F_SPATIAL | abi.F_AOI), ("poisson_stay", abi.F_GRAPH)])
def test_every_tuning_of_a_large_batch(case, flags, hip_lib, oracle_lib):
    specs, days = _enlarged(*CASES[case]())
    ref = _reference(oracle_lib, specs, days, flags)
    gpu = Engine(hip_lib, flags=flags)
    cands = gpu.tuning_candidates()
    cands += [dict(cands[0], ld_split=1), dict(cands[1], ld_split=64), dict(cands[2], xcd_order=1), dict(cands[3], xcd_order=2)]
    for cand in cands:
        print(f"[large] case={case} flags={flags} tuning={cand}", flush=True)
        gpu.init(specs, days)
        gpu.set_tuning(**cand)
        assert gpu.launch_shape() == {"small_batch": False, "waves_per_comm": cand["waves_per_comm"]}
        gpu.step(days)
        _compare(gpu, ref, flags, f"{case} {cand}")
    gpu.close()


@pytest.mark.parametrize("flags", [0, abi.F_SPATIAL | abi.F_AOI, abi.F_GRAPH])
def test_large_communities_of_a_large_batch(hip_lib, oracle_lib, flags):
    """Communities above 8,192 slots: the eight-wave demography kernel and the
    event kernel of eight spans a wave."""
    specs, days = _enlarged(*CASES["large"]())
    ref = _reference(oracle_lib, specs, days, flags)
    gpu = Engine(hip_lib, flags=flags)
    cands = gpu.tuning_candidates()
    for cand in (cands[0], cands[7], cands[-1]):
        print(f"[large] communities, flags={flags} tuning={cand}", flush=True)
        gpu.init(specs, days)
        gpu.set_tuning(**cand)
        assert gpu.launch_shape() == {"small_batch": False, "waves_per_comm": 8}
        gpu.step(days)
        _compare(gpu, ref, flags, f"large {cand}")
    gpu.close()


@pytest.mark.parametrize("k", range(N_RANDOM))
def test_random_simulations_in_a_large_batch(k, hip_lib, oracle_lib):
    specs, days = _enlarged(*random_case(k))
    flags = abi.F_SPATIAL | abi.F_AOI if k % 3 == 0 else abi.F_GRAPH if k % 3 == 1 else 0
    gpu = Engine(hip_lib, flags=flags)
    cand = gpu.tuning_candidates()[k % 12]
    print(f"[large] random {k} flags={flags} tuning={cand}", flush=True)
    gpu.init(specs, days)
    gpu.set_tuning(**cand)
    assert not gpu.launch_shape()["small_batch"]
    gpu.step(days)
    _compare(gpu, _reference(oracle_lib, specs, days, flags), flags, f"random {k}")
    gpu.close()

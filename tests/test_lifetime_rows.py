"""What sizes the mosquito lifetime rows (CPU): the host's walk over the days
against every row tabulated in full, compiled from the engine's own source.

A row is staged in LDS by every community and day, so its length is the
largest age at which a row reaches 2^24, no more; tables of less would cut
lifetimes off."""
import os
import subprocess

from arbo_gpu_fit_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <algorithm>
#include <cstdio>
#include "arbo_tables.h"
#include "arbo_rng.h"
using namespace arbo;

// The largest first age with threshold 2^24 over all rows, tabulated.
static uint32_t tabulated(const SimTables& t, const ArboParams& p, uint32_t days) {
    auto first = [&](uint32_t row) {
        uint32_t a = 1;
        for (; a < kMosqAgeTable - 1; ++a) {
            const double s = row == 0 ? (double)p.m_scale : t.scale[std::min(row - 1 + a, days - 1)];
            if (fixed24(weibull_cdf((double)a, s, (double)p.m_shape)) >= kOne24) break;
        }
        return a;
    };
    uint32_t most = 0;
    for (uint32_t r = 0; r < t.m_rows; ++r) most = std::max(most, first(r));
    return most;
}

int main() {
    int checked = 0, bad = 0;
    for (uint32_t days : {1u, 2u, 40u, 200u, 363u, 900u})
        for (int shape_of : {0, 1, 2, 3, 4})
            for (int kind = 0; kind < 6; ++kind) {
                std::vector<float> T(days + 1), H(days + 1), P(days + 1, 0.3f);
                for (uint32_t d = 0; d <= days; ++d) {
                    const int season = (int)(d % 365) - 180, wave = (int)((d * 7919u) % 13u);
                    T[d] = 25.0f + (kind == 1 ? season / 40.0f : kind == 2 ? -season / 40.0f : kind == 3 ? wave - 6.0f : 0.0f);
                    H[d] = kind == 4 ? (d < days / 2 ? 0.8f : 0.3f) : kind == 5 ? (d == days ? 0.9f : 0.2f) : 0.6f;
                }
                ArboClimate cl{};
                cl.temperature = T.data(); cl.humidity = H.data(); cl.precipitation = P.data(); cl.days = days + 1;
                cl.biting_rate = 0.5f; cl.scale_eip = 2.5f; cl.scale_mle = kind == 3 ? 1.0f : 2.5f; cl.scale_cc = 1.0f;
                cl.scale_humidity = 1.0f; cl.min_mos_to_human = 2.0f; cl.mos_net_growth = 0.3f;
                ArboParams p{};
                p.n_serotypes = 1; p.neighbourhood = 4; p.include_self = 1; p.iip_min = 4; p.iip_max = 7;
                p.recovery = 5.0f; p.eip = 10.0f; p.h_scale = 27000.0f; p.h_shape = 6.0f; p.m_ratio = 2.0f;
                p.m_scale = 10.0f;
                p.m_shape = shape_of == 0 ? 1.0f : shape_of == 1 ? 4.0f : shape_of == 2 ? 0.6f : shape_of == 3 ? 2.3f : 11.0f;
                const uint32_t humans[1] = {10};
                for (bool climate : {false, true}) {
                    ArboShape sh{};
                    sh.grid_w = sh.grid_h = 1; sh.humans = humans; sh.climate = climate ? &cl : nullptr;
                    SimTables t;
                    build_tables(sh, p, 1, days, t);
                    const uint32_t want = tabulated(t, p, days);
                    ++checked;
                    if (t.death_m_max != want) {
                        ++bad;
                        printf("days %u shape %g kind %d climate %d: %u, tabulated %u\n", days, p.m_shape, kind, climate,
                               t.death_m_max, want);
                    }
                }
            }
    printf("%d checked, %d differ\n", checked, bad);
    return bad != 0;
}
"""


# Scales whose certain age lies at a whole day, and the floats about them.
WHOLE_DAYS = r"""
#include <cmath>
#include <cstdio>
#include "arbo_tables.h"
#include "arbo_rng.h"
using namespace arbo;

int main() {
    int checked = 0, bad = 0;
    ArboParams p{};
    p.n_serotypes = 1; p.neighbourhood = 4; p.include_self = 1; p.iip_min = 4; p.iip_max = 7;
    p.recovery = 5.0f; p.eip = 10.0f; p.h_scale = 27000.0f; p.h_shape = 6.0f; p.m_ratio = 2.0f;
    const uint32_t humans[1] = {10};
    ArboShape sh{};
    sh.grid_w = sh.grid_h = 1; sh.humans = humans;
    for (float shape : {0.04f, 0.1f, 0.6f, 1.0f, 4.0f, 11.0f, 99.0f, 400.0f})
        for (uint32_t age : {1u, 2u, 3u, 17u, 150u, 1000u, 2045u, 2046u, 2047u, 2048u, 5000u}) {
            float scale = (float)(age / pow(54.0 * log(2.0), 1.0 / (double)shape));
            for (int k = 0; k < 4; ++k) scale = nextafterf(scale, 0.0f);
            for (int k = -4; k <= 4; ++k, scale = nextafterf(scale, 1e30f)) {
                if (!(scale > 0.0f)) continue;
                p.m_shape = shape;
                p.m_scale = scale;
                SimTables t;
                build_tables(sh, p, 1, 1, t);
                uint32_t want = 1;
                while (want < kMosqAgeTable - 1 && fixed24(weibull_cdf((double)want, (double)scale, (double)shape)) < kOne24) ++want;
                ++checked;
                if (t.death_m_max != want) {
                    ++bad;
                    printf("shape %g scale %.9g: %u, tabulated %u\n", shape, scale, t.death_m_max, want);
                }
            }
        }
    printf("%d checked, %d differ\n", checked, bad);
    return bad != 0;
}
"""


def _run(tmp_path, program):
    src, exe = tmp_path / "rows.cpp", tmp_path / "rows"
    src.write_text(program)
    csrc = os.path.join(ROOT, "arbo_gpu_fit_amd", "csrc")
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(build.hipcc())))
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    "-I", os.path.join(ROOT, "include"), "-I", csrc, "-o", str(exe), str(src), os.path.join(csrc, "arbo_tables.cpp")],
                   check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    print(out.stdout)
    assert out.returncode == 0, out.stdout


def test_rows_are_as_long_as_their_ages(tmp_path):
    _run(tmp_path, PROGRAM)


def test_ages_certain_at_a_whole_day(tmp_path):
    _run(tmp_path, WHOLE_DAYS)

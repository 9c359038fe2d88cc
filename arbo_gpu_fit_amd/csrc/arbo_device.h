// arbo_device.h — HBM layout of a batch of simulations, as the kernels see it.
//
// Every simulation of the batch is flattened into global arrays:
//   human words   u32  h_word[]  (4-element aligned per community)
//   human next    u16  h_next[]
//   human birth   i32  h_birth[]   (cold: written at rebirth only)
//   mosquito word u16  m_word[]  (32-element aligned per community)
//   mosquito next u16  m_next[]
//   alive bitmap  u32  alive[]   (bit j of word m_off/32 + j/32: slot alive after emergence)
// A community is the unit of work of both day kernels; its descriptor gives
// the offsets of its members and of its CSR row and in-edges.
#pragma once
#include <stdint.h>

#include "arbo_rng.h"

namespace arbo {

constexpr uint32_t kWave = 64;            // threads per workgroup: one wavefront per community
constexpr uint32_t kCntPerComm = 72;      // event counts of a source: [dir 2][serotype 4][row slot 9]
constexpr uint32_t kInboxEdges = 9;       // in-edges per destination (Moore-8 + self)
constexpr uint32_t kHumanAlign = 4;       // humans per 16-byte vector
constexpr uint32_t kMosqAlign = 128;      // mosquito slots per 16-byte group of alive-bitmap words
constexpr uint32_t kAoiRecord = 5000;     // ages per age-of-infection ring
// Per-community partials of a day, written by the demography kernel and
// summed by k_day_counts: word 0 mosquitoes alive after the
// births, 1 humans, 2-3 infectious humans (two 16-bit serotype pairs), 4-5
// E->I onsets (pairs), 6-7 the 16-byte census vectors of humans and of
// mosquitoes the day's scan read, 8-9 infectious mosquitoes (pairs); in small
// batches 8-23 the eight long-distance rates or counts (u64) instead.
constexpr uint32_t kPartWords = 24;
// Communities of a batch: a launch holds fewer than 2^32 threads, and the day
// kernels take at least 64 a community.
constexpr uint64_t kMaxCommunities = (1ull << 26) - 1;
// Communities of a workgroup of k_day_counts: 32, or fewer (4, 8, 16) while that
// makes no more than kCountBlocks workgroups.  The 256 threads share their
// communities' events, so fewer communities shorten an epidemic's days; on
// quiet days a workgroup more costs 2 ns.  One simulation, transmission rates
// 0.7, us a day with 32, 16, 8 and 4: 529 communities of 2,500 humans 127.4,
// 108.0, 97.3, 92.3, 1,024 of 1,000 humans 77.3, 67.4, 62.5, 59.8, 2,500 89.4,
// 81.1, 77.3, 77.0, 4,096 102.6, 93.9, 90.7, 92.5, 10,000 177.7, 171.9, 170.4,
// 177.8, 25,600 439.2, 437.9, 442.5, 459.1; rates 0.15 and no epidemic: 1,024
// 33.0, 32.5, 33.1, 32.3, 2,500 38.0, 38.1, 37.7, 38.5, 4,096 42.2, 41.5, 41.8,
// 43.4, 10,000 62.9, 63.5, 64.2, 68.1, 25,600 121.7, 124.1, 127.2, 134.5.
constexpr uint32_t kCountComms = 32;
constexpr uint32_t kCountBlocks = 320;
constexpr uint32_t kAoiBlock = 256;       // communities whose age-of-infection records are summed together
constexpr uint32_t kAoiWindow = 3650;     // rings record the days t with max_days - t <= this

// A workgroup of k_day_counts: n communities of one simulation from community
// c0, global index `first`, whose CSR rows are entries [row, row + rows); its
// sums go to record `total`.
struct CountBlock {
    uint32_t sim, c0, first, n, row, rows, total;
};

// Sums of a day over communities of one simulation, added by k_day_counts and
// read by the long-distance kernel: words (u64) 0-7 the long-distance rates in
// 2^-24 units (Poisson counts) or event counts (stochastic rounding), then as
// u32 humans, mosquitoes, infectious humans[4], onsets[4], census vectors read
// (humans, mosquitoes).  Integer atomics of different workgroups on one line
// follow each other 9 ns apart, so a simulation has a record per kTotalBlocks
// workgroups, up to kTotalRecords: with one, a quiet day of 480 x 480
// communities (7,200 workgroups) spent 63 of its 94 us in k_day_counts on them.
constexpr uint32_t kTotalWords = 16;
constexpr uint32_t kTotalBlocks = 64;
constexpr uint32_t kTotalRecords = 16;

struct CommDesc {
    uint64_t h_off;       // global offset of the first human
    uint64_t m_off;       // global offset of the first mosquito slot
    uint32_t sim;         // simulation index
    uint32_t c;           // community index within the simulation
    uint32_t n;           // humans
    uint32_t cap;         // mosquito slots
    uint32_t h_base;      // simulation-local index of the first human (Philox entity)
    uint32_t m_base;      // simulation-local index of the first slot (Philox entity)
    uint32_t row_off;     // global offset of the community's CSR row
    uint32_t row_len;
    uint32_t in_off;      // global offset of its in-edges
    uint32_t in_len;
    float base;           // m_ratio * n (f32)
    uint32_t flags;       // kCommIntro | kCommStay | self column << kCommSelfShift
};

constexpr uint32_t kCommIntro = 1u;      // the simulation has external introductions
constexpr uint32_t kCommStay = 2u;       // a fraction no_distance of the events stays at the source
constexpr uint32_t kCommSelfShift = 8u;  // bits 8..11: the source's own column on its CSR row

struct SimDesc {
    uint32_t k0, k1;              // Philox key = 64-bit seed
    uint32_t C, S;                // communities, serotypes
    uint32_t comm_off;            // global index of community 0
    float beta_hm, beta_mh, omega, recovery, eip, intro;
    uint32_t iip_min, iip_span;   // incubation uniform on [iip_min, iip_min + iip_span)
    uint32_t death_h_off;         // offsets into the shared table pools
    uint32_t death_h_guide_off;   // [kHumanGuide + 1] smallest death age of each slice of draws
    uint32_t death_m_off;
    uint32_t init_h_off;
    uint32_t init_m_off;
    uint32_t dens_off;
    uint32_t immune_off;          // [C*S] thresholds
    uint32_t seed_h, seed_m;
    uint32_t death_m_max;         // largest death age the mosquito table can return
    uint32_t death_m_guide_off;   // [256] smallest death age of each life_bucket() of draws
    uint32_t count_law;           // ARBO_COUNT_POISSON or ARBO_COUNT_STOCH_ROUND
    float no_distance;            // fraction of events staying at the source (communities with kCommStay)
    uint64_t series_off;          // this simulation's block in the series array
    uint64_t spatial_off;         // its block [(T+1)][S][C] of the per-community series (if kept)
    uint32_t total, totals;       // its records of the day's sums
    uint32_t aoi_block;           // its first block of kAoiBlock communities (age-of-infection rings)
    uint32_t aoi_blocks;
    uint32_t climate;             // 1: per-day beta/eip at clim_off and per-birth-day lifetime rows
    uint32_t clim_off;            // [max_days][3] beta_hm, beta_mh, eip in the dens pool
};

// Parameters of day t: the climate's or the constant ones.
struct DayParams {
    float beta_hm, beta_mh, eip;
};

__host__ __device__ inline DayParams day_params(const SimDesc& sd, const float* dens, uint32_t t) {
    if (!sd.climate) return DayParams{sd.beta_hm, sd.beta_mh, sd.eip};
    const float* d = dens + sd.clim_off + 3 * (size_t)t;
    return DayParams{d[0], d[1], d[2]};
}

// Lifetime row of mosquitoes born on day t (row 0: the t = 0 census).
__host__ __device__ inline uint32_t birth_row(const SimDesc& sd, uint32_t t) { return sd.climate ? t + 1 : 0u; }

// Series block of one simulation with room for T days (T+1 rows):
//   n_count[T+1] m_count[T+1] n_inf[(T+1)S] n_inc[(T+1)S] n_one[(T+1)S]
struct SeriesIdx {
    uint64_t n_count, m_count, n_inf, n_inc, n_one;
};

__host__ __device__ inline SeriesIdx series_index(uint64_t off, uint32_t T, uint32_t S) {
    SeriesIdx x;
    const uint64_t R = (uint64_t)T + 1;
    x.n_count = off;
    x.m_count = off + R;
    x.n_inf = off + 2 * R;
    x.n_inc = off + 2 * R + R * S;
    x.n_one = off + 2 * R + 2 * R * S;
    return x;
}

__host__ __device__ inline uint64_t series_words(uint32_t T, uint32_t S) {
    return ((uint64_t)T + 1) * (2 + 3 * (uint64_t)S);
}

struct EngineView {
    const CommDesc* comm;
    const SimDesc* sims;
    uint32_t* h_word;
    uint16_t* h_next;
    int32_t* h_birth;
    uint16_t* m_word;
    uint16_t* m_next;
    uint32_t* alive;               // [M/32] alive-slot bitmap of the current day
    uint32_t* cnt;                 // [G][9 in-edges][8 = dir*4 + serotype] local events arriving today
    uint32_t* nld;                 // [G][8] long-distance arrivals of the current day
    uint32_t* active;              // [G] 1 when events arrive today (set by the sources, cleared by the
                                   // destination's event kernel)
    uint32_t* hsum;                // [G][4] summary: earliest day any human has an event (0 = unknown),
                                   // infectious humans by serotype (two 16-bit pairs), mosquito scan
                                   // limit + 1 in 8-slot vectors (0 = unknown)
    unsigned long long* totals;    // [2 parity][n_totals][kTotalWords] sums of days of that parity
    uint32_t n_totals;
    uint32_t* series;
    uint32_t* part;                // [G][kPartWords] per-community partials of the day (see kPartWords)
    unsigned long long* scanned;   // [n_sims][2] census vectors read by the demography kernel (humans,
                                   // mosquitoes), summed over days
    uint32_t* spatial;             // per-community infectious humans [(T+1)][S][C] per simulation, or null
    int32_t* hist;                 // per human 4 infection-history words (one per serotype), or null
    uint8_t* aoi_mark;             // per human: 1 + ring when a mosquito event infected it today
                                   // (age-of-infection rings kept), else null
    uint32_t* aoi_cnt;             // [G][4] a community's infections of a day: day + 1, then the four
                                   // rings' counts as two 16-bit pairs (another day's: none today)
    uint32_t* aoi_sum;             // [2 parity][blocks][4] their sums over blocks of kAoiBlock communities
    uint32_t* aoi;                 // [n_sims][4][kAoiRecord] age-of-infection rings
    uint32_t* aoi_pos;             // [2 parity][n_sims][4] next position of each ring on days of that parity
    uint32_t aoi_nblocks;
    uint32_t aoi_from;             // first day whose infections enter the rings
    const uint32_t* csr_inbox;     // per CSR entry: inbox row (destination * 9 + in-edge index)
    const uint32_t* csr_thr;       // bits 0..24 threshold, 27..31 alias slot
    const uint32_t* in_edge;       // global source community
    const uint32_t* in_slot;       // slot of the destination in the source's row
    const uint32_t* tables;        // death / initial-age / immunity pools
    const float* dens;
    const uint32_t* day;           // device day counter (graph replay)
    uint32_t day_offset;           // the launch's day is *day + day_offset (a captured block of days
                                   // reads one counter, advanced once per block)
    uint32_t n_sims;
    uint32_t n_comm;
    uint32_t max_days;
    uint32_t death_m_lds;          // entries of the largest mosquito death table (LDS staging)
    const CountBlock* count_map;   // [count_blocks]
    uint32_t count_blocks;
    uint32_t small;                // 1: the event kernel also sums the day's series and draws the long-distance
                                   // events (kSmallCommunities), the demography kernel the local ones: no
                                   // k_day_counts and k_day_longdist
    uint32_t max_words;            // alive-bitmap words of the batch's largest community
};

// Batches whose event kernel sums the series and draws the long-distance
// events itself (EngineView.small), which spares the day two launches.  Every
// community's wave then reads its simulation's C partials and draws all its
// long-distance events, so all of these are bounded; us a day with it and
// without:
//  * C (the sums): one simulation of 484 communities of 200 and of 1,000
//    humans 32.0 and 32.6, 39.1 and 44.6; 529 33.2 and 33.5, 40.3 and 44.7; 676
//    35.5 and 34.2, 42.3 and 45.9; 1,024 40.8 and 34.9, 47.8 and 46.3;
//  * communities in all, whose waves have to run side by side for the repeated
//    work to cost only its latency: 28 simulations of 144 communities of 200 and
//    of 1,000 humans (4,032) 41.0 and 41.0, 62.8 and 63.5; 36 (5,184) 48.0 and
//    47.0, 74.5 and 75.2; 44 (6,336) 55.1 and 52.1, 89.6 and 86.8;
//  * the long-distance events: in proportion to omega, the transmission rates
//    and the mosquitoes, sent = omega x slots x (beta_hm + beta_mh), a wave's
//    share of them where a community has several, and times the waves per SIMD
//    that redraw them.  At rates of 0.7, 100 communities of 1,000 humans at
//    12,600 sent 47.4 and 53.7, 25,200 54.2 and 54.5, 42,000 62.8 and 54.8; 484
//    at 10,200 52.8 and 55.8, 18,300 57.3 and 56.3, 24,400 60.6 and 56.3; 16 x
//    144 at 6,800 71.5 and 73.2, 13,600 73.8 and 73.1, 27,200 78.5 and 73.0; at
//    0.15, without an epidemic, 22.0 and 28.5, 27.6 and 30.8, 33.4 and 36.2.  10
//    x 400 of 400 humans, the most sums that the limits admit, 68.3 and 63.3
//    at 2,600 sent, 34.8 and 33.1 without an epidemic.
constexpr uint32_t kSmallCommunities = 4096;
constexpr uint32_t kSmallSimulation = 512;
constexpr float kSmallSent = 24000.0f;
constexpr uint32_t kSimds = 1024;   // of the device: 256 CUs of four

// Launch knobs of the day kernels.  None of them changes a result: every
// random draw is keyed by model entities, never by workgroup or lane.
struct Tuning {
    uint32_t unroll;     // demography: 16-byte census loads in flight per lane
    uint32_t early_m;    // demography: of the first batch, mosquito loads issued before the humans
    uint32_t xcd;        // bit 0 demography, bit 1 events: the workgroups one XCD receives take a
                         // contiguous range of communities
    uint32_t ld_split;   // long-distance kernel: workgroups per simulation
    uint32_t wps;        // demography: 0 the compiler's register budget, 8 eight waves per SIMD
    uint32_t nw;         // demography: waves per community (1, 2, 4)
    bool chosen;         // nw was set, or found on a small batch; else a small batch's is left to the launch
};
constexpr uint32_t kDemographyShapes[][2] = {{4, 4}, {4, 2}, {8, 4}, {2, 2}};   // (unroll, early_m)
constexpr uint32_t kOccShapes[][2] = {{4, 2}, {2, 2}};   // shapes also built for 8 waves per SIMD
constexpr uint32_t kWideShapes[][3] = {{4, 2, 2}, {2, 2, 4}};   // (unroll, early_m, waves per community)
constexpr uint32_t kMaxLdSplit = 64;
constexpr uint32_t kXcds = 8;   // gfx950: workgroups go to the 8 XCDs in turn

// Community of workgroup b of n when the workgroups of XCD b % 8 take the
// contiguous range [x q + min(x, r), ...) of q + (x < r) communities, where
// n = 8 q + r.  A bijection of [0, n).
__host__ __device__ inline uint32_t xcd_block(uint32_t b, uint32_t n) {
    const uint32_t x = b % kXcds, i = b / kXcds, q = n / kXcds, r = n % kXcds;
    return x * q + (x < r ? x : r) + i;
}

// Lifetime tables to build in the pool: a human table of kHumanAgeTable
// thresholds and its guide, or the rows of one simulation's mosquitoes.
struct HumanTable {
    HumanLife life;
    uint32_t off, guide;
};
struct MosquitoTable {
    uint32_t off, guide;   // rows of dmax + 1 thresholds; [rows][256] guides
    uint32_t dmax, rows;
    float scale0, shape;   // row 0
    uint32_t scales, days; // rows 1..: the daily scales at `scales`, `days` of them
};

hipError_t launch_life_tables(uint32_t* pool, const HumanTable* humans, uint32_t n_humans,
                              const MosquitoTable* mosq, uint32_t n_mosq, uint32_t max_rows, const double* scales,
                              hipStream_t st);
hipError_t launch_init(const EngineView& v, uint32_t largest, hipStream_t st);
uint32_t demography_waves(const EngineView& v, const Tuning& tu);   // waves per community that it launches
hipError_t launch_demography(const EngineView& v, const Tuning& tu, hipStream_t st);
uint32_t event_waves(const EngineView& v);   // waves per community of the event kernel
hipError_t launch_events(const EngineView& v, const Tuning& tu, hipStream_t st);
hipError_t launch_longdist(const EngineView& v, const Tuning& tu, hipStream_t st);
hipError_t launch_advance(uint32_t* day, uint32_t n, hipStream_t st);
hipError_t launch_fill(uint32_t* p, uint64_t n, uint32_t value, hipStream_t st);
bool tuning_supported(const Tuning& tu);

}  // namespace arbo

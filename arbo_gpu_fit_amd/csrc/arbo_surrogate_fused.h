// arbo_surrogate_fused.h — the surrogate MLP's row-tile kernels on gfx950:
// k_mlp takes 16 rows through every layer of a pass (forward, and backward to
// the inputs or to the layers' dZ), k_wgrad turns the transposed dZ and layer
// inputs into weight gradients and, in training, applies Adam.
//
// What bounds them.  Rows are independent through the whole network, so one
// workgroup keeps its rows' activations in LDS and a pass is one launch; a
// product per launch costs 4.3 us of the stream for the launch alone, and took
// 17-20 us here: 64 x 64 tiles gave a 64-row pass four workgroups, each with a
// load latency per 64 k in series.  What is left is one workgroup's chain:
// it reads all the weights once per pass, 1.1 MB forward for the 6-256^4-260
// network, through six dependent stages of about 3 us each.  The reads alone
// are 7 us of the pass's 18.6 (a CU draws 64 B/clk out of L2, 52 with all of
// them reading), and the same loads hitting L1 end 5 us earlier; more of them
// in flight (32 to 256 KB a CU) measured the same.  Hence:
//  * the weights are kept a second time, split into bf16 halves (hi, lo) and
//    laid out in MFMA fragment order, once for the forward products and once
//    transposed for the backward ones: a lane's operand is one coalesced
//    16-byte load and needs no conversion;
//  * 16 rows a workgroup (v_mfma_f32_16x16x32_bf16), so 4,096 rows are 256
//    workgroups, one per CU; eight waves share the columns, two tiles each
//    (sixteen waves of one tile: 28 us for the pass's 20);
//  * the next 64 k of fragments (the next layer's first ones at a layer's
//    end) are in flight while the current ones multiply.
// A 64-row forward pass: 83 -> 18.5 us, 4,096 rows 95 -> 20.5, a training step
// of 512 rows (this pass there and back, then k_wgrad) 235 -> 56 us.
// The arithmetic is the bf16x3 split of k_gemm: hi*hi + hi*lo + lo*hi with
// float32 accumulation, biases, GELU and losses in float32.
#pragma once

namespace arbo {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kFuseRows = 16;       // rows of a workgroup
constexpr uint32_t kFuseWaves = 8;
constexpr uint32_t kFuseThreads = 64 * kFuseWaves;
constexpr uint32_t kFuseCols = 256;      // columns of a stage: two 16-column tiles a wave
constexpr uint32_t kFuseWidth = 512;     // widest layer: two stages
static_assert(kFuseThreads == 32 * kFuseRows && kFuseThreads >= kFuseWidth, "a thread per bias, 32 per row");
constexpr uint32_t kFrag = 64 * 8;       // elements of one fragment half: 16 columns x 32 k
constexpr uint32_t kGroup = 2;           // 32-k steps requested ahead
constexpr uint32_t kGroupK = 32 * kGroup;
constexpr uint32_t kNoFrag = 0xF0000000u;   // a byte offset past every buffer: loads return zeros, stores nothing

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Buffer resource over `bytes` bytes at p: a load at or past its end returns
// zeros, so the tiles and steps that a wave does not have need no branch
// (a branch around a load makes the compiler wait for it at the join).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00027000);
}
__device__ __forceinline__ bf16x8 load_frag(__amdgpu_buffer_rsrc_t r, uint32_t byte, uint32_t sbyte = 0) {
    return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, byte, sbyte, 0));
}

// float -> bf16 halves hi = bf16(x), lo = bf16(x - hi) (v_cvt_pk_bf16_f32, nearest even).
__device__ __forceinline__ void split_bf16(float x, uint16_t& hi, uint16_t& lo) {
    const __bf16 h = (__bf16)x;
    hi = __builtin_bit_cast(uint16_t, h);
    lo = __builtin_bit_cast(uint16_t, (__bf16)(x - (float)h));
}

// One product of a pass, up to kFuseCols columns of a layer: forward layers
// first to last, then backward ones.
struct Stage {
    uint32_t off;        // the layer's fragments in the packed weights (bytes)
    uint32_t K, N;       // reduction width and columns of the layer
    uint32_t steps;      // ceil(K / 32)
    uint32_t groups;     // ceil(steps / kGroup)
    uint32_t tiles;      // ceil(N / 16)
    uint32_t tile0;      // the stage's first column tile
    uint32_t buf;        // activation buffer it reads (its result goes to the other)
    uint32_t bias_at;    // forward: the layer's biases in LDS (floats behind the activations)
    uint32_t gg_at;      // gelu'(z) there [16][gg_row(N)]: written by a hidden layer, read going back; 0: none
    uint16_t* t;         // PASS_LOSS: the layer's input as k_wgrad's operand, written by its first stage
    uint32_t kind;       // STAGE_*
};

enum : uint32_t { STAGE_HIDDEN = 0, STAGE_OUTPUT = 1, STAGE_BACK = 2, STAGE_INPUT = 3 };
constexpr uint32_t kMaxStages = 4 * ARBO_SUR_MAX_LAYERS;   // every layer forward and back, two stages each

enum : uint32_t {
    PASS_FORWARD = 0,    // out = f(x)
    PASS_INPUT = 1,      // out = f(x), dx = (df / dx)^T dout
    PASS_LOSS = 2        // Poisson loss; layer inputs and dZ as operands of k_wgrad
};

struct Bias {
    const float* p;
    uint32_t at, n;
};

struct PassArgs {
    Stage st[kMaxStages];
    Bias bias[ARBO_SUR_MAX_LAYERS];   // of every layer, copied to LDS at the start
    uint32_t n, L, stages, w0;
    uint32_t ldk;            // LDS row of activations (bf16)
    uint32_t lds;            // LDS bytes of a workgroup
    uint32_t pack_bytes;
    const uint16_t* pack;
    const float* x;          // [*, w0]
    const uint32_t* rows;    // row r of the pass is row rows[r] of x and y, or null
    const float* y;          // targets (PASS_LOSS) or dout (PASS_INPUT) [*, w_L]
    float* out;              // [n, w_L] or null
    float* dx;               // PASS_INPUT [n, w0]
    uint16_t* tz;            // PASS_LOSS: dZ of the first layer as k_wgrad's operand
    uint32_t tzn;            // its columns
    float scale;             // PASS_LOSS: 1 / (rows * outputs)
    double* part;            // PASS_LOSS: loss sum of each workgroup
    double* acc;             // running loss sum, or null
};

// Floats of a row of gelu'(z) in LDS: 16-byte stores of 16 rows, 4 words apart
// mod 64, touch every bank once.
__host__ __device__ inline uint32_t gg_row(uint32_t N) { return ((N + 31u) & ~31u) + 4u; }

// Operands of k_wgrad, whose reduction runs over the rows: for 32 features and
// 16 rows (one workgroup of k_mlp) a 1 KB fragment of v_mfma_f32_32x32x16_bf16
// and its lo half behind it, [feature tile][16-row step][hi, lo][lane][8]: lane
// f % 32 + 32 (row / 8) holds rows row % 8 of feature f.  Written from the
// tile's activations in LDS: a thread gathers eight rows of a feature and
// stores 16 bytes.
__device__ __forceinline__ void store_operand(uint16_t* t, const uint16_t* act, uint32_t ldk, uint32_t N,
                                              uint32_t step, uint32_t steps, uint32_t tid) {
    const uint32_t plane = kFuseRows * ldk;
    for (uint32_t e = tid; e < 2 * ((N + 31u) & ~31u); e += kFuseThreads) {
        const uint32_t lane = e & 63u, f = (e >> 6) * 32u + (lane & 31u);
        if (f >= N) continue;
        const uint16_t* a = act + 8u * (lane >> 5) * ldk + f;
        typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
        u16x8 hi, lo;
#pragma unroll
        for (uint32_t r = 0; r < 8; ++r) {
            hi[r] = a[r * ldk];
            lo[r] = a[plane + r * ldk];
        }
        uint16_t* q = t + ((uint64_t)(e >> 6) * steps + step) * (2 * kFrag) + 8 * lane;
        *reinterpret_cast<u16x8*>(q) = hi;
        *reinterpret_cast<u16x8*>(q + kFrag) = lo;
    }
}

// The products are taken transposed (columns x rows: the weights are the first
// operand), so that a lane ends with four neighbouring columns of one row and
// LDS is written 8 or 16 bytes at a time.  Operands of
// v_mfma_f32_16x16x32_bf16: lane l holds A(l % 16, 8 (l / 16) + v) and
// B(8 (l / 16) + v, l % 16), v = 0..7; accumulator r of lane l is
// D(4 (l / 16) + r, l % 16).  Wave w has the stage's column tiles w and, with
// NT == 2, w + 8.
template <uint32_t MODE, uint32_t NT>
__global__ __launch_bounds__(kFuseThreads) void k_mlp(PassArgs g) {
    extern __shared__ __align__(16) uint16_t s_act[];   // [2 buffers][hi, lo][16 rows][ldk], biases, gelu'(z)
    __shared__ double s_loss[kFuseWaves];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t row0 = blockIdx.x * kFuseRows;
    const uint32_t left = g.n - row0 < kFuseRows ? g.n - row0 : kFuseRows;   // rows of this tile
    const uint32_t row = lane & 15u, c4 = 4u * (lane >> 4);   // the lane's row and its first column of a tile
    const uint32_t plane = kFuseRows * g.ldk;
    float* s_f = reinterpret_cast<float*>(s_act + 4 * plane);
    // hi and lo halves of the packed weights
    const __amdgpu_buffer_rsrc_t pk_hi = buffer_of(g.pack, g.pack_bytes), pk_lo = buffer_of(g.pack + kFrag, g.pack_bytes - 2 * kFrag);
    bf16x8 f[kGroup][NT][2];
    // Step u of group q of a stage, this wave's tiles, into slot u; vo: the
    // lane's offset, past the buffer for a tile the stage does not have.
    // Steps past the last repeat it: their activations are zeros.
    auto request = [&](uint32_t off, uint32_t steps, uint32_t tiles, uint32_t q, uint32_t u, const uint32_t (&vo)[NT]) {
        const uint32_t step = q * kGroup + u < steps ? q * kGroup + u : steps - 1;
        const uint32_t so = off + (step * tiles + wave) * (4 * kFrag);
#pragma unroll
        for (uint32_t i = 0; i < NT; ++i) {
            f[u][i][0] = load_frag(pk_hi, vo[i], so + i * kFuseWaves * (4 * kFrag));
            f[u][i][1] = load_frag(pk_lo, vo[i], so + i * kFuseWaves * (4 * kFrag));
        }
    };
    auto lanes_of = [&](uint32_t tile0, uint32_t tiles, uint32_t (&vo)[NT]) {
#pragma unroll
        for (uint32_t i = 0; i < NT; ++i) vo[i] = tile0 + wave + kFuseWaves * i < tiles ? 16 * lane : kNoFrag;
    };
    uint32_t vo[NT];
    lanes_of(g.st[0].tile0, g.st[0].tiles, vo);
#pragma unroll
    for (uint32_t u = 0; u < kGroup; ++u) request(g.st[0].off, g.st[0].steps, g.st[0].tiles, 0, u, vo);
    // the lane's row of x and y
    const uint64_t src = row < left ? (g.rows ? g.rows[row0 + row] : row0 + row) : 0u;
    {   // biases, and the rows' inputs, zero past the last row and column: 32 threads a row
        float b[ARBO_SUR_MAX_LAYERS];
#pragma unroll
        for (uint32_t l = 0; l < ARBO_SUR_MAX_LAYERS; ++l) b[l] = l < g.L && tid < g.bias[l].n ? g.bias[l].p[tid] : 0.0f;
        const uint32_t r = tid >> 5, kp = g.st[0].groups * kGroupK;
        const uint64_t xr = r < left ? (g.rows ? g.rows[row0 + r] : row0 + r) : 0u;
        // Eight loads of a row in flight where the inputs are many (one at a
        // time: 262,144 rows of 512-2-3 449 us for 252); columns past the last
        // read the first's, so that no branch waits for a load.
        const float* x = g.x + xr * g.w0;
#pragma unroll 4
        for (uint32_t c0 = tid & 31u; c0 < kp; c0 += 64) {   // kp is a multiple of 64
            float v[2];
#pragma unroll
            for (uint32_t u = 0; u < 2; ++u) v[u] = x[c0 + 32 * u < g.w0 ? c0 + 32 * u : 0u];
#pragma unroll
            for (uint32_t u = 0; u < 2; ++u) {
                const uint32_t c = c0 + 32 * u;
                uint16_t hi, lo;
                split_bf16(r < left && c < g.w0 ? v[u] : 0.0f, hi, lo);
                s_act[r * g.ldk + c] = hi;
                s_act[plane + r * g.ldk + c] = lo;
            }
        }
#pragma unroll
        for (uint32_t l = 0; l < ARBO_SUR_MAX_LAYERS; ++l)
            if (l < g.L && tid < g.bias[l].n) s_f[g.bias[l].at + tid] = b[l];
    }
    __syncthreads();
    double loss = 0.0;
    for (uint32_t st = 0; st < g.stages; ++st) {
        const Stage S = g.st[st];
        const bool more = st + 1 < g.stages;
        const Stage& next = g.st[more ? st + 1 : st];
        const uint32_t noff = next.off + next.tile0 * (4 * kFrag), nsteps = next.steps, ntiles = next.tiles;
        uint32_t no[NT];
        lanes_of(more ? next.tile0 : ntiles, ntiles, no);
        const uint16_t* in = s_act + S.buf * 2 * plane;
        uint16_t* outb = s_act + (S.buf ^ 1u) * 2 * plane;
        const uint16_t* a = in + row * g.ldk + 8 * (lane >> 4);
        if (MODE == PASS_LOSS && S.t) store_operand(S.t, in, g.ldk, S.K, blockIdx.x, gridDim.x, tid);
        f32x4 acc[NT] = {};
        // group q's products; each slot is refilled with the same step of group rq of the stage given
        auto multiply = [&](uint32_t q, uint32_t roff, uint32_t rsteps, uint32_t rtiles, uint32_t rq,
                            const uint32_t (&ro)[NT]) {
#pragma unroll
            for (uint32_t u = 0; u < kGroup; ++u) {
                const bf16x8 ah = *reinterpret_cast<const bf16x8*>(a + q * kGroupK + 32 * u);
                const bf16x8 al = *reinterpret_cast<const bf16x8*>(a + plane + q * kGroupK + 32 * u);
#pragma unroll
                for (uint32_t i = 0; i < NT; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[u][i][0], al, acc[i], 0, 0, 0);
#pragma unroll
                for (uint32_t i = 0; i < NT; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[u][i][1], ah, acc[i], 0, 0, 0);
#pragma unroll
                for (uint32_t i = 0; i < NT; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[u][i][0], ah, acc[i], 0, 0, 0);
                request(roff, rsteps, rtiles, rq, u, ro);
            }
        };
        for (uint32_t q = 0; q + 1 < S.groups; ++q)
            multiply(q, S.off + S.tile0 * (4 * kFrag), S.steps, S.tiles, q + 1, vo);
        // The last group requests the next stage's first.  The targets are
        // loaded ahead of those requests and without a branch, so that the
        // wait for them leaves the requests in flight.
        float side[NT][4] = {};
        if (MODE != PASS_FORWARD && S.kind == STAGE_OUTPUT) {
            if (MODE == PASS_INPUT && S.N % 4 == 0) {   // dout may be host memory: in segments, as `out` below
                const __amdgpu_buffer_rsrc_t y = buffer_of(g.y + (uint64_t)row0 * S.N, left * S.N * 4);
                f32x4 q[NT];
#pragma unroll
                for (uint32_t i = 0; i < NT; ++i) {
                    const uint32_t col = (S.tile0 + wave + kFuseWaves * i) * 16 + 4 * (lane & 3u);
                    q[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                         y, col < S.N ? ((lane >> 2) * S.N + col) * 4 : kNoFrag, 0, 0));
                }
#pragma unroll
                for (uint32_t i = 0; i < NT; ++i)
#pragma unroll
                    for (uint32_t r = 0; r < 4; ++r) side[i][r] = __shfl(q[i][r], 4 * (lane & 15u) + (lane >> 4), 64);
            } else {
#pragma unroll
                for (uint32_t i = 0; i < NT; ++i) {
                    const uint32_t col = (S.tile0 + wave + kFuseWaves * i) * 16 + c4;
#pragma unroll
                    for (uint32_t r = 0; r < 4; ++r)   // columns past the last read the first's
                        side[i][r] = g.y[src * S.N + (col + r < S.N ? col + r : 0u)];
                }
            }
        }
        multiply(S.groups - 1, noff, nsteps, ntiles, 0, no);
#pragma unroll
        for (uint32_t i = 0; i < NT; ++i) vo[i] = no[i];
        // results that leave the tile, through buffers that end with its
        // rows: columns past the last one store nothing, without a branch
        const bool back = S.kind == STAGE_INPUT;
        float* res_p = back ? g.dx : g.out;
        const __amdgpu_buffer_rsrc_t res =
            buffer_of(res_p ? res_p + (uint64_t)row0 * S.N : nullptr, res_p ? left * S.N * 4 : 0u);
#pragma unroll
        for (uint32_t i = 0; i < NT; ++i) {
            const uint32_t tile = S.tile0 + wave + kFuseWaves * i, col = tile * 16 + c4;
            if (tile >= ((S.N + 31u) >> 5) * 2) continue;   // wave-uniform: 32 columns at a time, the next k steps
            float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};           // what the next stage reads
            if (S.kind == STAGE_HIDDEN) {
                const f32x4 bias = *reinterpret_cast<const f32x4*>(s_f + S.bias_at + col);
                f32x4 gr;
#pragma unroll
                for (uint32_t r = 0; r < 4; ++r) {
                    const Gelu y = gelu_pair(acc[i][r] + bias[r]);
                    v[r] = y.h;
                    gr[r] = y.grad;
                }
                if (MODE != PASS_FORWARD) *reinterpret_cast<f32x4*>(s_f + S.gg_at + row * gg_row(S.N) + col) = gr;
            } else if (S.kind == STAGE_OUTPUT) {
                const f32x4 bias = *reinterpret_cast<const f32x4*>(s_f + S.bias_at + col);
                float z[4];
#pragma unroll
                for (uint32_t r = 0; r < 4; ++r) {
                    z[r] = acc[i][r] + bias[r];
                    v[r] = side[i][r];
                    if (MODE == PASS_LOSS) {
                        const float e = expf(z[r]);
                        if (col + r < S.N && row < left) loss += (double)e - (double)v[r] * (double)z[r];
                        v[r] = (e - v[r]) * g.scale;
                    }
                }
                // Four neighbouring lanes take a row's 64 bytes of the tile:
                // one write each, which matters where `out` is host memory.
                if (MODE != PASS_LOSS && S.N % 4 == 0) {
                    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
                    u32x4 q;
#pragma unroll
                    for (uint32_t r = 0; r < 4; ++r)
                        q[r] = (uint32_t)__shfl((int)__builtin_bit_cast(uint32_t, z[r]), 16 * (lane & 3u) + (lane >> 2), 64);
                    const uint32_t qc = tile * 16 + 4 * (lane & 3u);
                    __builtin_amdgcn_raw_buffer_store_b128(q, res, qc < S.N ? ((lane >> 2) * S.N + qc) * 4 : kNoFrag, 0, 0);
                } else if (MODE != PASS_LOSS) {
#pragma unroll
                    for (uint32_t r = 0; r < 4; ++r)
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, z[r]), res,
                                                              col + r < S.N ? (row * S.N + col + r) * 4 : kNoFrag, 0, 0);
                }
            } else if (S.kind == STAGE_BACK) {
                const f32x4 gr = *reinterpret_cast<const f32x4*>(s_f + S.gg_at + row * gg_row(S.N) + col);
#pragma unroll
                for (uint32_t r = 0; r < 4; ++r) v[r] = acc[i][r] * gr[r];
            } else {
#pragma unroll
                for (uint32_t r = 0; r < 4; ++r) {
                    const float dx = acc[i][r];
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, dx), res,
                                                          col + r < S.N ? (row * S.N + col + r) * 4 : kNoFrag, 0, 0);
                }
            }
            if (MODE == PASS_FORWARD && S.kind != STAGE_HIDDEN) continue;
            u16x4 hi, lo;
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) {
                uint16_t h, l;
                split_bf16(col + r < S.N && row < left ? v[r] : 0.0f, h, l);
                hi[r] = h;
                lo[r] = l;
            }
            *reinterpret_cast<u16x4*>(outb + row * g.ldk + col) = hi;
            *reinterpret_cast<u16x4*>(outb + plane + row * g.ldk + col) = lo;
        }
        // the next product's steps past this layer's columns are zeros
        if (S.tile0 == 0 && (MODE == PASS_FORWARD ? S.kind == STAGE_HIDDEN : S.kind != STAGE_INPUT)) {
            const uint32_t c0 = (S.N + 31u) & ~31u, kp = (S.N + kGroupK - 1) / kGroupK * kGroupK;
            uint16_t* z = outb + (tid >> 8) * plane + ((tid >> 4) & 15u) * g.ldk;
            for (uint32_t c = c0 + 8 * (tid & 15u); c < kp; c += 128)
                *reinterpret_cast<uint4*>(z + c) = make_uint4(0, 0, 0, 0);
        }
        __syncthreads();
    }
    if (MODE == PASS_LOSS) {
        store_operand(g.tz, s_act + (g.st[g.stages - 1].buf ^ 1u) * 2 * plane, g.ldk, g.tzn, blockIdx.x, gridDim.x, tid);
#pragma unroll
        for (uint32_t d = 32; d >= 1; d >>= 1) loss += __shfl_xor(loss, d, 64);
        if (lane == 0) s_loss[wave] = loss;
        __syncthreads();
        if (tid == 0) {
            double t = 0.0;
            for (uint32_t w = 0; w < kFuseWaves; ++w) t += s_loss[w];
            g.part[blockIdx.x] = t;
            if (g.acc) atomicAdd(g.acc, t);
        }
    }
}

// Where weight (n, k) of a layer sits in the packed arrays: the forward
// fragments (columns n, reduction k) and the backward ones (columns k,
// reduction n), each half 512 elements, lo behind hi.
__device__ __forceinline__ uint32_t frag_at(uint32_t off, uint32_t tiles, uint32_t red, uint32_t col) {
    return (off >> 1) + ((red >> 5) * tiles + (col >> 4)) * (2 * kFrag) + (((red >> 3) & 3u) * 16 + (col & 15u)) * 8 +
           (red & 7u);
}

// Both copies of the weights (n, k) and (n, k + 1), k even; past: k + 1 is no
// input (its place in the forward fragments is padding and stays zero).
__device__ __forceinline__ void pack_pair(uint16_t* pack, uint32_t foff, uint32_t ftiles, uint32_t boff,
                                          uint32_t btiles, uint32_t n, uint32_t k, float w0, float w1, bool past) {
    uint16_t h0, l0, h1, l1;
    split_bf16(w0, h0, l0);
    split_bf16(past ? 0.0f : w1, h1, l1);
    const uint32_t f = frag_at(foff, ftiles, k, n), b0 = frag_at(boff, btiles, n, k);
    *reinterpret_cast<uint32_t*>(pack + f) = pack2(h0, h1);
    *reinterpret_cast<uint32_t*>(pack + f + kFrag) = pack2(l0, l1);
    pack[b0] = h0;
    pack[b0 + kFrag] = l0;
    if (!past) {   // k and k + 1 are columns of one tile
        pack[b0 + 8] = h1;
        pack[b0 + 8 + kFrag] = l1;
    }
}

struct PackLayer {
    uint32_t first;            // of its pairs of weights (n, k), (n, k + 1) among all layers'
    uint32_t N, K;
    uint32_t foff, boff;       // in the packed weights (bytes)
    uint64_t w;                // weights in the parameter arrays
};

struct PackArgs {
    PackLayer l[ARBO_SUR_MAX_LAYERS];
    uint32_t L, pairs, n;      // pairs of weights, parameters (more of them: K weights and a bias a row)
    const float* P;
    float* M;
    float* V;
    uint16_t* pack;
};

// New parameters: their packed halves, and zero moments.  One launch for all
// layers: one each, and two for the moments, made a set_params of
// 6-256^4-260 94 us where it takes 74 (72 without packed weights), of
// 6-128^3-100 41 for 29 (30).
__global__ __launch_bounds__(256) void k_pack(PackArgs g) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= g.n) return;
    g.M[i] = 0.0f;
    g.V[i] = 0.0f;
    if (i >= g.pairs) return;
    uint32_t li = 0;
    while (li + 1 < g.L && i >= g.l[li + 1].first) ++li;
    const PackLayer& Y = g.l[li];
    const uint32_t pairs = (Y.K + 1) / 2, n = (i - Y.first) / pairs, k = 2 * ((i - Y.first) % pairs);   // N K <= 512^2
    const bool past = k + 1 >= Y.K;
    const float* W = g.P + Y.w + (uint64_t)n * Y.K + k;
    pack_pair(g.pack, Y.foff, (Y.N + 15) / 16, Y.boff, (Y.K + 15) / 16, n, k, W[0], past ? 0.0f : W[1], past);
}

struct GradLayer {
    uint32_t N, K;             // outputs, inputs
    uint32_t first, tx;        // its first workgroup and tiles along the inputs
    const uint16_t* dz;        // dZ and inputs as operands (store_operand)
    const uint16_t* h;
    uint64_t w, b;             // weights and biases in the parameter arrays
    uint32_t foff, boff;       // in the packed weights (bytes)
    uint32_t ftiles, btiles;
};

struct GradArgs {
    GradLayer l[ARBO_SUR_MAX_LAYERS];
    uint32_t L, steps;         // 16-row steps of the batch
    float* P;
    float* G;
    float* M;
    float* V;
    uint16_t* pack;
    float lr, c1, c2;
};

struct AdamState { float p, m, v; };

__device__ __forceinline__ float adam_update(const GradArgs& g, uint64_t at, const AdamState& o, float gi) {
    const float mi = 0.9f * o.m + 0.1f * gi;
    const float vi = 0.999f * o.v + 0.001f * gi * gi;
    g.M[at] = mi;
    g.V[at] = vi;
    const float p = o.p - g.lr * (mi / g.c1) / (sqrtf(vi / g.c2) + 1e-8f);
    g.P[at] = p;
    return p;
}

constexpr uint32_t kGradWaves = 8;

// [dW | db] = dZ^T [X | 1] of every layer in one launch, a 32 x 32 tile of dW
// a workgroup (272 tiles for 6-256^4-260, about one per CU).  The batch is the
// reduction: its 16-row steps are dealt to the eight waves in turn, so a
// minibatch of 512 is four steps a wave, all sixteen loads of them in flight
// at once, and the waves' partial tiles are added in LDS.  The bias gradient
// is the sum of the dZ operands the first tile column loads anyway.  ADAM:
// the update is applied here and the new weights' halves go to the packed
// arrays (each weight belongs to one thread); else the gradients are stored.
// With Adam 11 us of a step, about 4 each for the launch and the operands and
// 2 each for the update and the packed copies; the grouped products took 33.5
// and Adam's own launch 5.
template <bool ADAM>
__global__ __launch_bounds__(64 * kGradWaves) void k_wgrad(GradArgs g) {
    __shared__ float s_p[kGradWaves][32][33];
    __shared__ float s_b[kGradWaves][64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    uint32_t li = 0;
    while (li + 1 < g.L && blockIdx.x >= g.l[li + 1].first) ++li;
    const GradLayer& Y = g.l[li];
    const uint32_t b = blockIdx.x - Y.first, ti = b / Y.tx, tj = b % Y.tx, i0 = 32 * ti, j0 = 32 * tj;
    const uint32_t bytes = g.steps * (4 * kFrag);   // a feature tile's operands
    const __amdgpu_buffer_rsrc_t pa = buffer_of(Y.dz + (uint64_t)ti * (bytes >> 1), bytes);
    const __amdgpu_buffer_rsrc_t pb = buffer_of(Y.h + (uint64_t)tj * (bytes >> 1), bytes);
    // the thread's two weights of the tile, requested before the products
    const uint32_t row = tid >> 4, col = 2 * (tid & 15u), n = i0 + row, k = j0 + col;
    const uint64_t at = Y.w + (uint64_t)n * Y.K + k;
    const bool in[2] = {n < Y.N && k < Y.K, n < Y.N && k + 1 < Y.K};
    AdamState o[2] = {};
    if (ADAM) {
#pragma unroll
        for (uint32_t e = 0; e < 2; ++e)
            if (in[e]) o[e] = AdamState{g.P[at + e], g.M[at + e], g.V[at + e]};
    }
    f32x16 acc = {};
    float bsum = 0.0f;
    constexpr uint32_t U = 4;
    for (uint32_t s0 = wave; s0 < g.steps; s0 += U * kGradWaves) {
        bf16x8 ah[U], al[U], bh[U], bl[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {   // steps past the last read as zeros
            const uint32_t at0 = (s0 + u * kGradWaves) * (4 * kFrag) + 16 * lane;
            ah[u] = load_frag(pa, at0);
            al[u] = load_frag(pa, at0 + 2 * kFrag);
            bh[u] = load_frag(pb, at0);
            bl[u] = load_frag(pb, at0 + 2 * kFrag);
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[u], bh[u], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[u], bl[u], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[u], bh[u], acc, 0, 0, 0);
            if (j0 == 0) {
#pragma unroll
                for (uint32_t v = 0; v < 8; ++v) bsum += (float)ah[u][v] + (float)al[u][v];
            }
        }
    }
    // accumulator r of lane l is D(8 (r / 4) + 4 (l / 32) + r % 4, l % 32)
#pragma unroll
    for (uint32_t r = 0; r < 16; ++r) s_p[wave][8u * (r >> 2) + 4u * (lane >> 5) + (r & 3u)][lane & 31u] = acc[r];
    s_b[wave][lane] = bsum;
    __syncthreads();
    float gr[2] = {0.0f, 0.0f}, w2[2] = {0.0f, 0.0f};
#pragma unroll
    for (uint32_t e = 0; e < 2; ++e) {
        if (!in[e]) continue;
#pragma unroll
        for (uint32_t w = 0; w < kGradWaves; ++w) gr[e] += s_p[w][row][col + e];
        if (ADAM) w2[e] = adam_update(g, at + e, o[e], gr[e]);
        else g.G[at + e] = gr[e];
    }
    if (ADAM && in[0]) pack_pair(g.pack, Y.foff, Y.ftiles, Y.boff, Y.btiles, n, k, w2[0], w2[1], !in[1]);
    if (j0 == 0 && tid < 32 && i0 + tid < Y.N) {
        float gb = 0.0f;
#pragma unroll
        for (uint32_t w = 0; w < kGradWaves; ++w) gb += s_b[w][tid] + s_b[w][tid + 32];
        const uint64_t ab = Y.b + i0 + tid;
        if (ADAM) (void)adam_update(g, ab, AdamState{g.P[ab], g.M[ab], g.V[ab]}, gb);
        else g.G[ab] = gb;
    }
}

}  // namespace
}  // namespace arbo

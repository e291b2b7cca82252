// Single-query attention against an append-only K/V cache (the generation step).
//
// Replaces CudaCausalSelfAttention::attendCachedQuery (sentinel/NeuralNet/Cuda/CudaCausalSelfAttention.cu:318-341):
// there, per head, the cached K and V heads are copied out, a (length x 1) score GEMM, scale, mask, softmax and a
// (d x length)(length x 1) GEMM follow: 2 copies + 5 launches per head.  Here one launch reads the cache once:
// the cache stays in Sentinel's layout, fp32 [(head * d + dim), position] with `stride` positions per row
// (CudaKvCache, Cuda/CudaKvCache.hpp), which is position-contiguous, so lanes run along positions and every load is
// a coalesced row segment.  The work is bound by memory (2 * kv_heads * d * length * 4 bytes for O(length * d) FLOPs) and,
// for the contexts of one sequence, by latency: what counts is that a workgroup's loads are all in flight at once and that
// little code (instructions come from memory too when a kernel starts) and few dependent steps follow them.
// A workgroup takes 64 positions at a time of one K/V head for all query heads of its group, a wavefront 16 head dims.  Four and eight query
// heads per K/V head share the cache through the fp32 matrix instruction (v_mfma_f32_16x16x4_f32, heads padded to 16), which sums over
// positions without lane exchanges; one and two heads are cheaper in scalar multiply-adds.  The key axis is split over
// workgroups (flash-decoding), which leave unnormalised partials (reference, sum, acc[d]) in the workspace for a second small
// kernel; contexts of up to 64 positions per team of a workgroup take one workgroup per K/V head and no second launch.
// Exponentials are powers of two against a reference that is a whole number, 2^(s log2 e - n): changes of the reference, in a
// workgroup and in the merge, are then exact, and sums run in several short chains.  Error against float64 (relative 2-norm,
// geometric mean of 221 shapes from 16 to 32768 positions): 0.92 of the scalar kernel's this one replaced; chains through all positions of a
// workgroup and natural exponentials had 1.22 of it.
#include "cache_offsets.h"
#include "flash_common.h"
#include "mfma_tile.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

namespace sentinel_hip {

// Scratch of the entry point that allocates nothing (sentinel_hip_decode_attention_static): the partial
// (max, sum, acc[d]) records of decode_partial_kernel, in device memory that exists from the moment the code object is
// loaded.  Every device the library runs on holds its own copy of the array, at its own address, until the process
// ends.  In host code the array's name is only a handle for hipGetSymbolAddress: kernels get the address it returns.
static __device__ __align__(256) float decode_static_scratch[kDecodeStaticScratchBytes / sizeof(float)];

hipError_t decode_static_scratch_address(float** address) {
    constexpr int kMaxDevices = 64;
    static std::mutex mutex;
    static float* per_device[kMaxDevices] = {};
    int device = 0;
    hipError_t err = hipGetDevice(&device);
    if (err != hipSuccess) return err;
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mutex);
    if (!per_device[device]) {  // first call on this device, with it current: ask the runtime where its copy lives
        void* found = nullptr;
        err = hipGetSymbolAddress(&found, HIP_SYMBOL(decode_static_scratch));
        if (err != hipSuccess) return err;
        if (!found) return hipErrorInvalidSymbol;
        per_device[device] = static_cast<float*>(found);
    }
    *address = per_device[device];
    return hipSuccess;
}

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kChunk = 256;      // cache positions per workgroup and partial
constexpr int kSmallChunk = 64;  // ... for short caches, where 256 would leave most of the chip idle
constexpr int kSmallLength = 8192;
constexpr int kPassPositions = 64;
constexpr int kMostHeads = 8;   // query heads per K/V head
constexpr int kMostWaves = 8;   // of a team: one per 16 head dims
constexpr int kMostTeams = 4;
constexpr int kSingleWaves = 8;  // of the one workgroup of a short context
constexpr int kTeamsWaves = 16;  // of a workgroup of several teams

// Rows of one K/V head of a cache.  Normally through a buffer resource that ends with the head's last row: a load past the end gives
// zeros (cache_offsets.h).  WIDE: 64-bit addresses, positions past the used prefix repeat its last one.
template <bool WIDE>
struct CacheHead {
    __amdgpu_buffer_rsrc_t rsrc;
    const float* base;
    long long stride;
    int d, length, lane;
    __device__ __forceinline__ CacheHead(const float* cache, int kvh, int d_, long long stride_, int length_, int lane_)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(cache + (long long)kvh * d_ * stride_), 0,
                                                 WIDE ? 0 : (int)(unsigned)(d_ * stride_ * 4), 0x00020000)),
          base(cache + (long long)kvh * d_ * stride_), stride(stride_), d(d_), length(length_), lane(lane_) {}
    // as key_offset / value_offset
    __device__ __forceinline__ f32x4 key(int row0, int s, int p0) const {
        if (WIDE) return row0 + 4 * s < d ? wide(row0 + 4 * s + lane / 16, p0 + 4 * (lane % 16)) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        return narrow(key_offset(row0, s, p0, lane, d, (unsigned)stride));
    }
    __device__ __forceinline__ f32x4 value(int row0, int x, int p0) const {
        if (WIDE) return wide(min(row0 + lane % 16, d - 1), p0 + 16 * x + 4 * (lane / 16));
        return narrow(value_offset(row0, x, p0, lane, d, (unsigned)stride));
    }
    __device__ __forceinline__ f32x4 wide(int row, int position) const {
        const float* at = base + (long long)row * stride;
        f32x4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = at[min(position + i, length - 1)];
        return r;
    }
    __device__ __forceinline__ f32x4 narrow(CacheOffset at) const {
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(at.lane * 4u), (int)(at.scalar * 4u), 0));
    }
};

// The positions p0 .. p0 + 63 the query sees, one bit each
__device__ __forceinline__ unsigned long long visible_positions(int p0, int length, int global_tokens, int window_lo) {
    return low_bits(length - p0) & (low_bits(global_tokens - p0) | ~low_bits(window_lo - p0));
}
// A lane's values of V (positions 16 x + 4 g4 + e of the pass), zeros where the query does not see the position: those past the used prefix
// hold whatever was there before, and hidden ones may hold infinities, which a probability of zero would turn into NaN
struct VisibleValues {
    unsigned word[2];
    __device__ __forceinline__ VisibleValues(unsigned long long bits, int g4) {
        bits >>= 4 * g4;
        word[0] = (unsigned)bits;
        word[1] = (unsigned)(bits >> 32);
    }
    __device__ __forceinline__ float operator()(const f32x4 (&v)[4], int x, int e) const {
        const unsigned ones = (unsigned)__builtin_amdgcn_sbfe((int)word[x / 2], x % 2 * 16 + e, 1);
        return __builtin_bit_cast(float, __builtin_bit_cast(unsigned, (float)v[x][e]) & ones);
    }
};

// A workgroup owns a chunk of one K/V head: PASSES * 64 positions for each of its teams of a wavefront per 16 head dims (WAVES
// wavefronts at most).  In a pass
// wavefront w adds its dims' part of the scores, D[position][head] += K^T[position][4 dims] Q^T[4 dims][head] (lane l loads
// positions 4 (l % 16) .. + 3 of row l / 16: whole rows, one A operand each for four tiles of every fourth position), the parts
// meet in LDS, every wavefront derives the same softmax statistics, and forms acc[dim][head] += V[dim][4 positions] P[4
// positions][head] for its own 16 rows of V (lane l: positions 16 x + 4 (l / 16) .. + 3 of row l % 16).  The next pass's K is
// requested when this one's scores are done, its V when its products are; teams meet in LDS at the end.
// SINGLE: one workgroup sees the whole context and writes the result; otherwise a partial (reference of the scores, sum of
// exp, acc[d]) per query head goes to the workspace, numbered by workgroup.
template <int PASSES, int WAVES, bool SINGLE, bool WIDE>
__global__ __launch_bounds__(64 * WAVES, SINGLE || PASSES > 1 || WAVES > 8 ? 4 : 6) void decode_partial_kernel(
    const float* __restrict__ query, const float* __restrict__ key_cache, const float* __restrict__ value_cache,
    float* __restrict__ result, int kv_heads, int group, int d, long long stride, int length, float scale, int global_tokens,
    int window_lo, int global_chunks, int window_chunk) {
    constexpr bool TEAMS = SINGLE || WAVES > kMostWaves;
    __shared__ __attribute__((aligned(16))) float all_parts[WAVES][kMostHeads][kPassPositions];
    __shared__ __attribute__((aligned(16))) float all_scores[TEAMS ? kMostTeams : 1][kMostHeads][kPassPositions];
    const int waves = (d + 15) / 16;  // of a team
    const int teams = TEAMS ? blockDim.x / (64 * waves) : 1;
    const int team = TEAMS ? __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * waves)) : 0;
    const int tid = TEAMS ? threadIdx.x - team * 64 * waves : threadIdx.x;
    const int lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    auto& parts = *reinterpret_cast<float(*)[kMostWaves][kMostHeads][kPassPositions]>(all_parts[team * waves]);
    auto& scores = all_scores[team];
    const int m = lane & 15, g4 = lane >> 4;
    const int head = min(m, group - 1);  // (lanes of the padding heads repeat the last one and keep nothing)
    // Sparse mask of the layer (the query is position length - 1): visible are the global tokens [0, global_tokens)
    // and the window [window_lo, length).  Only chunks that hold a visible position are launched: the first
    // global_chunks ones and those from window_chunk on; partials are numbered by workgroup.
    const int slot = blockIdx.x;
    const int chunk = slot < global_chunks ? slot : slot - global_chunks + window_chunk;
    const int kvh = blockIdx.y;
    const int first = ((SINGLE ? 0 : chunk * teams) + team) * PASSES * kPassPositions;
    const int row0 = wave * 16;
    const CacheHead<WIDE> keys(key_cache, kvh, d, stride, length, lane);
    const CacheHead<WIDE> values(value_cache, kvh, d, stride, length, lane);

    const float c2 = scale * kLog2e;
    constexpr int kScoreChains = SINGLE ? 4 : 2, kChains = PASSES == 1 ? 8 : 4;

    // (head dims past the last are zeros in K and q alike; in V other rows stand in, whose rows of the result are not kept)
    f32x4 k[4], v[4];
    auto load_keys = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 4; ++s) k[s] = keys.key(row0, s, p0 < length ? p0 : 0);
    };
    auto load_values = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = values.value(row0, x, p0 < length ? p0 : 0);
    };
    load_keys(first);
    load_values(first);
    float q[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int c = row0 + 4 * s + g4;
        const float x = query[((long long)kvh * group + head) * d + min(c, d - 1)];
        q[s] = c < d ? x : 0.0f;
    }
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    float top = -__builtin_inff(), total = 0.0f;  // (total: this lane's share)
#pragma unroll 1
    for (int pass = 0; pass < PASSES; ++pass) {
        const int p0 = first + pass * kPassPositions;
        const bool more = pass + 1 < PASSES;
        f32x4 part[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32x4 sum[4];
#pragma unroll
            for (int c = 0; c < kScoreChains; ++c) sum[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < 4; ++s) sum[s % kScoreChains] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[s][j], q[s], sum[s % kScoreChains], 0, 0, 0);
            part[j] = kScoreChains == 4 ? (sum[0] + sum[1]) + (sum[2] + sum[3]) : sum[0] + sum[1];
        }
        __builtin_amdgcn_sched_barrier(0);  // (not earlier: into the same registers)
        if (more) load_keys(p0 + kPassPositions);
        // register i of tile j: position 16 g4 + 4 i + j
        if (m < group) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<f32x4*>(&parts[wave][m][16 * g4 + 4 * i]) = f32x4{part[0][i], part[1][i], part[2][i], part[3][i]};
        }
        __syncthreads();
        for (int idx = tid; idx < group * kPassPositions; idx += 64 * waves) {
            const int h = idx / kPassPositions, j = idx % kPassPositions;
            float dot = 0.0f;
            for (int w = 0; w < waves; ++w) dot += parts[w][h][j];
            scores[h][j] = visible_positions(p0, length, global_tokens, window_lo) >> j & 1 ? dot : -__builtin_inff();
        }
        __syncthreads();
        f32x4 p[4];
        float mx = -__builtin_inff();
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            p[x] = *reinterpret_cast<const f32x4*>(&scores[head][16 * x + 4 * g4]);
            mx = fmaxf(mx, fmaxf(fmaxf(p[x][0], p[x][1]), fmaxf(p[x][2], p[x][3])));
        }
        mx = fmaxf(top, __builtin_ceilf(column_max(mx) * c2));
        const float reference = mx == -__builtin_inff() ? 0.0f : mx;  // (no visible position so far; passes past the end add nothing)
        const float alpha = __builtin_amdgcn_exp2f(top - reference);
        total *= alpha;
        top = mx;
        f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int x = 0; x < 4; ++x) {
#pragma unroll
            for (int e = 0; e < 4; ++e) p[x][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(p[x][e], c2, -reference));
            sum[x] = (p[x][0] + p[x][1]) + (p[x][2] + p[x][3]);
        }
        total += (sum[0] + sum[1]) + (sum[2] + sum[3]);
        const VisibleValues seen(visible_positions(p0, length, global_tokens, window_lo), g4);
        // (one pass: always, in the shadow of the matrix instructions; several: where it matters, 3 % faster)
        if (PASSES > 1 && (p0 + kPassPositions > length || (p0 < window_lo && p0 + kPassPositions > global_tokens))) {
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[x][e] = seen(v, x, e);
        }
        f32x4 product[kChains];
#pragma unroll
        for (int c = 0; c < kChains; ++c) product[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 16; ++i) product[i % kChains] = __builtin_amdgcn_mfma_f32_16x16x4f32(PASSES > 1 ? v[i % 4][i / 4] : seen(v, i % 4, i / 4), p[i % 4][i / 4], product[i % kChains], 0, 0, 0);
#pragma unroll
        for (int half = kChains / 2; half; half /= 2)
#pragma unroll
            for (int c = 0; c < half; ++c) product[c] += product[c + half];
        acc = acc * alpha + product[0];
        __builtin_amdgcn_sched_barrier(0);
        if (more) load_values(p0 + kPassPositions);
    }
    total = column_sum(total);
    if (TEAMS && teams > 1) {  // the teams meet in LDS (nobody reads the score parts any more)
        __shared__ float stats[2][kMostTeams][16];
        f32x4* others = reinterpret_cast<f32x4*>(&all_parts[0][0][0]);
        if (g4 == 0 && wave == 0) {
            stats[0][team][m] = top;
            stats[1][team][m] = total;
        }
        if (team > 0) others[(team * waves + wave) * 64 + lane] = acc;
        __syncthreads();
        if (team > 0) return;
        const float own = top;
        for (int t = 1; t < teams; ++t) top = fmaxf(top, stats[0][t][m]);
        const float factor = __builtin_amdgcn_exp2f(own - top);
        total *= factor;
        acc *= factor;
        for (int t = 1; t < teams; ++t) {
            const float other = __builtin_amdgcn_exp2f(stats[0][t][m] - top);
            total += other * stats[1][t][m];
            acc += other * others[(t * waves + wave) * 64 + lane];
        }
    }
    if (m >= group) return;
    const int h = kvh * group + m;
    if (SINGLE) {
        const float inverse = 1.0f / total;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (row0 + 4 * g4 + i < d) result[(long long)h * d + row0 + 4 * g4 + i] = acc[i] * inverse;
    } else {
        float* record = result + ((long long)slot * kv_heads * group + h) * (d + 2);
        if (wave == 0 && g4 == 0) {
            record[0] = top;
            record[1] = total;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (row0 + 4 * g4 + i < d) record[2 + row0 + 4 * g4 + i] = acc[i];
    }
}

// One or two query heads per K/V head: their products are cheaper in scalar multiply-adds (16 + 16 per head, wavefront and pass) than on a
// matrix instruction of sixteen columns (32 of 32 cycles each).  Loads, passes and teams as in decode_partial_kernel, but after the parts of
// the scores have met in LDS every wavefront holds one position per lane (an exponential each instead of sixteen), and its sums over
// positions stay spread over the lanes until the end.  On the matrix instruction / here, us: 12 heads d64 1021 positions 5.9 / 5.1, 16000 22 / 20;
// 16 heads d64 20000 32 / 28; 12 query and 6 K/V heads d80 12000 17 / 14; 32 heads d128 4000 24.7 / 23.4; 8 and 4 heads d64 8000 8.6 / 7.9.
template <int HEADS, int PASSES, int WAVES, bool SINGLE, bool WIDE>
__global__ __launch_bounds__(64 * WAVES, 4) void decode_few_heads_kernel(
    const float* __restrict__ query, const float* __restrict__ key_cache, const float* __restrict__ value_cache,
    float* __restrict__ result, int kv_heads, int group, int d, long long stride, int length, float scale, int global_tokens,
    int window_lo, int global_chunks, int window_chunk) {
    constexpr bool TEAMS = SINGLE || WAVES > kMostWaves;
    __shared__ float all_parts[2][WAVES][HEADS][kPassPositions];  // (two buffers: one barrier per pass)
    __shared__ __attribute__((aligned(16))) float all_p[WAVES][HEADS][kPassPositions];  // a wavefront's own
    const int waves = (d + 15) / 16;  // of a team
    const int teams = TEAMS ? blockDim.x / (64 * waves) : 1;
    const int team = TEAMS ? __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * waves)) : 0;
    const int lane = threadIdx.x % 64;
    const int first_wave = team * waves;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64) - first_wave;
    const int m = lane & 15, g4 = lane >> 4;
    const int slot = blockIdx.x;
    const int chunk = slot < global_chunks ? slot : slot - global_chunks + window_chunk;
    const int kvh = blockIdx.y;
    const int first = ((SINGLE ? 0 : chunk * teams) + team) * PASSES * kPassPositions;
    const int row0 = wave * 16;
    const CacheHead<WIDE> keys(key_cache, kvh, d, stride, length, lane);
    const CacheHead<WIDE> values(value_cache, kvh, d, stride, length, lane);
    const float c2 = scale * kLog2e;

    f32x4 k[4], v[4];
    auto load_keys = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 4; ++s) k[s] = keys.key(row0, s, p0 < length ? p0 : 0);
    };
    auto load_values = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = values.value(row0, x, p0 < length ? p0 : 0);
    };
    load_keys(first);
    load_values(first);
    float q[HEADS][4];
#pragma unroll
    for (int h = 0; h < HEADS; ++h)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int c = row0 + 4 * s + g4;
            const float x = query[((long long)kvh * HEADS + h) * d + min(c, d - 1)];
            q[h][s] = c < d ? x : 0.0f;
        }
    float acc[HEADS], top[HEADS], total[HEADS];  // acc, total: this lane's share
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
        acc[h] = total[h] = 0.0f;
        top[h] = -__builtin_inff();
    }
#pragma unroll 1
    for (int pass = 0; pass < PASSES; ++pass) {
        const int p0 = first + pass * kPassPositions;
        const bool more = pass + 1 < PASSES;
        auto& parts = all_parts[pass & 1];
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            float part[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                part[e] = __builtin_fmaf(k[0][e], q[h][0], k[1][e] * q[h][1]) + __builtin_fmaf(k[2][e], q[h][2], k[3][e] * q[h][3]);
            // the sums over the four lanes of a column, one position in each of them
            swap_odd_even_rows(part[0], part[1]);
            swap_odd_even_rows(part[2], part[3]);
            float low = part[0] + part[1], high = part[2] + part[3];
            swap_halves(low, high);
            parts[first_wave + wave][h][4 * m + g4] = low + high;
        }
        __builtin_amdgcn_sched_barrier(0);  // (not earlier: into the same registers)
        if (more) load_keys(p0 + kPassPositions);
        __syncthreads();
        const VisibleValues seen(visible_positions(p0, length, global_tokens, window_lo), g4);
        if (PASSES > 1 && (p0 + kPassPositions > length || (p0 < window_lo && p0 + kPassPositions > global_tokens))) {
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[x][e] = seen(v, x, e);
        }
        float alpha[HEADS];
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            float dot = parts[first_wave][h][lane];
            for (int w = 1; w < waves; ++w) dot += parts[first_wave + w][h][lane];
            dot = visible_positions(p0, length, global_tokens, window_lo) >> lane & 1 ? dot : -__builtin_inff();
            const float mx = fmaxf(top[h], __builtin_ceilf(column_max(row_max(dot)) * c2));
            const float reference = mx == -__builtin_inff() ? 0.0f : mx;
            alpha[h] = __builtin_amdgcn_exp2f(top[h] - reference);
            top[h] = mx;
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(dot, c2, -reference));
            total[h] = total[h] * alpha[h] + p;
            all_p[first_wave + wave][h][lane] = p;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            float sum[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const f32x4 p = *reinterpret_cast<const f32x4*>(&all_p[first_wave + wave][h][16 * x + 4 * g4]);
                float u[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) u[e] = PASSES > 1 ? v[x][e] : seen(v, x, e);
                sum[x] = __builtin_fmaf(u[0], p[0], u[1] * p[1]) + __builtin_fmaf(u[2], p[2], u[3] * p[3]);
            }
            acc[h] = acc[h] * alpha[h] + ((sum[0] + sum[1]) + (sum[2] + sum[3]));
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (more) load_values(p0 + kPassPositions);
    }
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
        acc[h] = column_sum(acc[h]);
        total[h] = column_sum(row_sum(total[h]));
    }
    if (TEAMS && teams > 1) {  // the teams meet in LDS (nobody reads all_p or the stats' place any more)
        __shared__ float stats[kMostTeams][HEADS][2];
        float(*others)[HEADS][kPassPositions] = all_p;
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            if (team > 0 && g4 == 0) others[first_wave + wave][h][m] = acc[h];
            if (wave == 0 && lane == 0) {
                stats[team][h][0] = top[h];
                stats[team][h][1] = total[h];
            }
        }
        __syncthreads();
        if (team > 0) return;
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            const float own = top[h];
            for (int t = 1; t < teams; ++t) top[h] = fmaxf(top[h], stats[t][h][0]);
            const float factor = __builtin_amdgcn_exp2f(own - top[h]);
            total[h] *= factor;
            acc[h] *= factor;
            for (int t = 1; t < teams; ++t) {
                const float other = __builtin_amdgcn_exp2f(stats[t][h][0] - top[h]);
                total[h] += other * stats[t][h][1];
                acc[h] += other * others[t * waves + wave][h][m];
            }
        }
    }
    if (g4 > 0 || row0 + m >= d) return;
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
        const long long head = (long long)kvh * HEADS + h;
        if (SINGLE) {
            result[head * d + row0 + m] = acc[h] / total[h];
        } else {
            float* record = result + ((long long)slot * kv_heads * HEADS + head) * (d + 2);
            if (wave == 0 && m == 0) {
                record[0] = top[h];
                record[1] = total[h];
            }
            record[2 + row0 + m] = acc[h];
        }
    }
}

// out[h][c] = sum_chunks e^(m - M) acc[c] / sum_chunks e^(m - M) l.  One workgroup per (head, 32 head dims): 8 slices of the
// chunk list x 32 dims, each merged as it is read (one round of loads), the slices meet in LDS.
__global__ __launch_bounds__(256) void decode_merge_kernel(const float* __restrict__ partial, float* __restrict__ out,
                                                           int q_heads, int d, int chunks) {
    __shared__ float tops[8][32], denominators[8][32], sums[8][32];
    const int h = blockIdx.x;
    const int column = threadIdx.x % 32, slice = threadIdx.x / 32;
    const int c = min((int)blockIdx.y * 32 + column, d - 1);
    const long long step = (long long)q_heads * (d + 2);
    const float* base = partial + (long long)h * (d + 2);
    float top = -__builtin_inff(), denominator = 0.0f, sum = 0.0f;
    constexpr int kAhead = 4;
    for (int s0 = slice; s0 < chunks; s0 += 8 * kAhead) {
        float m[kAhead], l[kAhead], x[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int s = s0 + 8 * i;
            const float* record = base + min(s, chunks - 1) * step;
            m[i] = s < chunks ? record[0] : -__builtin_inff();
            l[i] = record[1];
            x[i] = record[2 + c];
        }
        float mx = top;
#pragma unroll
        for (int i = 0; i < kAhead; ++i) mx = fmaxf(mx, m[i]);
        const float alpha = __builtin_amdgcn_exp2f(top - mx);  // (a chunk's maximum is finite: one of its positions is visible)
        denominator *= alpha;
        sum *= alpha;
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const float factor = __builtin_amdgcn_exp2f(m[i] - mx);
            denominator += factor * l[i];
            sum += factor * x[i];
        }
        top = mx;
    }
    tops[slice][column] = top;
    denominators[slice][column] = denominator;
    sums[slice][column] = sum;
    __syncthreads();
    if (slice > 0 || (int)blockIdx.y * 32 + column >= d) return;
#pragma unroll
    for (int s = 1; s < 8; ++s) top = fmaxf(top, tops[s][column]);
    float l[8], x[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const float factor = __builtin_amdgcn_exp2f(tops[s][column] - top);
        l[s] = factor * denominators[s][column];
        x[s] = factor * sums[s][column];
    }
    denominator = ((l[0] + l[1]) + (l[2] + l[3])) + ((l[4] + l[5]) + (l[6] + l[7]));
    sum = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
    out[(long long)h * d + c] = sum / denominator;
}

}  // namespace

static int decode_chunk(int length) { return length <= kSmallLength ? kSmallChunk : kChunk; }

size_t decode_workspace_bytes(int q_heads, int head_dim, int length) {
    const int chunk = decode_chunk(length);
    const size_t chunks = (static_cast<size_t>(length) + chunk - 1) / chunk;
    return chunks * static_cast<size_t>(q_heads) * (head_dim + 2) * sizeof(float);
}

hipError_t launch_decode_attention(const float* query, const float* key_cache, const float* value_cache, float* out,
                                   int q_heads, int kv_heads, int head_dim, int stride, int length, float scale,
                                   int window, int global_tokens, float* workspace, hipStream_t stream) {
    const int group = q_heads / kv_heads;
    const int waves = (head_dim + 15) / 16;
    if (head_dim % 8 != 0 || waves > kMostWaves || group > kMostHeads) return hipErrorInvalidValue;
    const bool wide = (long long)head_dim * stride * 4 > 0xffffffffLL;
    // window <= 0 or >= length: every position is visible
    const bool sparse = window > 0 && window < length;
    const int window_lo = sparse ? length - window : 0;
    if (!sparse) global_tokens = 0;
    const auto launch = [&](auto kernel, dim3 grid, int teams, float* result, int globals, int first_chunk) {
        KernelTimer timer("decode_partial", stream);
        hipLaunchKernelGGL(kernel, grid, dim3(64 * waves * teams), 0, stream, query, key_cache, value_cache, result, kv_heads, group, head_dim,
                           (long long)stride, length, scale, global_tokens, window_lo, globals, first_chunk);
        return hipGetLastError();
    };
    // One launch while its workgroup has no more wavefronts than a split one's: 12 heads d64, 16 positions 3.9 us and 100
    // positions 4.7 us a call against 6.3 us with two launches; with sixteen wavefronts (256 positions) 6.5 us
    const int single_teams = (length + kPassPositions - 1) / kPassPositions;
    if (!wide && single_teams <= kMostTeams && single_teams * waves <= kSingleWaves) {
        const auto single = [&](auto kernel) { return launch(kernel, dim3(1, kv_heads), single_teams, out, 0, 0); };
        return group == 1   ? single(decode_few_heads_kernel<1, 1, kSingleWaves, true, false>)
               : group == 2 ? single(decode_few_heads_kernel<2, 1, kSingleWaves, true, false>)
                            : single(decode_partial_kernel<1, kSingleWaves, true, false>);
    }

    // Past 8192 positions a chunk is four passes of 64.  While a team has few wavefronts they go to four teams at once: one after the
    // other they are a chain of latencies that a few wavefronts per compute unit do not hide.  Four passes -> four teams, us: one head per
    // K/V head, 4 heads d16 9001 positions 7.3 -> 5.8, 8 heads d32 8.4 -> 7.7, 16 heads d64 17.3 -> 17.1 (more wavefronts than fit do not gain: 12 heads d64
    // 26000 28.1 -> 28.3); four heads, 8 / 2 d32 11.0 -> 7.9, 16 / 4 d64 20000 positions 15.7 -> 17.0.
    const bool several = length > kSmallLength && waves <= (group <= 2 ? 4 : 2);
    const int teams = several ? kMostTeams : 1;
    const int passes = decode_chunk(length) / kPassPositions / teams;
    const int chunk = teams * passes * kPassPositions;
    const int all_chunks = (length + chunk - 1) / chunk;
    const int global_chunks = sparse ? (std::min(global_tokens, window_lo) + chunk - 1) / chunk : 0;
    const int window_chunk = std::max(global_chunks, window_lo / chunk);
    const int chunks = global_chunks + (all_chunks - window_chunk);
    const auto split = [&](auto kernel) { return launch(kernel, dim3(chunks, kv_heads), teams, workspace, global_chunks, window_chunk); };
    // (std::integral_constants)
    const auto with_width = [&](auto passes_tag, auto waves_tag, auto wide_tag) {
        constexpr int PASSES = decltype(passes_tag)::value, WAVES = decltype(waves_tag)::value;
        constexpr bool WIDE = decltype(wide_tag)::value;
        return group == 1   ? split(decode_few_heads_kernel<1, PASSES, WAVES, false, WIDE>)
               : group == 2 ? split(decode_few_heads_kernel<2, PASSES, WAVES, false, WIDE>)
                            : split(decode_partial_kernel<PASSES, WAVES, false, WIDE>);
    };
    const auto with_waves = [&](auto passes_tag, auto waves_tag) {
        return wide ? with_width(passes_tag, waves_tag, std::true_type{}) : with_width(passes_tag, waves_tag, std::false_type{});
    };
    constexpr std::integral_constant<int, kMostWaves> one_team;
    constexpr std::integral_constant<int, kTeamsWaves> many_teams;
    constexpr std::integral_constant<int, 1> one_pass;
    constexpr std::integral_constant<int, kChunk / kPassPositions> all_passes;
    static_assert(kSmallChunk == kPassPositions && kChunk == kMostTeams * kPassPositions, "a chunk is one pass, or one per team");
    const hipError_t err = several ? with_waves(one_pass, many_teams) : passes == 1 ? with_waves(one_pass, one_team) : with_waves(all_passes, one_team);
    if (err != hipSuccess) return err;
    KernelTimer timer("decode_merge", stream);
    hipLaunchKernelGGL(decode_merge_kernel, dim3(q_heads, (head_dim + 31) / 32), dim3(256), 0, stream, workspace, out, q_heads,
                       head_dim, chunks);
    return hipGetLastError();
}

}  // namespace sentinel_hip

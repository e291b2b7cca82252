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
// A workgroup takes 64 positions of one K/V head for all query heads of its group.  Both products run on the fp32 matrix
// instruction (v_mfma_f32_16x16x4_f32, heads padded to 16): it sums over positions without lane exchanges and costs
// the same for every group; even one head in sixteen leaves it three times as fast as memory delivers.  The key axis is split over
// workgroups (flash-decoding), which leave unnormalised partials (max, sum, acc[d]) in the workspace for a second small
// kernel; contexts of up to 64 positions per team of a workgroup take one workgroup per K/V head and no second launch.
#include "cache_offsets.h"
#include "flash_common.h"
#include "mfma_tile.h"

#include <algorithm>
#include <mutex>

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

constexpr int kChunk = 256;      // cache positions per workgroup
constexpr int kSmallChunk = 64;  // ... for short caches, where 256 would leave most of the chip idle
constexpr int kSmallLength = 8192;
constexpr int kPassPositions = 64;
constexpr int kMostHeads = 8;   // query heads per K/V head
constexpr int kMostWaves = 8;   // one per 16 head dims
constexpr int kSingleTeams = 4;  // teams of such wavefronts in the one workgroup of a short context
constexpr int kSingleWaves = 8;

// sum / maximum over the four lanes that share a column of a 16 x 16 result: lanes l, l ^ 16, l ^ 32, l ^ 48
__device__ __forceinline__ void row_exchange(float x, float& even, float& odd) {
    even = x;
    odd = x;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(even), "+v"(odd));
}
__device__ __forceinline__ float column_sum(float x) {
    float even, odd;
    row_exchange(x, even, odd);
    return half_sum(even + odd);
}
__device__ __forceinline__ float column_max(float x) {
    float even, odd;
    row_exchange(x, even, odd);
    return half_max(fmaxf(even, odd));
}

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

// A workgroup owns `passes` * 64 positions of one K/V head (a chunk) and has a wavefront per 16 head dims.  In a pass
// wavefront w adds its dims' part of the scores, D[position][head] += K^T[position][4 dims] Q^T[4 dims][head] (lane l loads
// positions 4 (l % 16) .. + 3 of row l / 16: whole rows, one A operand each for four tiles of every fourth position), the parts
// meet in LDS, every wavefront derives the same softmax statistics, and forms acc[dim][head] += V[dim][4 positions] P[4
// positions][head] for its own 16 rows of V (lane l: positions 16 x + 4 (l / 16) .. + 3 of row l % 16).  The next pass's K is
// requested when this one's scores are done, its V when its products are.
// SINGLE: one workgroup sees the whole context, 64 positions per team of wavefronts, and writes the result; otherwise a partial (max of the scaled scores, sum of
// exp, acc[d]) per query head goes to the workspace, numbered by workgroup.
template <int PASSES, bool SINGLE, bool WIDE>
__global__ __launch_bounds__(64 * (SINGLE ? kSingleWaves : kMostWaves), SINGLE || PASSES > 1 ? 4 : 6) void decode_partial_kernel(const float* __restrict__ query, const float* __restrict__ key_cache,
                                                                            const float* __restrict__ value_cache, float* __restrict__ result,
                                                                            int kv_heads, int group, int d, long long stride,
                                                                            int length, float scale, int global_tokens,
                                                                            int window_lo, int global_chunks, int window_chunk) {
    __shared__ __attribute__((aligned(16))) float all_parts[SINGLE ? kSingleWaves : kMostWaves][kMostHeads][kPassPositions];
    __shared__ __attribute__((aligned(16))) float all_scores[SINGLE ? kSingleTeams : 1][kMostHeads][kPassPositions];
    const int waves = (d + 15) / 16;  // of a team
    const int team = SINGLE ? __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * waves)) : 0;
    const int tid = SINGLE ? threadIdx.x - team * 64 * waves : threadIdx.x;
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
    const int first = (SINGLE ? team : chunk * PASSES) * kPassPositions;
    const int row0 = wave * 16;
    const CacheHead<WIDE> keys(key_cache, kvh, d, stride, length, lane);
    const CacheHead<WIDE> values(value_cache, kvh, d, stride, length, lane);

    const auto visible = [&](int position) { return position < length && (position < global_tokens || position >= window_lo); };

    // (head dims past the last are zeros in K and q alike; in V other rows stand in, whose rows of the result are not kept)
    f32x4 k[4], v[4];
    auto load_keys = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 4; ++s) k[s] = keys.key(row0, s, p0);
    };
    auto load_values = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = values.value(row0, x, p0);
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
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
        const int p0 = first + pass * kPassPositions;
        const bool more = pass + 1 < PASSES;
        const int next = p0 + kPassPositions < length ? p0 + kPassPositions : p0;  // (past the end: loaded again, not used)
        f32x4 part[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) part[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = 0; j < 4; ++j) part[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[s][j], q[s], part[j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);  // (not earlier: into the same registers)
        if (more) load_keys(next);
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
            scores[h][j] = visible(p0 + j) ? dot * scale : -__builtin_inff();
        }
        __syncthreads();
        f32x4 p[4];
        float mx = top;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            p[x] = *reinterpret_cast<const f32x4*>(&scores[head][16 * x + 4 * g4]);
            mx = fmaxf(mx, fmaxf(fmaxf(p[x][0], p[x][1]), fmaxf(p[x][2], p[x][3])));
        }
        mx = column_max(mx);
        const float reference = mx == -__builtin_inff() ? 0.0f : mx;  // (no visible position so far; passes past the end add nothing)
        const float alpha = __expf(top - reference);
        total *= alpha;
        acc *= alpha;
        top = mx;
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                p[x][e] = __expf(p[x][e] - reference);
                total += p[x][e];
            }
        // positions past the used prefix hold whatever was there before, and hidden ones may hold infinities
        if (p0 + kPassPositions > length || (p0 < window_lo && p0 + kPassPositions > global_tokens)) {
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (!visible(p0 + 16 * x + 4 * g4 + e)) v[x][e] = 0.0f;
        }
        f32x4 odd = {0.0f, 0.0f, 0.0f, 0.0f};  // (two chains: neither waits for its predecessor)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int x = 0; x < 4; x += 2) {
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(v[x][e], p[x][e], acc, 0, 0, 0);
                odd = __builtin_amdgcn_mfma_f32_16x16x4f32(v[x + 1][e], p[x + 1][e], odd, 0, 0, 0);
            }
        acc += odd;
        __builtin_amdgcn_sched_barrier(0);
        if (more) load_values(next);
    }
    total = column_sum(total);
    if (SINGLE && blockDim.x > 64 * waves) {  // the teams meet in LDS (nobody reads the score parts any more)
        __shared__ float stats[2][kSingleTeams][16];
        f32x4* others = reinterpret_cast<f32x4*>(&all_parts[0][0][0]);
        if (g4 == 0 && wave == 0) {
            stats[0][team][m] = top;
            stats[1][team][m] = total;
        }
        if (team > 0) others[(team * waves + wave) * 64 + lane] = acc;
        __syncthreads();
        if (team > 0) return;
        const int teams = blockDim.x / (64 * waves);
        const float own = top;
        for (int t = 1; t < teams; ++t) top = fmaxf(top, stats[0][t][m]);
        const float factor = __expf(own - top);
        total *= factor;
        acc *= factor;
        for (int t = 1; t < teams; ++t) {
            const float other = __expf(stats[0][t][m] - top);
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
        const float alpha = __expf(top - mx);  // (a chunk's maximum is finite: one of its positions is visible)
        denominator *= alpha;
        sum *= alpha;
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const float factor = __expf(m[i] - mx);
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
    denominator = 0.0f;
    sum = 0.0f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const float factor = __expf(tops[s][column] - top);
        denominator += factor * denominators[s][column];
        sum += factor * sums[s][column];
    }
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
    const int chunk = decode_chunk(length);
    const int all_chunks = (length + chunk - 1) / chunk;
    // window <= 0 or >= length: every position is visible
    const bool sparse = window > 0 && window < length;
    const int window_lo = sparse ? length - window : 0;
    if (!sparse) global_tokens = 0;
    const int global_chunks = sparse ? (std::min(global_tokens, window_lo) + chunk - 1) / chunk : 0;
    const int window_chunk = std::max(global_chunks, window_lo / chunk);
    const int chunks = global_chunks + (all_chunks - window_chunk);
    const int group = q_heads / kv_heads;
    const int waves = (head_dim + 15) / 16;
    if (head_dim % 8 != 0 || waves > kMostWaves || group > kMostHeads) return hipErrorInvalidValue;
    const bool wide = (long long)head_dim * stride * 4 > 0xffffffffLL;
    const auto launch = [&](auto kernel, dim3 grid, int teams, float* result, int globals, int first_chunk) {
        KernelTimer timer("decode_partial", stream);
        hipLaunchKernelGGL(kernel, grid, dim3(64 * waves * teams), 0, stream, query, key_cache, value_cache, result, kv_heads, group, head_dim,
                           (long long)stride, length, scale, global_tokens, window_lo, globals, first_chunk);
        return hipGetLastError();
    };
    // One launch while its workgroup has no more wavefronts than a split one's: 12 heads d64, 16 positions 3.9 us and 100
    // positions 4.7 us a call against 6.3 us with two launches; with sixteen wavefronts (256 positions) 6.5 us
    const int teams = (length + kPassPositions - 1) / kPassPositions;
    if (!wide && teams <= kSingleTeams && teams * waves <= kSingleWaves)
        return launch(decode_partial_kernel<1, true, false>, dim3(1, kv_heads), teams, out, 0, 0);
    const auto split = [&](auto kernel) { return launch(kernel, dim3(chunks, kv_heads), 1, workspace, global_chunks, window_chunk); };
    constexpr int kPasses = kChunk / kPassPositions;
    static_assert(kSmallChunk == kPassPositions, "a short cache's chunk is one pass");
    const hipError_t err = chunk == kSmallChunk ? (wide ? split(decode_partial_kernel<1, false, true>) : split(decode_partial_kernel<1, false, false>))
                                                : (wide ? split(decode_partial_kernel<kPasses, false, true>) : split(decode_partial_kernel<kPasses, false, false>));
    if (err != hipSuccess) return err;
    KernelTimer timer("decode_merge", stream);
    hipLaunchKernelGGL(decode_merge_kernel, dim3(q_heads, (head_dim + 31) / 32), dim3(256), 0, stream, workspace, out, q_heads,
                       head_dim, chunks);
    return hipGetLastError();
}

}  // namespace sentinel_hip

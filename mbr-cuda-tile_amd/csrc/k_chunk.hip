// Chunk overlap-add of the chunked inference driver (src/chunk_cuda_tile.cu:18-83,
// src/inference_app.cpp:72-232): each model output chunk is weighted by its fade window and
// added into the song-length output at its offset, the window itself into a weight sum;
// at the end the output is divided by the weight sum where that exceeds 1e-8.
//
// The reference adds with float atomics.  Within one call every (channel, sample) is
// written once, and calls on one stream run in order, so plain read-modify-write gives the
// same sums in a fixed order: the result is deterministic and equals an ordered f32
// accumulation bit for bit (the product src * w and the sum are rounded separately, as the
// reference's atomic add of a rounded product is).
//
// Memory-bound: per call C*n reads of src, C*n read-modify-writes of dest, n of the window
// and n read-modify-writes of the weight sum.  A thread owns four sample positions
// (of one channel, or of all channels for the normalize).  16-byte accesses also off 16-byte
// addresses, where a song of odd length puts its second channel and a chunk at an odd offset all
// of its rows, when there is much to move (MBRT_CHUNK_ANY, MBRT_NORM_ANY).
#include "abi_common.hpp"

namespace mbrt {
namespace {

// 4 floats at any float address through the vector helpers
struct F4 {
    float v[4];
};
template <int NT>
__device__ __forceinline__ F4 ld4(const float* p) {
    return __builtin_bit_cast(F4, ld_any<NT, 4>(p));
}
template <int NT>
__device__ __forceinline__ void st4(float* p, const F4& x) {
    st_any<NT, 4>(p, __builtin_bit_cast(u32x4, x));
}

constexpr int kThreads = 256;
static_assert(MBRT_CHUNK_CPB >= 1 && MBRT_CHUNK_CPB <= 16, "one wave per channel, 1 to 16 of them in a block");

struct AccArgs {
    float* __restrict__ dest;       // [C, dest_len]
    float* __restrict__ wsum;       // [dest_len]
    const float* __restrict__ src;  // [C, n]
    const float* __restrict__ win;  // [n]
    int64_t n;            // chunk length
    int64_t dest_len;
    int64_t offset;
    int64_t channels;
    uint32_t vblocks;     // blocks over whole vectors; one more takes the n % 4 samples left
};

// d + s w with the product rounded before the add (no contraction into an FMA).
__device__ __forceinline__ float acc1(float d, float s, float w) {
#pragma clang fp contract(off)
    return d + s * w;
}

__device__ __forceinline__ void accumulate1(const AccArgs& a, int64_t c, int64_t k, bool wsum) {
    const float w = a.win[k];
    float* d = a.dest + c * a.dest_len + a.offset + k;
    *d = acc1(*d, a.src[c * a.n + k], w);
    if (wsum) a.wsum[a.offset + k] = a.wsum[a.offset + k] + w;
}

// One sample per lane, a channel per grid row: unaligned chunks of few samples, where a
// quarter of the waves with wider accesses take longer.
__global__ __launch_bounds__(kThreads) void accumulate_scalar_kernel(AccArgs a) {
    for (int64_t k = (int64_t)blockIdx.x * kThreads + threadIdx.x; k < a.n; k += (int64_t)gridDim.x * kThreads)
        accumulate1(a, blockIdx.y, k, blockIdx.y == 0);
}

// One wave per channel: a block of CPB waves takes channels [CPB y, CPB y + CPB) over the
// same 64 consecutive 4-sample positions of the chunk, so the window's repeated reads are
// made by waves of one CU, close together in time.  Dest, weight sum and window addresses are
// only sample-aligned where a song's length or a chunk's offset is odd, and 16-byte accesses
// take that (ld_any).  The samples after the last whole vector go to a block of their own: in
// the vectors' loop one lane's three read-modify-writes held its wave for two more round trips.
template <int CPB>
__global__ __launch_bounds__(64 * CPB) void accumulate_cw_kernel(AccArgs a) {
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
    const int64_t c = (int64_t)blockIdx.y * CPB + w;
    const bool wsum = blockIdx.y == 0 && w == 0;
    if (c >= a.channels) return;
    if (blockIdx.x >= a.vblocks) {
        const int64_t k = (a.n & ~int64_t(3)) + lane;
        if (k < a.n) accumulate1(a, c, k, wsum);
        return;
    }
    for (int64_t k = 4 * ((int64_t)blockIdx.x * 64 + lane); k + 4 <= a.n; k += 4 * (int64_t)a.vblocks * 64) {
        float* dp = a.dest + c * a.dest_len + a.offset + k;
        const F4 wv = ld4<0>(a.win + k);
        const F4 s = ld4<MBRT_NT_CHUNK & 1>(a.src + c * a.n + k);
        F4 d = ld4<MBRT_NT_CHUNK & 1>(dp);
        __builtin_amdgcn_sched_barrier(0);  // all three loads out before the first is waited for
#pragma unroll
        for (int e = 0; e < 4; ++e) d.v[e] = acc1(d.v[e], s.v[e], wv.v[e]);
        st4<MBRT_NT_CHUNK & 2>(dp, d);
        if (wsum) {
            float* wp = a.wsum + a.offset + k;
            F4 ws = ld4<0>(wp);
#pragma unroll
            for (int e = 0; e < 4; ++e) ws.v[e] = ws.v[e] + wv.v[e];
            st4<0>(wp, ws);
        }
    }
}

struct NormArgs {
    float* __restrict__ data;        // [C, len]
    const float* __restrict__ wsum;  // [len]
    int64_t len;
    int64_t channels;
    uint32_t vblocks;     // blocks over whole vectors; one more takes the len % 4 samples left
};

__device__ __forceinline__ float norm1(float v, float w) { return w > 1.0e-8f ? v / w : v; }

// One sample position per thread, walked over the channels.
__global__ __launch_bounds__(kThreads) void normalize_scalar_kernel(NormArgs a) {
    for (int64_t k = (int64_t)blockIdx.x * kThreads + threadIdx.x; k < a.len; k += (int64_t)gridDim.x * kThreads) {
        const float w = a.wsum[k];
        for (int64_t c = 0; c < a.channels; ++c) a.data[c * a.len + k] = norm1(a.data[c * a.len + k], w);
    }
}

// A thread owns 4 sample positions and walks the channels, whose rows are only sample-aligned
// where the length is not a multiple of 4.  The samples after the last whole vector go to a block
// of their own, one (channel, sample) per thread: walked by one lane they took half of [16, 999].
__global__ __launch_bounds__(kThreads) void normalize_vec_kernel(NormArgs a) {
    if (blockIdx.x >= a.vblocks) {
        const int64_t k0 = a.len & ~int64_t(3), tail = a.len - k0;
        for (int64_t i = threadIdx.x; i < tail * a.channels; i += kThreads) {
            const int64_t c = i / tail, k = k0 + i % tail;
            a.data[c * a.len + k] = norm1(a.data[c * a.len + k], a.wsum[k]);
        }
        return;
    }
    for (int64_t k = 4 * ((int64_t)blockIdx.x * kThreads + threadIdx.x); k + 4 <= a.len;
         k += 4 * (int64_t)a.vblocks * kThreads) {
        const F4 w = ld4<0>(a.wsum + k);
#pragma unroll 4
        for (int64_t c = 0; c < a.channels; ++c) {
            float* p = a.data + c * a.len + k;
            F4 v = ld4<MBRT_NT_CHUNK & 1>(p);
#pragma unroll
            for (int e = 0; e < 4; ++e) v.v[e] = norm1(v.v[e], w.v[e]);
            st4<MBRT_NT_CHUNK & 2>(p, v);
        }
    }
}

int64_t grid_for(int64_t work) { return std::min<int64_t>(ceil_div(work, kThreads), int64_t(1) << 14); }

}  // namespace
}  // namespace mbrt

using namespace mbrt;

extern "C" {

int mbrt_chunk_accumulate(float* dest, float* weight_sum, const float* src, const float* window, int64_t channels,
                          int64_t chunk_len, int64_t dest_len, int64_t offset, mbrt_stream_t stream) {
    const char* op = "mbrt_chunk_accumulate";
    MBRT_REQUIRE(channels >= 0 && chunk_len >= 0 && dest_len >= 0, MBRT_E_SHAPE, "%s: negative extent", op);
    MBRT_REQUIRE(offset >= 0 && offset + chunk_len <= dest_len, MBRT_E_SHAPE,
                 "%s: chunk [%lld, %lld) outside an output of %lld samples", op, (long long)offset,
                 (long long)(offset + chunk_len), (long long)dest_len);
    if (channels == 0 || chunk_len == 0) return MBRT_OK;
    MBRT_REQUIRE(dest && weight_sum && src && window, MBRT_E_INVALID_ARG, "%s: NULL pointer", op);
    AccArgs a{dest, weight_sum, src, window, chunk_len, dest_len, offset, channels, 0};
    hipStream_t st = as_stream(stream);
    MBRT_REQUIRE(channels <= 65535, MBRT_E_SHAPE, "%s: too many channels", op);
    // 16-byte accesses where all of them are aligned, and at any alignment where there is much to move
    const bool vec = chunk_len % 4 == 0 && dest_len % 4 == 0 && offset % 4 == 0 && aligned(dest, 16) &&
                     aligned(weight_sum, 16) && aligned(src, 16) && aligned(window, 16);
    if (!vec && (chunk_len < 4 || channels * chunk_len < MBRT_CHUNK_ANY)) {
        hipLaunchKernelGGL(accumulate_scalar_kernel, dim3((unsigned)grid_for(chunk_len), (unsigned)channels),
                           dim3(kThreads), 0, st, a);
        return check_launch(op);
    }
    auto launch = [&](auto cpb) {
        constexpr int CPB = decltype(cpb)::value;
        a.vblocks = (uint32_t)std::min<int64_t>(ceil_div(chunk_len / 4, 64), int64_t(1) << 16);
        const unsigned gx = a.vblocks + (chunk_len % 4 != 0 ? 1 : 0);
        hipLaunchKernelGGL(accumulate_cw_kernel<CPB>, dim3(gx, (unsigned)ceil_div(channels, CPB)), dim3(64 * CPB), 0, st,
                           a);
    };
    // no more waves in a block than there are channels
    if (channels <= 1) launch(std::integral_constant<int, 1>{});
    else if (channels <= 2) launch(std::integral_constant<int, 2>{});
    else launch(std::integral_constant<int, MBRT_CHUNK_CPB>{});
    return check_launch(op);
}

int mbrt_chunk_normalize(float* data, const float* weight_sum, int64_t channels, int64_t length,
                         mbrt_stream_t stream) {
    const char* op = "mbrt_chunk_normalize";
    MBRT_REQUIRE(channels >= 0 && length >= 0, MBRT_E_SHAPE, "%s: negative extent", op);
    if (channels == 0 || length == 0) return MBRT_OK;
    MBRT_REQUIRE(data && weight_sum, MBRT_E_INVALID_ARG, "%s: NULL pointer", op);
    NormArgs a{data, weight_sum, length, channels, (uint32_t)grid_for(length / 4)};
    // as the accumulate: 16-byte accesses where aligned, and at any alignment where there is much to move
    const bool vec = length % 4 == 0 && aligned(data, 16) && aligned(weight_sum, 16);
    if (!vec && (length < MBRT_NORM_ANY || channels * length < 3 * MBRT_NORM_ANY)) {
        hipLaunchKernelGGL(normalize_scalar_kernel, dim3((unsigned)grid_for(length)), dim3(kThreads), 0,
                           as_stream(stream), a);
        return check_launch(op);
    }
    hipLaunchKernelGGL(normalize_vec_kernel, dim3(a.vblocks + (length % 4 != 0 ? 1 : 0)), dim3(kThreads), 0,
                       as_stream(stream), a);
    return check_launch(op);
}

int mbrt_chunk_fade_window(float* window, int64_t chunk_size, int64_t fade_size, int first, int last) {
    MBRT_REQUIRE(chunk_size >= 0 && fade_size >= 0 && 2 * fade_size <= chunk_size, MBRT_E_SHAPE,
                 "mbrt_chunk_fade_window: fade %lld does not fit a chunk of %lld", (long long)fade_size,
                 (long long)chunk_size);
    if (chunk_size == 0) return MBRT_OK;
    MBRT_REQUIRE(window != nullptr, MBRT_E_INVALID_ARG, "mbrt_chunk_fade_window: NULL pointer");
    for (int64_t i = 0; i < chunk_size; ++i) window[i] = 1.0f;
    if (fade_size == 1) {
        if (!first) window[0] = 0.0f;
        if (!last) window[chunk_size - 1] = 0.0f;
    } else if (fade_size > 1) {
        for (int64_t i = 0; i < fade_size; ++i) {
            const float alpha = (float)i / (float)(fade_size - 1);
            if (!first) window[i] = alpha;
            if (!last) window[chunk_size - fade_size + i] = 1.0f - alpha;
        }
    }
    return MBRT_OK;
}

}  // extern "C"

// Layout kernels: strided copy (permute / contiguous / clone of views), index_select,
// constant and reflect pad, concatenation.  All copies are bit-exact byte moves.
//
// Strided copy strategy (replaces tensor_tile::strided_copy_glue,
// src/tensor_cuda_glue.cu:146-188, 615-638, which divides/modulos every element over
// all dims and uploads its metadata with a synchronous H2D memcpy):
//   1. drop size-1 dims and merge dims that are contiguous in the source;
//   2. if the innermost remaining dim has source stride 1, every output row is a
//      contiguous run in both tensors: copy it with the widest vector (16/8/4/2/1 B)
//      that divides the run, the source row pitches and both base addresses;
//   3. otherwise, if one source dim is unit-stride, stage 64x64-element tiles through
//      LDS so that both the read and the write are coalesced;
//   4. otherwise copy element by element.
// The bf16 [4,801,60,384] <-> [4,60,801,384] permute takes path 2 with 768-byte rows of
// 16-byte vectors.
#include "abi_common.hpp"

#include <algorithm>
#include <cstring>

namespace mbrt {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxOuter = MBRT_MAX_DIMS;

template <int W>
struct WordOf;
template <> struct WordOf<16> { typedef u32x4 T; };
template <> struct WordOf<8> { typedef u32x2 T; };
template <> struct WordOf<4> { typedef uint32_t T; };
template <> struct WordOf<2> { typedef uint16_t T; };
template <> struct WordOf<1> { typedef uint8_t T; };

// Simplified view of a copy: output is contiguous with shape `shape` (outermost first),
// the source element (c_0..c_{n-1}) lives at sum c_d * stride[d] (elements).
struct Dims {
    int nd = 0;
    int64_t shape[kMaxOuter];
    int64_t stride[kMaxOuter];
};

Dims simplify(const int64_t* shape, const int64_t* stride, int nd) {
    Dims r;
    for (int d = 0; d < nd; ++d) {
        if (shape[d] == 1) continue;
        if (r.nd > 0 && r.stride[r.nd - 1] == stride[d] * shape[d]) {
            r.shape[r.nd - 1] *= shape[d];
            r.stride[r.nd - 1] = stride[d];
        } else {
            r.shape[r.nd] = shape[d];
            r.stride[r.nd] = stride[d];
            ++r.nd;
        }
    }
    if (r.nd == 0) {
        r.nd = 1;
        r.shape[0] = 1;
        r.stride[0] = 1;
    }
    return r;
}

// ---- path 2: contiguous runs --------------------------------------------------------

struct RowCopyArgs {
    const char* src;
    char* dst;
    uint32_t total_vec;      // rows * vectors per row
    FastDiv vpr;             // vectors per row
    int64_t dst_pitch;       // output row pitch in bytes
    int nd;                  // number of outer dims
    int cold;                // the source is too large to be cached
    FastDiv outer[kMaxOuter];        // outer dim extents, innermost first
    int64_t outer_stride[kMaxOuter]; // source pitch in bytes, innermost first
};

template <int W, int U>
__global__ __launch_bounds__(kThreads) void row_copy_kernel(RowCopyArgs a) {
    typedef typename WordOf<W>::T Word;
    const uint32_t base = blockIdx.x * (kThreads * U) + threadIdx.x;
    Word v[U];
    int64_t dst_off[U], src_off[U];
    // all loads first (index clamped into the copy), then predicated stores
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t i = min(base + u * kThreads, a.total_vec - 1);
        uint32_t row, col;
        fdivmod(i, a.vpr, row, col);
        int64_t off = (int64_t)col * W;
        dst_off[u] = (int64_t)row * a.dst_pitch + (int64_t)col * W;
#pragma unroll
        for (int d = 0; d < kMaxOuter; ++d) {
            if (d < a.nd) {
                uint32_t q, r;
                fdivmod(row, a.outer[d], q, r);
                off += (int64_t)r * a.outer_stride[d];
                row = q;
            }
        }
        src_off[u] = off;
    }
    load_by<MBRT_NT_ROW>(a.cold, [&](auto nt) {
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = gld<decltype(nt)::value>(reinterpret_cast<const Word*>(a.src + src_off[u]));
    });
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (base + u * kThreads < a.total_vec) gst<MBRT_NT_ROW>(reinterpret_cast<Word*>(a.dst + dst_off[u]), v[u]);
    }
}

// Rows whose addresses, pitches or length are only element-aligned (a slice at an odd sample,
// a row of odd length): 16-byte accesses all the same, which global memory takes at any
// 2-byte-aligned address (unaligned access mode), with each row's last vector moved back to end
// at the row's end, so that it rewrites a few of the previous vector's bytes with the same
// values.  A is the alignment that all rows have.  Copying with words of that size instead
// is bound by the number of accesses: the 18 slice copies of a one-minute song's chunks
// ([2, 352800] f32 and the final crop of [2, 2645017]) took 4.85 us on average, now 3.58: the
// whole slices 4.37 -> 3.22, the crop 14.5 -> 9.8.  (All of them with ordinary stores 9 % more, with
// non-temporal loads as well 14 %.)
struct RowCopyUArgs {
    RowCopyArgs r;
    int64_t last;  // offset of a row's last vector: row bytes - 16
};

template <int A>
__global__ __launch_bounds__(kThreads) void row_copy_any_kernel(RowCopyUArgs a) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= a.r.total_vec) return;
    uint32_t row, col;
    fdivmod(i, a.r.vpr, row, col);
    const int64_t c = min((int64_t)col * 16, a.last);
    int64_t off = c;
    const int64_t dst_off = (int64_t)row * a.r.dst_pitch + c;
#pragma unroll
    for (int d = 0; d < kMaxOuter; ++d) {
        if (d < a.r.nd) {
            uint32_t q, r;
            fdivmod(row, a.r.outer[d], q, r);
            off += (int64_t)r * a.r.outer_stride[d];
            row = q;
        }
    }
    st_any<MBRT_NT_ROWU, A>(a.r.dst + dst_off, ld_any<MBRT_NT_ROWU, A>(a.r.src + off));
}

// 64-bit fallback for copies of more than 2^32 vectors.
struct RowCopyArgs64 {
    const char* src;
    char* dst;
    int64_t total_vec;
    int64_t vpr;
    int64_t dst_pitch;
    int nd;
    int64_t outer[kMaxOuter];
    int64_t outer_stride[kMaxOuter];
};

template <int W>
__global__ __launch_bounds__(kThreads) void row_copy_kernel64(RowCopyArgs64 a) {
    typedef typename WordOf<W>::T Word;
    int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const int64_t step = (int64_t)gridDim.x * kThreads;
    for (; i < a.total_vec; i += step) {
        int64_t row = i / a.vpr;
        const int64_t col_bytes = (i - row * a.vpr) * W;
        const int64_t dst_off = row * a.dst_pitch + col_bytes;
        int64_t off = col_bytes;
        for (int d = 0; d < a.nd; ++d) {
            int64_t q = row / a.outer[d];
            off += (row - q * a.outer[d]) * a.outer_stride[d];
            row = q;
        }
        *reinterpret_cast<Word*>(a.dst + dst_off) = *reinterpret_cast<const Word*>(a.src + off);
    }
}

template <int W>
int launch_row_copy(const char* src, char* dst, const Dims& dm, int esize, int64_t dst_pitch,
                    hipStream_t st) {
    const int64_t run_bytes = dm.shape[dm.nd - 1] * esize;
    const int64_t vpr = run_bytes / W;
    int64_t rows = 1;
    for (int d = 0; d < dm.nd - 1; ++d) rows *= dm.shape[d];
    const int64_t total = rows * vpr;
    bool small = total < (1ll << 31) && vpr < (1ll << 31);  // 32-bit vector indices cannot wrap
    for (int d = 0; d < dm.nd - 1; ++d) small = small && dm.shape[d] < (1ll << 31);
    if (small) {
        RowCopyArgs a;
        a.src = src;
        a.dst = dst;
        a.total_vec = (uint32_t)total;
        a.vpr = make_fastdiv((uint32_t)vpr);
        a.dst_pitch = dst_pitch;
        a.nd = dm.nd - 1;
        a.cold = cold_input(total * W);
        for (int d = 0; d < a.nd; ++d) {
            int src_d = dm.nd - 2 - d;
            a.outer[d] = make_fastdiv((uint32_t)dm.shape[src_d]);
            a.outer_stride[d] = dm.stride[src_d] * esize;
        }
        constexpr int U = MBRT_ROW_U;
        int64_t grid = ceil_div(total, (int64_t)kThreads * U);
        hipLaunchKernelGGL((row_copy_kernel<W, U>), dim3((unsigned)grid), dim3(kThreads), 0, st, a);
    } else {
        RowCopyArgs64 a;
        a.src = src;
        a.dst = dst;
        a.total_vec = total;
        a.vpr = vpr;
        a.dst_pitch = dst_pitch;
        a.nd = dm.nd - 1;
        for (int d = 0; d < a.nd; ++d) {
            int src_d = dm.nd - 2 - d;
            a.outer[d] = dm.shape[src_d];
            a.outer_stride[d] = dm.stride[src_d] * esize;
        }
        int64_t grid = std::min<int64_t>(ceil_div(total, kThreads), 1 << 20);
        hipLaunchKernelGGL((row_copy_kernel64<W>), dim3((unsigned)grid), dim3(kThreads), 0, st, a);
    }
    return MBRT_OK;
}

// Element-aligned rows in 16-byte vectors (row_copy_any_kernel); false when the rows are short
// or the vectors too many for 32-bit indices.  Rows below MBRT_ROWU_MIN bytes keep the
// element-sized words: the overlapping last vector is then a large part of a row.
template <int A>
bool try_row_copy_any(const char* src, char* dst, const Dims& dm, int esize, int64_t dst_pitch, hipStream_t st) {
    const int64_t run_bytes = dm.shape[dm.nd - 1] * esize;
    if (run_bytes < MBRT_ROWU_MIN) return false;
    const int64_t vpr = ceil_div(run_bytes, 16);
    if (vpr >= (1ll << 31)) return false;
    int64_t rows = 1;
    for (int d = 0; d < dm.nd - 1; ++d) {
        if (dm.shape[d] >= (1ll << 31)) return false;
        rows *= dm.shape[d];
        if (rows * vpr >= (1ll << 31)) return false;
    }
    RowCopyUArgs a;
    a.r.src = src;
    a.r.dst = dst;
    a.r.total_vec = (uint32_t)(rows * vpr);
    a.r.vpr = make_fastdiv((uint32_t)vpr);
    a.r.dst_pitch = dst_pitch;
    a.r.nd = dm.nd - 1;
    for (int d = 0; d < a.r.nd; ++d) {
        const int src_d = dm.nd - 2 - d;
        a.r.outer[d] = make_fastdiv((uint32_t)dm.shape[src_d]);
        a.r.outer_stride[d] = dm.stride[src_d] * esize;
    }
    a.last = run_bytes - 16;
    hipLaunchKernelGGL(row_copy_any_kernel<A>, dim3((unsigned)ceil_div(rows * vpr, kThreads)), dim3(kThreads), 0, st, a);
    return true;
}

// ---- path 3: LDS-tiled transpose ----------------------------------------------------
// The copy is viewed as out[batch, p, m, q] = in(batch, p, m, q) where q is the
// innermost output dim (source stride sq != 1) and p is the output dim that is
// unit-stride in the source.  A 64x64 tile over (p, q) is read along p (coalesced in
// the source) and written along q (coalesced in the output).  `batch` and `m`
// enumerate the remaining dims (outer to p, and between p and q).

constexpr int kTile = 64;

struct TransposeArgs {
    const char* src;
    char* dst;
    int64_t P, Q;                 // extents of p and q
    int64_t sq;                   // source stride of q (elements); source stride of p is 1
    int64_t out_p_pitch;          // output stride of p (elements) = M * Q
    int nb;                       // number of "other" dims (batch and m together)
    int64_t other_shape[kMaxOuter];
    int64_t other_src_stride[kMaxOuter];
    int64_t other_dst_stride[kMaxOuter];
    int64_t tiles_p, tiles_q;
};

template <int E>
__global__ __launch_bounds__(kThreads) void transpose_kernel(TransposeArgs a) {
    typedef typename WordOf<E>::T Elem;
    __shared__ Elem tile[kTile][kTile + 1];
    int64_t t = blockIdx.x;
    const int64_t tq = t % a.tiles_q;
    t /= a.tiles_q;
    const int64_t tp = t % a.tiles_p;
    t /= a.tiles_p;
    int64_t src_base = 0, dst_base = 0;
    for (int d = a.nb - 1; d >= 0; --d) {
        int64_t c = t % a.other_shape[d];
        t /= a.other_shape[d];
        src_base += c * a.other_src_stride[d];
        dst_base += c * a.other_dst_stride[d];
    }
    const int64_t p0 = tp * kTile, q0 = tq * kTile;
    const int lane = threadIdx.x % kTile;
    const int grp = threadIdx.x / kTile;  // 4 groups of 64
    // read: for each q row of the tile, 64 consecutive p (unit stride in source)
    for (int r = grp; r < kTile; r += kThreads / kTile) {
        int64_t p = p0 + lane, q = q0 + r;
        if (p < a.P && q < a.Q) {
            tile[r][lane] = gld<MBRT_NT_TR>(reinterpret_cast<const Elem*>(a.src) + src_base + q * a.sq + p);
        }
    }
    __syncthreads();
    // write: for each p row of the tile, 64 consecutive q (unit stride in output)
    for (int r = grp; r < kTile; r += kThreads / kTile) {
        int64_t p = p0 + r, q = q0 + lane;
        if (p < a.P && q < a.Q) {
            gst<MBRT_NT_TR>(reinterpret_cast<Elem*>(a.dst) + dst_base + p * a.out_p_pitch + q, tile[lane][r]);
        }
    }
}

// ---- path 4: generic element copy --------------------------------------------------

struct ElemCopyArgs {
    const char* src;
    char* dst;
    int64_t total;
    int nd;
    int64_t shape[kMaxOuter];   // outermost first
    int64_t stride[kMaxOuter];  // elements
};

template <int E>
__global__ __launch_bounds__(kThreads) void elem_copy_kernel(ElemCopyArgs a) {
    typedef typename WordOf<E>::T Elem;
    int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const int64_t step = (int64_t)gridDim.x * kThreads;
    for (; i < a.total; i += step) {
        int64_t rem = i, off = 0;
        for (int d = a.nd - 1; d >= 0; --d) {
            int64_t q = rem / a.shape[d];
            off += (rem - q * a.shape[d]) * a.stride[d];
            rem = q;
        }
        reinterpret_cast<Elem*>(a.dst)[i] = reinterpret_cast<const Elem*>(a.src)[off];
    }
}

int launch_elem_copy(const void* src, void* dst, const Dims& dm, int esize, hipStream_t st) {
    ElemCopyArgs a;
    a.src = static_cast<const char*>(src);
    a.dst = static_cast<char*>(dst);
    a.nd = dm.nd;
    a.total = 1;
    for (int d = 0; d < dm.nd; ++d) {
        a.shape[d] = dm.shape[d];
        a.stride[d] = dm.stride[d];
        a.total *= dm.shape[d];
    }
    int64_t grid = std::min<int64_t>(ceil_div(a.total, kThreads), 1 << 20);
    switch (esize) {
        case 1: hipLaunchKernelGGL(elem_copy_kernel<1>, dim3((unsigned)grid), dim3(kThreads), 0, st, a); break;
        case 2: hipLaunchKernelGGL(elem_copy_kernel<2>, dim3((unsigned)grid), dim3(kThreads), 0, st, a); break;
        case 4: hipLaunchKernelGGL(elem_copy_kernel<4>, dim3((unsigned)grid), dim3(kThreads), 0, st, a); break;
        default: hipLaunchKernelGGL(elem_copy_kernel<8>, dim3((unsigned)grid), dim3(kThreads), 0, st, a); break;
    }
    return MBRT_OK;
}

// Try the tiled transpose: needs a unit-stride source dim p that is not the innermost.
bool try_transpose(const void* src, void* dst, const Dims& dm, int esize, hipStream_t st) {
    const int q = dm.nd - 1;
    int p = -1;
    for (int d = 0; d < q; ++d) {
        if (dm.stride[d] == 1) p = d;
    }
    if (p < 0 || dm.shape[p] < 16 || dm.shape[q] < 16) return false;
    TransposeArgs a;
    a.src = static_cast<const char*>(src);
    a.dst = static_cast<char*>(dst);
    a.P = dm.shape[p];
    a.Q = dm.shape[q];
    a.sq = dm.stride[q];
    // output strides (contiguous, outermost first)
    int64_t ostride[kMaxOuter];
    int64_t acc = 1;
    for (int d = dm.nd - 1; d >= 0; --d) {
        ostride[d] = acc;
        acc *= dm.shape[d];
    }
    a.out_p_pitch = ostride[p];
    a.nb = 0;
    for (int d = 0; d < dm.nd; ++d) {
        if (d == p || d == q) continue;
        a.other_shape[a.nb] = dm.shape[d];
        a.other_src_stride[a.nb] = dm.stride[d];
        a.other_dst_stride[a.nb] = ostride[d];
        ++a.nb;
    }
    a.tiles_p = ceil_div(a.P, kTile);
    a.tiles_q = ceil_div(a.Q, kTile);
    int64_t blocks = a.tiles_p * a.tiles_q;
    for (int d = 0; d < a.nb; ++d) blocks *= a.other_shape[d];
    if (blocks > kMaxGridX) return false;
    switch (esize) {
        case 1: hipLaunchKernelGGL(transpose_kernel<1>, dim3((unsigned)blocks), dim3(kThreads), 0, st, a); break;
        case 2: hipLaunchKernelGGL(transpose_kernel<2>, dim3((unsigned)blocks), dim3(kThreads), 0, st, a); break;
        case 4: hipLaunchKernelGGL(transpose_kernel<4>, dim3((unsigned)blocks), dim3(kThreads), 0, st, a); break;
        default: hipLaunchKernelGGL(transpose_kernel<8>, dim3((unsigned)blocks), dim3(kThreads), 0, st, a); break;
    }
    return true;
}

int esize_of(int dt) { return dt_size(dt); }

int validate_meta_dims(const char* op, int nd, const int64_t* shape) {
    MBRT_REQUIRE(nd >= 1 && nd <= MBRT_MAX_DIMS, MBRT_E_INVALID_ARG, "%s: ndim %d out of [1, 8]", op, nd);
    for (int d = 0; d < nd; ++d) {
        MBRT_REQUIRE(shape[d] >= 0, MBRT_E_SHAPE, "%s: negative extent %lld at dim %d", op,
                     (long long)shape[d], d);
    }
    return MBRT_OK;
}

}  // namespace

// Copies `dm` (already simplified) from src to dst.  The output is contiguous except
// that, when the innermost dim is a unit-stride run, consecutive runs may be placed
// `dst_pitch` bytes apart (dst_pitch < 0: packed).
int strided_copy_dims(const void* src, void* dst, int esize, const Dims& dm, int64_t dst_pitch,
                      hipStream_t st) {
    const int64_t inner_stride = dm.stride[dm.nd - 1];
    if (inner_stride == 1) {
        const int64_t run_bytes = dm.shape[dm.nd - 1] * esize;
        if (dst_pitch < 0) dst_pitch = run_bytes;
        uintptr_t align_bits = reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst) |
                               (uintptr_t)run_bytes | (uintptr_t)dst_pitch;
        for (int d = 0; d < dm.nd - 1; ++d) align_bits |= (uintptr_t)(dm.stride[d] * esize);
        const char* s = (const char*)src;
        char* o = (char*)dst;
        if ((align_bits & 15) == 0) return launch_row_copy<16>(s, o, dm, esize, dst_pitch, st);
        if ((align_bits & 3) == 0 && try_row_copy_any<4>(s, o, dm, esize, dst_pitch, st)) return MBRT_OK;
        if ((align_bits & 7) == 0) return launch_row_copy<8>(s, o, dm, esize, dst_pitch, st);
        if ((align_bits & 3) == 0) return launch_row_copy<4>(s, o, dm, esize, dst_pitch, st);
        if ((align_bits & 1) == 0 && try_row_copy_any<2>(s, o, dm, esize, dst_pitch, st)) return MBRT_OK;
        if ((align_bits & 1) == 0) return launch_row_copy<2>(s, o, dm, esize, dst_pitch, st);
        return launch_row_copy<1>(s, o, dm, esize, dst_pitch, st);
    }
    if (try_transpose(src, dst, dm, esize, st)) return MBRT_OK;
    return launch_elem_copy(src, dst, dm, esize, st);
}

}  // namespace mbrt

using namespace mbrt;

extern "C" {

int mbrt_strided_copy(const void* src, void* dst, int dtype, const mbrt_strided_meta* meta,
                      mbrt_stream_t stream) {
    MBRT_REQUIRE(meta != nullptr, MBRT_E_INVALID_ARG, "mbrt_strided_copy: meta is NULL");
    MBRT_REQUIRE(is_valid_dt(dtype), MBRT_E_UNSUPPORTED_DTYPE, "mbrt_strided_copy: bad dtype %d", dtype);
    int s = validate_meta_dims("mbrt_strided_copy", meta->ndim, meta->dst_shape);
    if (s != MBRT_OK) return s;
    int64_t total = 1;
    for (int d = 0; d < meta->ndim; ++d) total *= meta->dst_shape[d];
    if (total == 0) return MBRT_OK;
    MBRT_REQUIRE(src != nullptr && dst != nullptr, MBRT_E_INVALID_ARG, "mbrt_strided_copy: NULL pointer");
    Dims dm = simplify(meta->dst_shape, meta->src_strides, meta->ndim);
    s = strided_copy_dims(src, dst, esize_of(dtype), dm, -1, as_stream(stream));
    if (s != MBRT_OK) return s;
    return check_launch("mbrt_strided_copy");
}

}  // extern "C"

// ---- index_select, pads, cat ---------------------------------------------------------

namespace mbrt {
namespace {

struct IndexSelectArgs {
    const char* src;
    char* dst;
    const void* idx;
    int idx_i64;
    int64_t total;
    int nd;
    int sel;
    int64_t shape[kMaxOuter];
    int64_t stride[kMaxOuter];
};

template <int E>
__global__ __launch_bounds__(kThreads) void index_select_kernel(IndexSelectArgs a) {
    typedef typename WordOf<E>::T Elem;
    int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const int64_t step = (int64_t)gridDim.x * kThreads;
    for (; i < a.total; i += step) {
        int64_t rem = i, off = 0;
        for (int d = a.nd - 1; d >= 0; --d) {
            int64_t q = rem / a.shape[d];
            int64_t c = rem - q * a.shape[d];
            if (d == a.sel) {
                c = a.idx_i64 ? reinterpret_cast<const int64_t*>(a.idx)[c]
                              : (int64_t)reinterpret_cast<const int32_t*>(a.idx)[c];
            }
            off += c * a.stride[d];
            rem = q;
        }
        reinterpret_cast<Elem*>(a.dst)[i] = reinterpret_cast<const Elem*>(a.src)[off];
    }
}

struct PadArgs {
    const char* src;
    char* dst;
    int64_t total;
    int nd;
    int64_t src_shape[kMaxOuter];
    int64_t dst_shape[kMaxOuter];
    int64_t before[kMaxOuter];
    uint64_t pad_bits;  // the pad value's bit pattern in the element type
    int reflect;
};

// The pad value's bits as one element (an 8-byte element is a vector of two dwords).
template <int E>
__device__ __forceinline__ typename WordOf<E>::T pad_elem(uint64_t bits) {
    if constexpr (E == 8) return u32x2{(uint32_t)bits, (uint32_t)(bits >> 32)};
    else return (typename WordOf<E>::T)bits;
}

template <int E>
__global__ __launch_bounds__(kThreads) void pad_kernel(PadArgs a) {
    typedef typename WordOf<E>::T Elem;
    int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const int64_t step = (int64_t)gridDim.x * kThreads;
    for (; i < a.total; i += step) {
        int64_t rem = i, src_lin = 0, src_pitch = 1;
        bool inside = true;
        for (int d = a.nd - 1; d >= 0; --d) {
            int64_t q = rem / a.dst_shape[d];
            int64_t c = rem - q * a.dst_shape[d] - a.before[d];
            rem = q;
            const int64_t n = a.src_shape[d];
            if (a.reflect) {
                if (c < 0) c = -c;
                if (c >= n) c = 2 * (n - 1) - c;
                c = c < 0 ? 0 : (c > n - 1 ? n - 1 : c);
            } else {
                inside = inside && c >= 0 && c < n;
            }
            src_lin += c * src_pitch;
            src_pitch *= n;
        }
        Elem v;
        if (inside) {
            v = reinterpret_cast<const Elem*>(a.src)[src_lin];
        } else {
            v = pad_elem<E>(a.pad_bits);
        }
        reinterpret_cast<Elem*>(a.dst)[i] = v;
    }
}

// Pads of the innermost dim only (the chunk and signal pads): rows of n elements in, m out.
// A thread writes 16 bytes of a row (the row's last vector moved back to end at the row's end,
// as in row_copy_any_kernel) from one 16-byte load wherever its elements are all inside the
// source or, reversed, all inside one reflected border; the few vectors across an edge go
// element by element.  The general kernel divides in 64 bits per element and dim: the reflect
// pad of a [1, 2, 2645017] f32 song took 32.3 us, here 9.8.
struct PadRowArgs {
    const char* src;
    char* dst;
    uint32_t total_vec;
    FastDiv vpr;         // vectors per output row
    int n, m;            // elements per source and output row
    int before;
    uint64_t pad_bits;
    int reflect;
};

// Positions are 32-bit: across an edge each element's index is worked out by itself, and eight 64-bit
// ones (2-byte elements) kept a small pad waiting for its arithmetic, [64, 100 -> 200] bf16 4.0 us.
template <int E>
__global__ __launch_bounds__(kThreads) void pad_row_kernel(PadRowArgs a) {
    typedef typename WordOf<E>::T Elem;
    constexpr int V = 16 / E;
    constexpr int A = E < 4 ? E : 4;
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= a.total_vec) return;
    uint32_t row, col;
    fdivmod(i, a.vpr, row, col);
    const int j = min((int)col * V, a.m - V);
    const int c = j - a.before;  // source index of the vector's first element
    const Elem* src = reinterpret_cast<const Elem*>(a.src) + (int64_t)row * a.n;
    union {
        u32x4 w;
        Elem e[V];
    } x, y;
    // where a whole vector's elements lie, as one load: forward, or reversed from lo
    int lo = c;
    bool rev = false;
    if (a.reflect && c + V <= 1) {         // |c|: all of c .. c + V - 1 at or left of 0
        lo = -(c + V - 1);
        rev = true;
    } else if (a.reflect && c >= a.n - 1) { // 2 (n - 1) - c: all at or right of n - 1
        lo = 2 * (a.n - 1) - (c + V - 1);
        rev = true;
    }
    if (lo >= 0 && lo <= a.n - V) {
        x.w = ld_any<0, A>(src + lo);
#pragma unroll
        for (int k = 0; k < V; ++k) y.e[k] = rev ? x.e[V - 1 - k] : x.e[k];
    } else {
#pragma unroll
        for (int k = 0; k < V; ++k) {
            int s = c + k;
            const bool inside = s >= 0 && s < a.n;
            if (a.reflect) {
                if (s < 0) s = -s;
                if (s >= a.n) s = 2 * (a.n - 1) - s;
            }
            s = max(min(s, a.n - 1), 0);
            const Elem v = src[s];  // always loaded: a load per branch would be waited for in it
            y.e[k] = a.reflect || inside ? v : pad_elem<E>(a.pad_bits);
        }
    }
    st_any<0, A>(reinterpret_cast<Elem*>(a.dst) + (int64_t)row * a.m + j, y.w);
}

// pad_row_kernel when only the innermost dim differs between source and output, its output
// rows hold at least one vector, the source is not empty and positions and vector indices fit 32
// bits.
bool try_pad_rows(const PadArgs& p, int esize, hipStream_t st) {
    const int last = p.nd - 1;
    int64_t rows = 1;
    for (int d = 0; d < last; ++d) {
        if (p.before[d] != 0 || p.src_shape[d] != p.dst_shape[d]) return false;
        rows *= p.dst_shape[d];
    }
    const int64_t n = p.src_shape[last], m = p.dst_shape[last], before = p.before[last];
    const int64_t v = 16 / esize, vpr = ceil_div(m, v), lim = int64_t(1) << 29;
    if (n < 1 || m < v || rows * vpr >= (1ll << 31)) return false;
    if (n >= lim || m >= lim || before <= -lim || before >= lim) return false;
    PadRowArgs a;
    a.n = (int)n;
    a.m = (int)m;
    a.before = (int)before;
    a.src = p.src;
    a.dst = p.dst;
    a.total_vec = (uint32_t)(rows * vpr);
    a.vpr = make_fastdiv((uint32_t)vpr);
    a.pad_bits = p.pad_bits;
    a.reflect = p.reflect;
    const dim3 grid((unsigned)ceil_div(rows * vpr, kThreads));
    switch (esize) {
        case 2: hipLaunchKernelGGL(pad_row_kernel<2>, grid, dim3(kThreads), 0, st, a); break;
        case 4: hipLaunchKernelGGL(pad_row_kernel<4>, grid, dim3(kThreads), 0, st, a); break;
        default: hipLaunchKernelGGL(pad_row_kernel<8>, grid, dim3(kThreads), 0, st, a); break;
    }
    return true;
}

// ---- cat: up to kCatSrcs sources in one launch ---------------------------------------
// Bound by launches where the sources are small: the 60 per-band tensors of a chunk
// ([1, 801, 28..520] f32, 51 MB moved) took 60 row copies of 2-3 us on the GPU, each ~2.5 us to
// enqueue; one launch takes 12.3-12.7 us (4.1 TB/s; a plain copy of 50 MB: 4.8).  A thread
// keeps one vector column of the sources and walks kCatU rows of it, so the column's source
// is looked up once (binary search of the columns in LDS), a wave writes up to 1 KB of
// consecutive output, and a source's rows are read whole.  2 or 8 rows per thread: 13.7-13.9
// and 13.6-14.0 us against 13.4-13.8 for 4, with non-temporal loads; the sources have usually
// just been written, so ordinary loads are kept: 12.3-12.7 (and 12.7-12.9 with ordinary
// stores too).
// Vectors are of 16 bytes at any even alignment: one word size for all sources, the largest that
// every address, row and offset allows, moved all of them in 2-byte words for one odd view.
// Two bf16 sources of 64 MB, one of them off by an element: 93 us by one copy each, 187 in 2-byte
// words, 60 as now; eight of 16 MB 70, 196 and 47.
constexpr int kCatSrcs = 64;
constexpr int kCatU = 4;  // rows per thread, all loads in flight before the first store

struct CatArgs {
    const char* src[kCatSrcs];
    int64_t dst[kCatSrcs];   // byte offset of the source in an output row
    int64_t run[kCatSrcs];   // bytes per source row
    uint32_t col[kCatSrcs];  // first of the source's vector columns, ascending
    char* out;
    int64_t dst_pitch;       // bytes between output rows
    int64_t outer;           // rows
    uint32_t cols;           // vector columns of all sources
    uint32_t col_blocks;     // blocks side by side over the columns
    int n;
    int tx_shift;            // log2 of the columns per block
};

// Vectors of V bytes at addresses aligned to A.  With A < V (V = 16) a source row's last vector is
// moved back to end at the row's end, as in row_copy_any_kernel; else every row holds whole vectors.
template <int V, int A>
__global__ __launch_bounds__(kThreads) void cat_kernel(CatArgs a) {
    typedef typename WordOf<V>::T Word;
    __shared__ const char* src[kCatSrcs];
    __shared__ int64_t dst[kCatSrcs], run[kCatSrcs];
    __shared__ uint32_t col[kCatSrcs];
    if ((int)threadIdx.x < a.n) {
        src[threadIdx.x] = a.src[threadIdx.x];
        dst[threadIdx.x] = a.dst[threadIdx.x];
        run[threadIdx.x] = a.run[threadIdx.x];
        col[threadIdx.x] = a.col[threadIdx.x];
    }
    __syncthreads();
    const uint32_t rb = blockIdx.x / a.col_blocks, cb = blockIdx.x - rb * a.col_blocks;
    const uint32_t tx = threadIdx.x & ((1u << a.tx_shift) - 1), ty = threadIdx.x >> a.tx_shift;
    const uint32_t ry = kThreads >> a.tx_shift;  // rows per step of the block
    const bool live = (cb << a.tx_shift) + tx < a.cols;
    const uint32_t c = min((cb << a.tx_shift) + tx, a.cols - 1);
    int s = 0;  // the last source that starts at or before the column
#pragma unroll
    for (int step = kCatSrcs / 2; step > 0; step >>= 1)
        if (s + step < a.n && col[s + step] <= c) s += step;
    const int64_t pitch = run[s];
    int64_t in = (int64_t)(c - col[s]) * V;
    if constexpr (A < V) in = min(in, pitch - V);
    const char* sp = src[s] + in;
    char* dp = a.out + dst[s] + in;
    const int64_t row0 = (int64_t)rb * (ry * kCatU) + ty;
    Word v[kCatU];
#pragma unroll
    for (int u = 0; u < kCatU; ++u) {
        const char* p = sp + min(row0 + (int64_t)(u * ry), a.outer - 1) * pitch;
        if constexpr (A < V) v[u] = ld_any<MBRT_NT_CAT, A>(p);
        else v[u] = gld<MBRT_NT_CAT>(reinterpret_cast<const Word*>(p));
    }
#pragma unroll
    for (int u = 0; u < kCatU; ++u) {
        const int64_t row = row0 + (int64_t)(u * ry);
        if (!live || row >= a.outer) continue;
        if constexpr (A < V) st_any<MBRT_NT_CAT, A>(dp + row * a.dst_pitch, v[u]);
        else gst<MBRT_NT_CAT>(reinterpret_cast<Word*>(dp + row * a.dst_pitch), v[u]);
    }
}

template <int V, int A>
void launch_cat(CatArgs& a, hipStream_t st) {
    int sh = 0;
    while ((1u << sh) < a.cols && (1 << sh) < kThreads) ++sh;
    a.tx_shift = sh;
    a.col_blocks = (uint32_t)ceil_div(a.cols, int64_t(1) << sh);
    const int64_t rows = (int64_t)(kThreads >> sh) * kCatU;
    const int64_t blocks = ceil_div(a.outer, rows) * a.col_blocks;
    hipLaunchKernelGGL((cat_kernel<V, A>), dim3((unsigned)blocks), dim3(kThreads), 0, st, a);
}

// The sources in launches of at most kCatSrcs when they lie in ascending order without
// overlap (a concat's always do), none of them lies in the output's memory (one that does may hold
// what an earlier source is to write there: copied one after another, they are in order) and the
// grid and column indices fit 32 bits; false otherwise, and nothing is launched: the caller
// copies them one after another.
bool try_cat(char* out, const mbrt_cat_src* srcs, int n, int64_t outer, int64_t total_cat_dim, int64_t inner_bytes,
             hipStream_t st) {
    const int64_t pitch = total_cat_dim * inner_bytes;
    uintptr_t bits = reinterpret_cast<uintptr_t>(out) | (uintptr_t)pitch;
    int64_t end = 0, used = 0, shortest = pitch, live = 0;
    for (int i = 0; i < n; ++i) {
        const int64_t run = srcs[i].dim_size * inner_bytes;
        if (run == 0) continue;
        if (srcs[i].dim_offset < end) return false;
        end = srcs[i].dim_offset + srcs[i].dim_size;
        const char* p = static_cast<const char*>(srcs[i].ptr);
        if (p < out + outer * pitch && out < p + outer * run) return false;
        bits |= reinterpret_cast<uintptr_t>(p) | (uintptr_t)run | (uintptr_t)(srcs[i].dim_offset * inner_bytes);
        used += run;
        shortest = std::min(shortest, run);
        ++live;
    }
    if (live < 2) return false;
    // long rows of large sources: a launch apiece costs little
    if (used / live >= MBRT_CAT_ROW && used * outer >= std::max(live * MBRT_CAT_SRC, MBRT_CAT_ALL)) return false;
    // the alignment that all addresses, rows and offsets have; 16-byte vectors at any even one where
    // every row holds one
    const int A = (bits & 15) == 0 ? 16 : (bits & 7) == 0 ? 8 : (bits & 3) == 0 ? 4 : (bits & 1) == 0 ? 2 : 1;
    const int V = A > 1 && shortest >= 16 ? 16 : A;
    const int64_t most = pitch / V + live;  // columns
    // blocks <= (outer / kCatU + 1) * (columns / kThreads + 1), kept below the grid limit
    if (most >= (int64_t(1) << 31) || outer >= (int64_t(1) << 32) ||
        (outer / kCatU + 1) * (most / kThreads + 1) > kMaxGridX)
        return false;
    CatArgs a{};
    a.out = out;
    a.dst_pitch = pitch;
    a.outer = outer;
    for (int i = 0; i < n; ++i) {
        const int64_t run = srcs[i].dim_size * inner_bytes;
        if (run == 0) continue;
        a.src[a.n] = static_cast<const char*>(srcs[i].ptr);
        a.dst[a.n] = srcs[i].dim_offset * inner_bytes;
        a.run[a.n] = run;
        a.col[a.n] = a.cols;
        a.cols += (uint32_t)ceil_div(run, V);
        ++a.n;
        --live;
        if (a.n < kCatSrcs && live > 0) continue;
        if (V == 16 && A == 16) launch_cat<16, 16>(a, st);
        else if (V == 16 && A >= 4) launch_cat<16, 4>(a, st);
        else if (V == 16) launch_cat<16, 2>(a, st);
        else if (V == 8) launch_cat<8, 8>(a, st);
        else if (V == 4) launch_cat<4, 4>(a, st);
        else if (V == 2) launch_cat<2, 2>(a, st);
        else launch_cat<1, 1>(a, st);
        a.n = 0;
        a.cols = 0;
    }
    return true;
}

int launch_pad(const void* src, void* dst, int dtype, const mbrt_pad_meta* m, float value,
               int reflect, const char* op, hipStream_t st) {
    MBRT_REQUIRE(m != nullptr, MBRT_E_INVALID_ARG, "%s: meta is NULL", op);
    MBRT_REQUIRE(is_valid_dt(dtype), MBRT_E_UNSUPPORTED_DTYPE, "%s: bad dtype %d", op, dtype);
    int s = validate_meta_dims(op, m->ndim, m->dst_shape);
    if (s != MBRT_OK) return s;
    PadArgs a;
    a.src = static_cast<const char*>(src);
    a.dst = static_cast<char*>(dst);
    a.nd = m->ndim;
    a.total = 1;
    int64_t src_total = 1;
    for (int d = 0; d < m->ndim; ++d) {
        a.src_shape[d] = m->src_shape[d];
        a.dst_shape[d] = m->dst_shape[d];
        a.before[d] = m->pad_before[d];
        a.total *= m->dst_shape[d];
        src_total *= m->src_shape[d];
        MBRT_REQUIRE(m->src_shape[d] >= 0, MBRT_E_SHAPE, "%s: negative source extent", op);
    }
    if (a.total == 0) return MBRT_OK;
    MBRT_REQUIRE(src_total > 0 || !reflect, MBRT_E_SHAPE, "%s: reflect pad of an empty source", op);
    a.reflect = reflect;
    // pad value in the element type (the reference converts the float pad value the same way)
    switch (dtype) {
        case F32: { uint32_t b; std::memcpy(&b, &value, 4); a.pad_bits = b; break; }
        case F16: { _Float16 h = (_Float16)value; uint16_t b; std::memcpy(&b, &h, 2); a.pad_bits = b; break; }
        case BF16: { __bf16 h = (__bf16)value; uint16_t b; std::memcpy(&b, &h, 2); a.pad_bits = b; break; }
        case I64: { int64_t v = (int64_t)value; std::memcpy(&a.pad_bits, &v, 8); break; }
        default: { int32_t v = (int32_t)value; uint32_t b; std::memcpy(&b, &v, 4); a.pad_bits = b; break; }
    }
    if (src_total == 0) a.reflect = 0;
    const bool rows = dt_size(dtype) > 2 || a.total >= MBRT_PAD2_MIN;
    if (rows && src_total > 0 && try_pad_rows(a, dt_size(dtype), st)) return check_launch(op);
    int64_t grid = std::min<int64_t>(ceil_div(a.total, kThreads), 1 << 20);
    switch (dt_size(dtype)) {
        case 2: hipLaunchKernelGGL(pad_kernel<2>, dim3((unsigned)grid), dim3(kThreads), 0, st, a); break;
        case 4: hipLaunchKernelGGL(pad_kernel<4>, dim3((unsigned)grid), dim3(kThreads), 0, st, a); break;
        default: hipLaunchKernelGGL(pad_kernel<8>, dim3((unsigned)grid), dim3(kThreads), 0, st, a); break;
    }
    return check_launch(op);
}

}  // namespace
}  // namespace mbrt

extern "C" {

int mbrt_index_select(const void* src, void* dst, int dtype, const void* indices,
                      int index_dtype, int64_t n_idx, int64_t src_dim_size,
                      const mbrt_strided_meta* meta, int select_dim, mbrt_stream_t stream) {
    const char* op = "mbrt_index_select";
    MBRT_REQUIRE(meta != nullptr, MBRT_E_INVALID_ARG, "%s: meta is NULL", op);
    MBRT_REQUIRE(is_valid_dt(dtype), MBRT_E_UNSUPPORTED_DTYPE, "%s: bad dtype %d", op, dtype);
    MBRT_REQUIRE(is_index_dt(index_dtype), MBRT_E_UNSUPPORTED_DTYPE, "%s: indices must be I32/I64", op);
    int s = validate_meta_dims(op, meta->ndim, meta->dst_shape);
    if (s != MBRT_OK) return s;
    MBRT_REQUIRE(select_dim >= 0 && select_dim < meta->ndim, MBRT_E_INVALID_ARG, "%s: select_dim %d", op, select_dim);
    MBRT_REQUIRE(meta->dst_shape[select_dim] == n_idx, MBRT_E_SHAPE,
                 "%s: dst extent %lld != number of indices %lld", op,
                 (long long)meta->dst_shape[select_dim], (long long)n_idx);
    (void)src_dim_size;
    IndexSelectArgs a;
    a.src = static_cast<const char*>(src);
    a.dst = static_cast<char*>(dst);
    a.idx = indices;
    a.idx_i64 = index_dtype == I64;
    a.nd = meta->ndim;
    a.sel = select_dim;
    a.total = 1;
    for (int d = 0; d < meta->ndim; ++d) {
        a.shape[d] = meta->dst_shape[d];
        a.stride[d] = meta->src_strides[d];
        a.total *= meta->dst_shape[d];
    }
    if (a.total == 0) return MBRT_OK;
    hipStream_t st = as_stream(stream);
    int64_t grid = std::min<int64_t>(ceil_div(a.total, kThreads), 1 << 20);
    switch (dt_size(dtype)) {
        case 2: hipLaunchKernelGGL(index_select_kernel<2>, dim3((unsigned)grid), dim3(kThreads), 0, st, a); break;
        case 4: hipLaunchKernelGGL(index_select_kernel<4>, dim3((unsigned)grid), dim3(kThreads), 0, st, a); break;
        default: hipLaunchKernelGGL(index_select_kernel<8>, dim3((unsigned)grid), dim3(kThreads), 0, st, a); break;
    }
    return check_launch(op);
}

int mbrt_pad_const(const void* src, void* dst, int dtype, const mbrt_pad_meta* meta, float value,
                   mbrt_stream_t stream) {
    return launch_pad(src, dst, dtype, meta, value, 0, "mbrt_pad_const", as_stream(stream));
}

int mbrt_pad_reflect(const void* src, void* dst, int dtype, const mbrt_pad_meta* meta,
                     mbrt_stream_t stream) {
    return launch_pad(src, dst, dtype, meta, 0.0f, 1, "mbrt_pad_reflect", as_stream(stream));
}

int mbrt_cat(void* out, const mbrt_cat_src* srcs, int n_srcs, int64_t outer_size,
             int64_t total_cat_dim, int64_t inner_bytes, mbrt_stream_t stream) {
    const char* op = "mbrt_cat";
    MBRT_REQUIRE(n_srcs >= 0 && (n_srcs == 0 || srcs != nullptr), MBRT_E_INVALID_ARG, "%s: bad source list", op);
    MBRT_REQUIRE(outer_size >= 0 && total_cat_dim >= 0 && inner_bytes >= 0, MBRT_E_SHAPE, "%s: negative size", op);
    hipStream_t st = as_stream(stream);
    int64_t used = 0;
    for (int i = 0; i < n_srcs; ++i) {
        MBRT_REQUIRE(srcs[i].dim_size >= 0 && srcs[i].dim_offset >= 0 &&
                         srcs[i].dim_offset + srcs[i].dim_size <= total_cat_dim,
                     MBRT_E_SHAPE, "%s: source %d does not fit the concat dim", op, i);
        used += srcs[i].dim_size;
    }
    (void)used;
    if (outer_size > 0 && try_cat(static_cast<char*>(out), srcs, n_srcs, outer_size, total_cat_dim, inner_bytes, st))
        return check_launch(op);
    for (int i = 0; i < n_srcs; ++i) {
        const int64_t run = srcs[i].dim_size * inner_bytes;
        if (run == 0 || outer_size == 0) continue;
        // one source = a [outer, run] byte matrix copied into [outer, total*inner] at an offset
        Dims dm;
        dm.nd = 2;
        dm.shape[0] = outer_size;
        dm.stride[0] = run;
        dm.shape[1] = run;
        dm.stride[1] = 1;
        char* dst = static_cast<char*>(out) + srcs[i].dim_offset * inner_bytes;
        // [outer, run] source bytes land in rows `total_cat_dim * inner_bytes` apart
        const int64_t dst_pitch = total_cat_dim * inner_bytes;
        int s = strided_copy_dims(srcs[i].ptr, dst, 1, dm, dst_pitch, st);
        if (s != MBRT_OK) return s;
    }
    return check_launch(op);
}

}  // extern "C"

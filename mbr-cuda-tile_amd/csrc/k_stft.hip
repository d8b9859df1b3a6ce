// STFT and iSTFT for n_fft = win_length = 2048 (src/stft_cuda_tile.cu:530-717): the
// spectrogram producer in front of the band gather and the waveform consumer after the
// mask merge, in the layouts those ops use ([B, 1025, T, 2] f32 spectra).
//
// The 2048-point real transform is a 1024-point complex FFT of z[m] = x[2m] + i x[2m+1]
// with the standard real-input split X[f] = (Z[f] + Z*[1024-f])/2 - i W^f (Z[f] -
// Z*[1024-f])/2 (W = exp(-2 pi i / 2048)), and the inverse split for the iSTFT.
// One wave transforms one frame; lane l holds z[l + 64a], a = 0..15, in registers.  The
// 1024-point FFT runs as three Stockham passes, radix 16, 16 and 4, with two exchanges
// through the frame's LDS slot, real parts and then imaginary parts (fft1024).  The last
// pass takes its butterflies in mirror pairs, so the real split needs no exchange.
//
// Workgroup = kTF waves = kTF consecutive frames of one signal.  The frames' spectra pass
// through LDS so that the [B, F, T] layout is written (STFT) or read (iSTFT) as runs of kTF
// consecutive frames per bin, instead of one 8-byte element per 8*T bytes.
//
// STFT   one kernel: the workgroup's sample span ((kTF - 1) hop + 2048 samples, reflect
//        padded at the signal ends) and the window are staged once into the frame slots
//        with coalesced loads (hops up to 658; larger hops read frame by frame), each wave
//        takes its windowed frame from there, then FFT, real
//        split, transposed store.  The split's 1/2 and the optional 1/sqrt(2048) scale the
//        window.
// iSTFT  two kernels: (1) per block of kTF frames of one signal: transposed spectrum load
//        (f32 or bf16), inverse split, inverse FFT, window, then the block's frames
//        overlap-added in LDS (frame order) into a partial signal in a caller workspace;
//        (2) per output sample: the partials of the blocks covering it (block order), times
//        1/2048 (sqrt(2048)/2048 when normalized), divided by the window sum of squares where
//        that exceeds 1e-8; centre trim and the `length` trim / zero fill are part of the
//        same pass.  No atomics: the result is deterministic.
//
// LDS costs that the layouts below are chosen for (measured, cycles per wave instruction
// without conflicts): 32-bit reads and writes 2 (32 lanes a cycle on 32 banks), 64-bit reads 2
// (32 lanes on 64 banks), 64-bit writes 4 (16 lanes on 32 banks), 128-bit reads 4, writes 8.
#include "abi_common.hpp"

#include <atomic>

#include <cmath>

namespace mbrt {
namespace {

constexpr int kN = 2048;        // n_fft = win_length
constexpr int kBins = kN / 2 + 1;
constexpr int kTF = 8;          // frames per workgroup, one wave per frame
constexpr int kNT = 64 * kTF;   // threads per workgroup
#ifndef MBRT_STFT_SUB
#define MBRT_STFT_SUB 4
#endif
constexpr int kSub = MBRT_STFT_SUB;         // frames of an STFT workgroup that takes part of a group
#ifndef MBRT_STFT_XCD
#define MBRT_STFT_XCD 32
#endif
#ifndef MBRT_ISTFT_XCD
#define MBRT_ISTFT_XCD 8
#endif
#ifndef MBRT_STFT_WPE
#define MBRT_STFT_WPE 4
#endif
#ifndef MBRT_ISTFT_WPE
#define MBRT_ISTFT_WPE 4
#endif
// MBRT_STFT_WPE, MBRT_ISTFT_WPE: waves per SIMD the register budgets allow for at least.  The STFT
// needs 64 VGPRs (four workgroups, 32 waves, per CU by registers and LDS), the iSTFT's block kernel 78 and
// twice the LDS (two workgroups).
//
// Frame blocks are dealt to the XCDs in runs of this many consecutive blocks, so the blocks
// that share the cache lines of a bin row ([B, 1025, T] holds kTF frames of a bin in
// 8 kTF bytes) meet in one L2, and so do the STFT's overlapping sample spans.
constexpr uint32_t kXcdRun = MBRT_STFT_XCD;
constexpr uint32_t kXcdRunInv = MBRT_ISTFT_XCD;
// LDS slot of one frame, in floats: one component (real, then imaginary) of 1024 points at
// padded indices (up to 1071), or half a spectrum (513 complex, and two more places) on its
// way out.  Eight of them and the twiddles are 38.8 KB.
constexpr int kSlot = 1088;

// ---- twiddles W^i = exp(-2 pi i i / 2048), built at compile time -----------------------
// cos/sin on [0, pi/4] by their Taylor series in double, extended to the circle by the
// octant symmetries, then rounded once to f32.
struct TwiddleTable {
    float v[2 * kN];  // (re, im) pairs
};

constexpr void taylor_cos_sin(double x, double& c, double& s) {
    double tc = 1.0, ts = x;
    const double x2 = x * x;
    c = 0.0;
    s = 0.0;
    for (int k = 0; k < 16; ++k) {
        c += tc;
        s += ts;
        tc *= -x2 / (double)((2 * k + 1) * (2 * k + 2));
        ts *= -x2 / (double)((2 * k + 2) * (2 * k + 3));
    }
}

constexpr TwiddleTable make_twiddles() {
    TwiddleTable t{};
    constexpr double kPi = 3.14159265358979323846;
    for (int i = 0; i < kN; ++i) {
        const int quarter = i / 512, j = i % 512;
        double c = 0.0, s = 0.0;
        if (j <= 256) {
            taylor_cos_sin(kPi * j / 1024.0, c, s);
        } else {
            double c2 = 0.0, s2 = 0.0;
            taylor_cos_sin(kPi * (512 - j) / 1024.0, c2, s2);
            c = s2;
            s = c2;
        }
        double cc = c, ss = s;  // cos, sin of quarter * pi/2 + theta
        if (quarter == 1) { cc = -s; ss = c; }
        if (quarter == 2) { cc = -c; ss = -s; }
        if (quarter == 3) { cc = s; ss = -c; }
        t.v[2 * i] = (float)cc;
        t.v[2 * i + 1] = (float)(-ss);
    }
    return t;
}

// The twiddles a workgroup keeps in LDS, each read at a lane-linear address plus a constant
// (no index arithmetic, no bank conflicts), forward values:
//   V  W256^(q n),  q = 1..3, n = k + 16 r < 64   pass 2, between its two radix-4 steps
//   U  W64^(q k),   q = 1..3, k < 16              pass 2, on its inputs
//   P  W1024^(q l), q = 1..3, l <= 64             pass 3 (further ones by reflection)
//   S  W2048^l,     l <= 64, inverse l <= 256     real split (further ones by rotation, in the
//                                                 inverse by swaps)
// Error of the result (relative, rms, against 64 bits; twelve inputs, hops 256 to 1000), beside
// 1.30e-7 and 1.38e-7 (STFT, iSTFT) of the form that formed pass 2's twiddles from products:
// 1.28e-7 and 1.36e-7.  The inverse with S rotated too: 1.40e-7 at 32.3 us a call on the chunk
// instead of 32.5, which is why it reads all of S.  With P up to l = 192 as well, and all of S,
// the STFT has 1.26e-7 but takes 19.1 us instead of 18.3.
constexpr int kTwV = 0, kTwU = kTwV + 3 * 64, kTwP = kTwU + 3 * 16, kTwS = kTwP + 3 * 65;
constexpr int kTwFwd = kTwS + 65, kTwSlots = kTwS + 257;  // slots of the STFT, and of the iSTFT
static_assert(kTwFwd <= kNT && kTwSlots > kNT && kTwSlots <= 2 * kNT, "one twiddle per thread, and two");

struct FftTable {
    float v[2 * kTwSlots];
};
constexpr FftTable make_fft_table() {
    const TwiddleTable w = make_twiddles();
    FftTable t{};
    auto put = [&](int at, int i) {
        t.v[2 * at] = w.v[2 * i];
        t.v[2 * at + 1] = w.v[2 * i + 1];
    };
    for (int q = 1; q <= 3; ++q) {
        for (int n = 0; n < 64; ++n) put(kTwV + (q - 1) * 64 + n, 8 * q * n);
        for (int k = 0; k < 16; ++k) put(kTwU + (q - 1) * 16 + k, 32 * q * k);
        for (int l = 0; l <= 64; ++l) put(kTwP + (q - 1) * 65 + l, 2 * q * l);
    }
    for (int l = 0; l <= 256; ++l) put(kTwS + l, l);
    return t;
}

__constant__ const FftTable kFftTable = make_fft_table();

struct cf {
    float x, y;
};
__device__ __forceinline__ cf cadd(cf a, cf b) { return {a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ cf csub(cf a, cf b) { return {a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ cf cmul(cf a, cf b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
// times -i (forward) or +i (inverse)
template <bool INV>
__device__ __forceinline__ cf rot(cf a) {
    return INV ? cf{-a.y, a.x} : cf{a.y, -a.x};
}
// a w (forward) or a conj(w) (inverse)
template <bool INV>
__device__ __forceinline__ cf cmulw(cf a, cf w) {
    return INV ? cf{a.x * w.x + a.y * w.y, a.y * w.x - a.x * w.y} : cmul(a, w);
}
// exp(-i angle) from the angle's cosine and sine
__device__ __forceinline__ cf unit(float c, float s) { return {c, -s}; }

template <bool INV>
__device__ __forceinline__ void dft4(cf& a0, cf& a1, cf& a2, cf& a3) {
    const cf t0 = cadd(a0, a2), t1 = csub(a0, a2), t2 = cadd(a1, a3), t3 = rot<INV>(csub(a1, a3));
    a0 = cadd(t0, t2);
    a2 = csub(t0, t2);
    a1 = cadd(t1, t3);
    a3 = csub(t1, t3);
}

// a * W16^E (conjugated for the inverse)
template <bool INV, int E>
__device__ __forceinline__ cf mul_w16(cf a) {
    constexpr float C1 = 0.92387953251128675613f, S1 = 0.38268343236508977173f, H = 0.70710678118654752440f;
    if constexpr (E == 4) return rot<INV>(a);
    constexpr float re = E == 1 ? C1 : E == 2 ? H : E == 3 ? S1 : E == 6 ? -H : -C1;  // E = 9
    constexpr float im = E == 1 ? -S1 : E == 2 ? -H : E == 3 ? -C1 : E == 6 ? -H : S1;
    return cmul(a, cf{re, INV ? -im : im});
}

// Second half of a 16-point DFT (radix 4 x 4): v[q0 + 4 r0] holds the twiddled outputs of the
// first radix-4 step; v[r0 + 4 r1] <- their DFT over q0.
template <bool INV>
__device__ __forceinline__ void dft16_tail(cf (&v)[16]) {
    cf o[16];
#pragma unroll
    for (int r0 = 0; r0 < 4; ++r0) {
        cf a0 = v[4 * r0], a1 = v[4 * r0 + 1], a2 = v[4 * r0 + 2], a3 = v[4 * r0 + 3];
        dft4<INV>(a0, a1, a2, a3);
        o[r0] = a0;
        o[r0 + 4] = a1;
        o[r0 + 8] = a2;
        o[r0 + 12] = a3;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = o[r];
}

// 16-point DFT in place: v[r] <- sum_q v[q] W16^(q r)
template <bool INV>
__device__ __forceinline__ void dft16(cf (&v)[16]) {
#pragma unroll
    for (int q0 = 0; q0 < 4; ++q0) dft4<INV>(v[q0], v[q0 + 4], v[q0 + 8], v[q0 + 12]);
    // v[q0 + 4 r0] now holds A[q0][r0]; twiddle by W16^(q0 r0)
    v[5] = mul_w16<INV, 1>(v[5]);
    v[9] = mul_w16<INV, 2>(v[9]);
    v[13] = mul_w16<INV, 3>(v[13]);
    v[6] = mul_w16<INV, 2>(v[6]);
    v[10] = mul_w16<INV, 4>(v[10]);
    v[14] = mul_w16<INV, 6>(v[14]);
    v[7] = mul_w16<INV, 3>(v[7]);
    v[11] = mul_w16<INV, 6>(v[11]);
    v[15] = mul_w16<INV, 9>(v[15]);
    dft16_tail<INV>(v);
}

// Orders this wave's LDS accesses: lanes of one wave exchange data through the slot.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ cf lds_ld(const float2* s, int i) {
    const float2 t = s[i];
    return {t.x, t.y};
}
__device__ __forceinline__ void lds_st(float2* s, int i, cf v) { s[i] = make_float2(v.x, v.y); }

// One exchange of the FFT: element r of a lane's v goes to slot index at(r), element q of the
// result comes from from(q).  The slot holds one component at a time, half the LDS of a
// complex exchange, at a third more LDS cycles (2 + 2 per component against 4 + 2).
template <class At, class From>
__device__ __forceinline__ void exchange(cf (&v)[16], float* slot, At at, From from) {
    float re[16];
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < 16; ++r) slot[at(r)] = v[r].x;
    wave_lds_sync();
#pragma unroll
    for (int q = 0; q < 16; ++q) re[q] = slot[from(q)];
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < 16; ++r) slot[at(r)] = v[r].y;
    wave_lds_sync();
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = cf{re[q], slot[from(q)]};
}

// 1024-point FFT of one frame by one wave.  In: lane l holds z[l + 64a] in v[a].  Out: the four
// radix-4 butterflies of the last pass that the lane took, in mirror pairs: butterfly j yields
// Z[j + 256 r], r = 0..3, in its z[r], for
//   A: j = l,   B: j = 256 - l (lane 0: 128),   C: j = 128 + m,   D: j = 128 - m
// with m = l (lane 0: 64), so that Z[f] and Z[1024 - f] of every f sit in one lane.
template <bool INV>
__device__ __forceinline__ void fft1024(cf (&v)[16], float* slot, const float2* tw, int lane, cf (&zA)[4], cf (&zB)[4],
                                        cf (&zC)[4], cf (&zD)[4]) {
    const int k = lane & 15;
    // pass 1: radix 16 over z[j + 64q]; y[16j + r]
    dft16<INV>(v);
    // (index i at i + i / 32: 32 lanes 16 apart and 32 consecutive ones both cover the 32 banks)
    const int w1 = 16 * lane + (lane >> 1), r1 = lane + (lane >> 5);
    exchange(v, slot, [&](int r) { return w1 + r; }, [&](int q) { return r1 + 66 * q; });
    // pass 2: radix 16, span 16: inputs y[j + 64q] W256^(qk), k = j % 16; outputs
    // y2[(j - k) 16 + k + 16 r].  With q = q0 + 4 q1, W256^(qk) = W64^(q1 k) W256^(q0 k): the first
    // factor goes on the inputs, the second joins the W16^(q0 r0) between the radix-4 steps.
    {
        const float2* t = tw + k;
#pragma unroll
        for (int q1 = 1; q1 < 4; ++q1) {
            const cf w = lds_ld(t, kTwU + (q1 - 1) * 16);
#pragma unroll
            for (int q0 = 0; q0 < 4; ++q0) v[q0 + 4 * q1] = cmulw<INV>(v[q0 + 4 * q1], w);
        }
#pragma unroll
        for (int q0 = 0; q0 < 4; ++q0) dft4<INV>(v[q0], v[q0 + 4], v[q0 + 8], v[q0 + 12]);
#pragma unroll
        for (int q0 = 1; q0 < 4; ++q0)
#pragma unroll
            for (int r0 = 0; r0 < 4; ++r0)
                v[q0 + 4 * r0] = cmulw<INV>(v[q0 + 4 * r0], lds_ld(t, kTwV + (q0 - 1) * 64 + 16 * r0));
        dft16_tail<INV>(v);
    }
    const int m = lane ? lane : 64;
    const int jb[4] = {lane, lane ? 256 - lane : 128, 128 + m, 128 - m};
    // (index i at i + 16 (i / 256): the writes of 32 lanes are two runs of 16, 16 banks apart)
    const int w2 = 272 * (lane >> 4) + k;
    exchange(v, slot, [&](int r) { return w2 + 16 * r; }, [&](int q) { return jb[q >> 2] + 272 * (q & 3); });
    // pass 3: radix 4, span 256: inputs y2[j + 256q] W1024^(qj)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        zA[q] = v[q];
        zB[q] = v[4 + q];
        zC[q] = v[8 + q];
        zD[q] = v[12 + q];
    }
    constexpr float H = 0.70710678118654752440f;
    {
        const cf a1 = lds_ld(tw, kTwP + lane), a2 = lds_ld(tw, kTwP + 65 + lane), a3 = lds_ld(tw, kTwP + 130 + lane);
        zA[1] = cmulw<INV>(zA[1], a1);
        zA[2] = cmulw<INV>(zA[2], a2);
        zA[3] = cmulw<INV>(zA[3], a3);
        // angles q (256 - l) 2 pi / 1024 = q pi / 2 - (those of A); lane 0: q pi / 4
        cf b1 = unit(-a1.y, a1.x), b2 = unit(-a2.x, -a2.y), b3 = unit(a3.y, -a3.x);
        if (lane == 0) {
            b1 = unit(H, H);
            b2 = unit(0.0f, 1.0f);
            b3 = unit(-H, H);
        }
        zB[1] = cmulw<INV>(zB[1], b1);
        zB[2] = cmulw<INV>(zB[2], b2);
        zB[3] = cmulw<INV>(zB[3], b3);
    }
    {
        // angles q (128 +- m) 2 pi / 1024 = q pi / 4 +- phi_q
        const cf p1 = lds_ld(tw, kTwP + m), p2 = lds_ld(tw, kTwP + 65 + m), p3 = lds_ld(tw, kTwP + 130 + m);
        const float s1 = H * (p1.x - p1.y), d1 = H * (p1.x + p1.y);  // h (cos + sin), h (cos - sin)
        const float s3 = H * (p3.x - p3.y), d3 = H * (p3.x + p3.y);
        zC[1] = cmulw<INV>(zC[1], unit(d1, s1));
        zD[1] = cmulw<INV>(zD[1], unit(s1, d1));
        zC[2] = cmulw<INV>(zC[2], unit(p2.y, p2.x));
        zD[2] = cmulw<INV>(zD[2], unit(-p2.y, p2.x));
        zC[3] = cmulw<INV>(zC[3], unit(-s3, d3));
        zD[3] = cmulw<INV>(zD[3], unit(-d3, s3));
    }
    dft4<INV>(zA[0], zA[1], zA[2], zA[3]);
    dft4<INV>(zB[0], zB[1], zB[2], zB[3]);
    dft4<INV>(zC[0], zC[1], zC[2], zC[3]);
    dft4<INV>(zD[0], zD[1], zD[2], zD[3]);
}

// Real-input split of one mirror pair: X[f] and X[1024 - f], twice over, from Z[f] and
// Z[1024 - f] (W^f = wf); f = 0 with zg = Z[0] yields X[0] and X[1024].  (The factor 1/2 is
// folded into the window.)
__device__ __forceinline__ void r2c_pair(cf zf, cf zg, cf wf, cf& xf, cf& xg) {
    const cf A{zf.x + zg.x, zf.y - zg.y}, Bv{zf.x - zg.x, zf.y + zg.y};
    const cf P = cmul(wf, Bv);
    xf = cf{A.x + P.y, A.y - P.x};
    xg = cf{A.x - P.y, -(A.y + P.x)};
}

// ---- STFT -------------------------------------------------------------------------------
struct StftArgs {
    const float* x;    // [B, L]
    const float* w;    // [2048]
    float2* out;       // [B, 1025, T] complex
    int L;
    uint32_t T;        // frames per signal
    FastDiv ntb;       // groups of kTF frames per signal: group -> (signal, group in signal)
    uint32_t whole;    // groups that one workgroup takes whole
    int hop;
    int offset;        // 1024 when centred (reflect padding), else 0
    int staged;        // the frame slots hold the workgroup's sample span and the window
    float scale;       // 1/2 (of the real split), times 1/sqrt(2048) when normalized
};

// Sample c of a signal of L samples, reflected once about the ends, then clamped (the
// reference's pad_reflect rule).
__device__ __forceinline__ int reflect_index(int c, int L) {
    if (c < 0) c = -c;
    if (c >= L) c = 2 * (L - 1) - c;
    return c < 0 ? 0 : (c > L - 1 ? L - 1 : c);
}

typedef float f32x2_any __attribute__((ext_vector_type(2), aligned(4)));  // two floats at any float address
__device__ __forceinline__ float2 ld2_any(const float* p) {
    const f32x2_any v = *reinterpret_cast<const f32x2_any*>(p);
    return make_float2(v.x, v.y);
}

// Samples n = 2 (lane + 64 q), n + 1 of a frame that starts at sample `start` of signal xb, straight
// from memory.
__device__ __forceinline__ void load_frame(const StftArgs& a, const float* xb, int start, int lane, cf (&v)[16]) {
    if (start >= 0 && start + kN <= a.L) {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const float2 p = ld2_any(xb + start + 2 * (lane + 64 * q));
            v[q] = cf{p.x, p.y};
        }
    } else {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int n = start + 2 * (lane + 64 * q);
            v[q] = cf{xb[reflect_index(n, a.L)], xb[reflect_index(n + 1, a.L)]};
        }
    }
}

__device__ __forceinline__ float4 ld4_any(const float* p) { return __builtin_bit_cast(float4, ld_any<0, 4>(p)); }

// Stages `span` (>= 2048) samples from sample s of signal xb into LDS, the even ones at xst and the
// odd ones KH floats further (a frame's sample pairs are then two runs of consecutive words
// whatever the frame's first sample), and the twiddles and the scaled window beside
// them.  Every load is in flight before the first LDS write where the span lies inside the
// signal: KS vectors per thread, the vector index clamped to the last whole one.
template <int KS, int KH>
__device__ __forceinline__ void stage_span(const StftArgs& a, float* xst, float* wst, float2* tw, const float* xb, int s,
                                           int span) {
    const int tid = threadIdx.x;
    const float2 t = reinterpret_cast<const float2*>(kFftTable.v)[min(tid, kTwFwd - 1)];
    const float4 w = ld4_any(a.w + 4 * tid);
    if (s >= 0 && s + span <= a.L) {
        const int last = (span >> 2) - 1, tail = min((span & ~3) + tid, span - 1);
        float4 xv[KS];
#pragma unroll
        for (int k = 0; k < KS; ++k) xv[k] = ld4_any(xb + s + 4 * min(tid + kNT * k, last));
        float xt = 0.0f;
        if (tid < 3) xt = xb[s + tail];
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const int i = 2 * min(tid + kNT * k, last);
            *reinterpret_cast<float2*>(xst + i) = make_float2(xv[k].x, xv[k].z);
            *reinterpret_cast<float2*>(xst + KH + i) = make_float2(xv[k].y, xv[k].w);
        }
        if (tid < 3) xst[(tail & 1) * KH + (tail >> 1)] = xt;
    } else {
        for (int j0 = tid; j0 < span; j0 += 6 * kNT) {
            float xv[6];
#pragma unroll
            for (int k = 0; k < 6; ++k) xv[k] = xb[reflect_index(s + min(j0 + k * kNT, span - 1), a.L)];
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                const int i = j0 + k * kNT;
                if (i < span) xst[(i & 1) * KH + (i >> 1)] = xv[k];
            }
        }
    }
    if (tid < kTwFwd) tw[tid] = t;
    *reinterpret_cast<float4*>(wst + 4 * tid) = make_float4(w.x * a.scale, w.y * a.scale, w.z * a.scale, w.w * a.scale);
}

// Bound by vector arithmetic and LDS together, and by how evenly the CUs are loaded.  Per frame:
// 837 vector instructions (8.7 us of SIMD time on the chunk, [8, 352800] -> 6,408 frames) and 729
// LDS cycles (7.6 us), beside 64 MB of HBM (11 us).  65 of the LDS cycles are bank conflicts: the
// exchanges, the window, the twiddles and the transposed accesses have none by their indices, so
// they are likely the staging's, whose surplus threads all write the span's last vector again.
// The kernel that kept whole complex slots (two workgroups per CU) and computed its twiddle indices
// took 1,121 instructions and 726 cycles, of which 154 were conflicts.  25.7 us then, 19.7 now
// (rocprofv3, one box).  The same with layouts padded by p/16, whose 32-bit reads conflict: 28.4.
__global__ __launch_bounds__(kNT) __attribute__((amdgpu_waves_per_eu(MBRT_STFT_WPE))) void stft_kernel(StftArgs a) {
    __shared__ __attribute__((aligned(16))) float lds[kTF * kSlot + 2 * kTwFwd];
    float2* tw = reinterpret_cast<float2*>(lds + kTF * kSlot);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    // workgroup = frames t0 .. t0 + nf - 1 of signal b: one of the first `whole` groups of kTF frames,
    // or a kSub-frame part of one of the others
    uint32_t b, tb, sub = 0, nfm = kTF, g = xcd_runs<kXcdRun>(blockIdx.x, min(a.whole, gridDim.x));
    if (blockIdx.x >= a.whole) {
        const uint32_t q = blockIdx.x - a.whole;
        g = a.whole + q / (kTF / kSub);
        sub = q % (kTF / kSub) * kSub;
        nfm = kSub;
    }
    fdivmod(g, a.ntb, b, tb);
    const uint32_t t0 = tb * kTF + sub;
    if (t0 >= a.T) return;
    const int nf = (int)min(nfm, a.T - t0);
    const bool live = wave < nf;
    const float* xb = a.x + (int64_t)b * a.L;
    const int s = (int)t0 * a.hop - a.offset;
    cf v[16];
    if (a.staged) {
        // the frames of a workgroup overlap (hop < 2048): their span and the window are read
        // from HBM once, coalesced, into the frame slots, and each wave takes its frame there
        constexpr int KH = (kTF * kSlot - kN) / 2;
        float* xst = lds + kN;
        const int span = (nf - 1) * a.hop + kN;
        if (span <= 3 * 4 * kNT) stage_span<3, KH>(a, xst, lds, tw, xb, s, span);
        else stage_span<4, KH>(a, xst, lds, tw, xb, s, span);
        __syncthreads();
        if (live) {
            // samples h + 2 m and h + 2 m + 1 of the span, h the frame's first
            const int h = wave * a.hop;
            const float* x0 = xst + (h & 1) * KH + (h >> 1) + lane;
            const float* x1 = xst + (1 - (h & 1)) * KH + ((h + 1) >> 1) + lane;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const float2 w = reinterpret_cast<const float2*>(lds)[lane + 64 * q];
                v[q] = cf{x0[64 * q] * w.x, x1[64 * q] * w.y};
            }
        }
        __syncthreads();  // the staging area becomes the frame slots
    } else {
        if (threadIdx.x < kTwFwd) tw[threadIdx.x] = reinterpret_cast<const float2*>(kFftTable.v)[threadIdx.x];
        if (live) {
            load_frame(a, xb, s + wave * a.hop, lane, v);
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const float2 w = ld2_any(a.w + 2 * (lane + 64 * q));
                v[q] = cf{v[q].x * (w.x * a.scale), v[q].y * (w.y * a.scale)};
            }
        }
        __syncthreads();
    }
    // The spectra leave through LDS in two halves: bins f < 512, then their mirrors 1024 - f
    // (with bin 512 = its own), both at position f of the frame's slot, rotated by the frame
    // (f ^ 4 wave within 32) so that the transposed reads (8 frames x 4 bins in 32 lanes) fall on
    // different banks.
    float* slot = lds + wave * kSlot;
    float2* sc = reinterpret_cast<float2*>(slot);
    // places of a lane's pairs: f = p0, p0 + 256, p1 + 256, p1, p2, p2 + 256, p3 + 256, p3
    const int rot = wave << 2, m = lane ? lane : 64;
    const int p0 = lane ^ rot, p1 = (256 - lane) ^ rot, p2 = (128 + m) ^ rot, p3 = (128 - m) ^ rot;
    cf xg[8];
    if (live) {
        cf zA[4], zB[4], zC[4], zD[4];
        fft1024<false>(v, slot, tw, lane, zA, zB, zC, zD);
        wave_lds_sync();
        // W^f of every pair from W^l and W^m: angles l, pi/4 -+ l, pi/2 - l, and pi/8, 3 pi/8 +- m
        const cf sl = lds_ld(tw, kTwS + lane), sm = lds_ld(tw, kTwS + m);
        constexpr float H = 0.70710678118654752440f, C1 = 0.92387953251128675613f, S1 = 0.38268343236508977173f;
        auto pair = [&](int place, cf zf, cf zg, cf w, cf& g) {
            cf x;
            r2c_pair(zf, zg, w, x, g);
            lds_st(sc, place, x);
        };
        if (lane == 0) {  // butterfly 128 is its own mirror
            cf g;  // its mirrors wait in the slot's last two places
            pair(128 ^ rot, zB[0], zB[3], unit(C1, S1), g);
            lds_st(sc, kSlot / 2 - 1, g);
            pair(384 ^ rot, zB[1], zB[2], unit(S1, C1), g);
            lds_st(sc, kSlot / 2 - 2, g);
            // and so is A: Z[256 (4 - r)]
#pragma unroll
            for (int r = 0; r < 4; ++r) zB[r] = zA[(r + 1) & 3];
        }
        {
            const float c = sl.x, n = -sl.y, p4 = H * (c + n), m4 = H * (c - n);
            pair(p0, zA[0], zB[3], unit(c, n), xg[0]);
            pair(p0 + 256, zA[1], zB[2], unit(m4, p4), xg[1]);
            pair(p1 + 256, zB[1], zA[2], unit(n, c), xg[2]);
            pair(p1, zB[0], zA[3], unit(p4, m4), xg[3]);
        }
        {
            const float cm = sm.x, nm = -sm.y;
            const float cp = C1 * cm - S1 * nm, sp = S1 * cm + C1 * nm;  // pi/8 + m
            const float cq = C1 * cm + S1 * nm, sq = S1 * cm - C1 * nm;  // pi/8 - m
            pair(p2, zC[0], zD[3], unit(cp, sp), xg[4]);
            pair(p2 + 256, zC[1], zD[2], unit(sq, cq), xg[5]);
            pair(p3 + 256, zD[1], zC[2], unit(sp, cp), xg[6]);
            pair(p3, zD[0], zC[3], unit(cq, sq), xg[7]);
        }
    }
    __syncthreads();
    // transposed store: thread -> (frame t0 + tl, bins fr + 64 i, then 1024 - fr - 64 i)
    const int tl = threadIdx.x % kTF, fr = threadIdx.x / kTF;
    const float2* src = reinterpret_cast<const float2*>(lds + tl * kSlot) + (fr ^ (tl << 2));
    f32x2* dst = reinterpret_cast<f32x2*>(a.out) + ((int64_t)b * kBins * a.T + t0 + tl);
    const int64_t step = (int64_t)64 * a.T;
    float2 X[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) X[i] = src[64 * i];
    __syncthreads();
    if (tl < nf) {
        f32x2* p = dst + (int64_t)fr * a.T;
#pragma unroll
        for (int i = 0; i < 8; ++i) gst<MBRT_NT_STFT & 2>(p + i * step, f32x2{X[i].x, X[i].y});
    }
    if (live) {
        lds_st(sc, p0, xg[0]);
        lds_st(sc, p0 + 256, xg[1]);
        lds_st(sc, p1 + 256, xg[2]);
        lds_st(sc, p1, xg[3]);
        lds_st(sc, p2, xg[4]);
        lds_st(sc, p2 + 256, xg[5]);
        lds_st(sc, p3 + 256, xg[6]);
        lds_st(sc, p3, xg[7]);
        if (lane == 0) {
            lds_st(sc, 128 ^ rot, lds_ld(sc, kSlot / 2 - 1));
            lds_st(sc, 384 ^ rot, lds_ld(sc, kSlot / 2 - 2));
        }
    }
    __syncthreads();
    if (tl >= nf) return;
    f32x2* p = dst + (int64_t)(kN / 2 - fr) * a.T;
#pragma unroll
    for (int i = 0; i < 8; ++i) X[i] = src[64 * i];
#pragma unroll
    for (int i = 0; i < 8; ++i) gst<MBRT_NT_STFT & 2>(p - i * step, f32x2{X[i].x, X[i].y});
    if (fr == 0) {
        const float2 h = reinterpret_cast<const float2*>(lds + tl * kSlot)[512 + (tl << 2)];
        gst<MBRT_NT_STFT & 2>(dst + (int64_t)512 * a.T, f32x2{h.x, h.y});
    }
}

// ---- iSTFT ------------------------------------------------------------------------------
// Block kernel: one workgroup = kTF consecutive frames of one signal.  Their spectra are
// loaded transposed, each wave inverts one frame, and the workgroup overlap-adds its frames
// in LDS (frame order) and writes the block's partial signal, (nf - 1) hop + 2048 samples
// from sample t0 hop.  The final kernel adds, per output sample, the partials of the blocks
// that cover it (block order), scales and divides by the window sum.
struct IstftBlockArgs {
    const void* spec;   // [B, 1025, T] complex, f32 or bf16
    const float* w;
    float* part;        // [B, nTB, span] block partials, times 2048 / spectrum scale
    uint32_t T;
    FastDiv ntb;        // blocks per signal
    FastDiv hop;
    uint32_t span;      // (kTF - 1) hop + 2048: stride of a block's partial
    uint32_t blocks;    // B * nTB
};

// LDS slot of one frame, in floats: two runs of 513 bins (places up to 512 + 14), kHi apart, or
// the frame's 2048 samples.
constexpr int kHi = 528;
constexpr int kSlotInv = 2 * (kHi + 528);
static_assert(kSlotInv >= kN && kSlotInv >= kSlot, "a slot holds a frame and an exchange");

template <int SDT>
struct SpecElem {
    typedef f32x2 T;
};
template <>
struct SpecElem<BF16> {
    typedef uint32_t T;
};
__device__ __forceinline__ float2 bin_f32(f32x2 v) { return make_float2(v.x, v.y); }
__device__ __forceinline__ float2 bin_f32(uint32_t u) { return make_float2(bf16_lo(u), bf16_hi(u)); }

// Inverse real split of bin k (with its mirror 1024 - k), times 2: Z[k] (MIRROR: Z[1024 - k])
// from X[k], X[1024 - k] and W^-k = (c, s).
template <bool MIRROR>
__device__ __forceinline__ cf c2r_bin(float2 xk, float2 xg, float c, float s) {
    const cf A{xk.x + xg.x, xk.y - xg.y}, Bv{xk.x - xg.x, xk.y + xg.y};
    const cf Q = cmul(Bv, cf{c, s});
    return MIRROR ? cf{A.x + Q.y, Q.x - A.y} : cf{A.x - Q.y, A.y + Q.x};
}

// Bound by its chain of phases: load, inverse split, FFT, window, overlap-add, with two
// workgroups per CU by LDS.  Per frame 1,042 vector instructions (1,422 before) and 653 LDS cycles
// (837 before), no bank conflicts.  Chunk [8, 1025, 801] f32: 29.9 -> 28.0 us; two signals of 620
// frames, bf16, 156 workgroups: 12.0 -> 11.6 to 12.0.  Half slots as the STFT's, with the spectra
// and the overlap-add in two rounds each (four workgroups per CU), ran 0.3 and 2.6 us longer.
template <int SDT>
__global__ __launch_bounds__(kNT) __attribute__((amdgpu_waves_per_eu(MBRT_ISTFT_WPE))) void istft_block_kernel(IstftBlockArgs a) {
    typedef typename SpecElem<SDT>::T Elem;
    __shared__ __attribute__((aligned(16))) float lds[kTF * kSlotInv + 2 * kTwSlots];
    float2* tw = reinterpret_cast<float2*>(lds + kTF * kSlotInv);
    const uint32_t blk = xcd_runs<kXcdRunInv>(blockIdx.x, gridDim.x);
    uint32_t b, tb;
    fdivmod(blk, a.ntb, b, tb);
    const uint32_t t0 = tb * kTF;
    const int nf = (int)min((uint32_t)kTF, a.T - t0);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const bool live = wave < nf;
    // transposed spectrum load: thread -> (frame tl, bins fr + 64 j and their mirrors
    // 1024 - fr - 64 j, j = 0..7, and bin 512 for fr = 0), all in flight before the first LDS
    // write.  Frames past the block's last read that frame again.
    const int tl = threadIdx.x % kTF, fr = threadIdx.x / kTF;
    Elem lo[8], hi[8], mid;
    {
        const Elem* src = static_cast<const Elem*>(a.spec) + ((int64_t)b * kBins * a.T + t0 + min(tl, nf - 1));
        const int64_t step = (int64_t)64 * a.T;
        const Elem* pl = src + (int64_t)fr * a.T;
        const Elem* ph = src + (int64_t)(kN / 2 - fr) * a.T;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            lo[j] = gld<MBRT_NT_STFT & 1>(pl + j * step);
            hi[j] = gld<MBRT_NT_STFT & 1>(ph - j * step);
        }
        mid = gld<MBRT_NT_STFT & 1>(src + (int64_t)512 * a.T);
    }
    const float2* table = reinterpret_cast<const float2*>(kFftTable.v);
    const float2 tlo = table[threadIdx.x], thi = table[min((int)threadIdx.x + kNT, kTwSlots - 1)];
    // The spectra enter through LDS: X[k], k <= 512, at place k of the frame's slot and
    // X[1024 - k] kHi further.  Places are rotated by the frame (p ^ 2 frame within 16), so that
    // the 8 frames x 2 bins that 16 lanes write at a time fall on different banks.
    float2* st = reinterpret_cast<float2*>(lds + tl * kSlotInv);
    const int rt = tl << 1, fp = fr ^ rt;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        st[fp + 64 * j] = bin_f32(lo[j]);
        st[kHi + fp + 64 * j] = bin_f32(hi[j]);
    }
    if (fr == 0) {
        // the imaginary parts of bins 0 and 1024 drop out
        st[rt].y = 0.0f;
        st[kHi + rt].y = 0.0f;
        st[512 + rt] = bin_f32(mid);
        st[kHi + 512 + rt] = bin_f32(mid);
    }
    tw[threadIdx.x] = tlo;
    if (threadIdx.x + kNT < kTwSlots) tw[threadIdx.x + kNT] = thi;
    __syncthreads();
    // Each lane forms the 16 bins of its first radix-16 pass, Z[l + 64 a]: for a < 8 from pair
    // k = l + 64 a, for a = 15 - h as the mirror of pair k = m + 64 h, m = 64 - l.  The twiddles W^-k
    // of k and 512 - k have each other's cosine and sine, so eight reads serve all sixteen.
    float* slot = lds + wave * kSlotInv;
    cf zA[4], zB[4], zC[4], zD[4];
    if (live) {
        const float2* xk = reinterpret_cast<const float2*>(slot);
        const int rw = wave << 1, p = lane ^ rw, m = (64 - lane) ^ rw;
        const float2 *tp = tw + kTwS + lane, *tm = tw + kTwS - lane;
        cf v[16];
#pragma unroll
        for (int a = 0; a < 4; ++a) {  // k = l + 64 a and 512 - k, and k = 64 (a + 1) - l and 512 - k
            const cf w = lds_ld(tp, 64 * a), u = lds_ld(tm, 64 * (a + 1));
            const int a7 = 7 - a;
            v[a] = c2r_bin<false>(xk[p + 64 * a], xk[kHi + p + 64 * a], w.x, -w.y);
            v[8 + a] = c2r_bin<true>(xk[m + 64 * a7], xk[kHi + m + 64 * a7], -w.y, w.x);
            v[a7] = c2r_bin<false>(xk[p + 64 * a7], xk[kHi + p + 64 * a7], -u.y, u.x);
            v[15 - a] = c2r_bin<true>(xk[m + 64 * a], xk[kHi + m + 64 * a], u.x, -u.y);
        }
        fft1024<true>(v, slot, tw, lane, zA, zB, zC, zD);
    }
    // zX[r] = 2048 (x[2i], x[2i + 1]), i = j + 256 r: the windowed frames go back to LDS, 2048 floats
    // each, and the workgroup adds them, in frame order, to the block's partial (partial[u],
    // u = s - t0 hop).
    __syncthreads();  // the slots are no longer read
    if (live) {
        const int wm = lane ? lane : 64;
        const int jb[4] = {lane, lane ? 256 - lane : 128, 128 + wm, 128 - wm};
        float2* fs = reinterpret_cast<float2*>(lds + wave * kN);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const cf(&z)[4] = i == 0 ? zA : i == 1 ? zB : i == 2 ? zC : zD;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int k = jb[i] + 256 * r;
                const float2 w = ld2_any(a.w + 2 * k);
                fs[k] = make_float2(z[r].x * w.x, z[r].y * w.y);
            }
        }
    }
    __syncthreads();
    const uint32_t hop = a.hop.d;
    const uint32_t span = (nf - 1) * hop + kN;
    float* part = a.part + (int64_t)blk * a.span;
    // chunks of 128 positions per wave and step, two per lane
    for (uint32_t u0 = wave * 128; u0 < span; u0 += 128 * kTF) {
        // frames that reach the chunk's first position, and its last
        const uint32_t jlo = u0 >= (uint32_t)kN ? fdiv(u0 - kN, a.hop) + 1 : 0;
        const uint32_t jhi = min((uint32_t)nf - 1, fdiv(u0 + 127, a.hop));
        float acc0 = 0.0f, acc1 = 0.0f;
        for (uint32_t j = jlo; j <= jhi; ++j) {
            const float* f = lds + j * kN;
            const uint32_t i0 = u0 - j * hop;  // wraps where the frame starts later
            if (i0 <= (uint32_t)(kN - 128)) {  // the frame covers the whole chunk
                acc0 += f[i0 + lane];
                acc1 += f[i0 + lane + 64];
            } else {
                const uint32_t n0 = i0 + lane, n1 = n0 + 64;
                const float x0 = f[min(n0, kN - 1u)], x1 = f[min(n1, kN - 1u)];
                acc0 += n0 < (uint32_t)kN ? x0 : 0.0f;
                acc1 += n1 < (uint32_t)kN ? x1 : 0.0f;
            }
        }
        const uint32_t u = u0 + lane;
        if (u < span) gst<MBRT_NT_ISTFT & 2>(part + u, acc0);
        if (u + 64 < span) gst<MBRT_NT_ISTFT & 2>(part + u + 64, acc1);
    }
}

struct IstftFinalArgs {
    const float* part;    // [B, nTB, span]
    const float* w;
    float* out;           // [B, out_len]
    uint32_t batch;
    uint32_t out_len;
    FastDiv hop;
    FastDiv bhop;         // kTF * hop: block stride in samples
    uint32_t span;
    uint32_t ntb;
    uint32_t T;
    uint32_t valid;       // samples of the (trimmed) signal; out_len - valid zeros follow
    uint32_t offset;      // 1024 when centred
    float scale;          // of the partials: spectrum scale / 2048
};

// One thread per output sample position, for every signal of the batch: the window sum
// (the same for all signals) is formed once.
__global__ __launch_bounds__(256) void istft_final_kernel(IstftFinalArgs a) {
    const uint32_t hop = a.hop.d, bhop = a.bhop.d;
    for (uint32_t so = blockIdx.x * 256 + threadIdx.x; so < a.out_len; so += gridDim.x * 256) {
        if (so >= a.valid) {
            for (uint32_t b = 0; b < a.batch; ++b) gst<(MBRT_NT_ISTFT & 4) ? 2 : 0>(a.out + (int64_t)b * a.out_len + so, 0.0f);
            continue;
        }
        const uint32_t s = so + a.offset;
        // window sum of squares in frame order (f32), as the reference's window_sum; the
        // loads go 8 at a time, all in flight before their terms are added
        const uint32_t thi = min(a.T - 1, fdiv(s, a.hop));
        const uint32_t tlo = s >= (uint32_t)kN ? fdiv(s - kN, a.hop) + 1 : 0;
        float ws = 0.0f;
        for (uint32_t t = tlo; t <= thi; t += 8) {
            float wv[8];
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) wv[k] = a.w[t + k <= thi ? s - (t + k) * hop : 0];
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {
#pragma clang fp contract(off)
                if (t + k <= thi) ws = ws + wv[k] * wv[k];
            }
        }
        // blocks covering s, in block order; a block's partial is shorter when it is the last
        // one of its signal
        const uint32_t bhi = min(a.ntb - 1, fdiv(s, a.bhop));
        const uint32_t blo = s >= a.span ? fdiv(s - a.span, a.bhop) + 1 : 0;
        if (bhi <= blo + 1) {
            // at most two blocks (every hop >= 256): the same two offsets for every signal,
            // whose loads go 4 signals at a time
            bool v[2];
            int64_t off[2];
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) {
                const uint32_t tb = blo + i, u = s - tb * bhop;
                v[i] = tb <= bhi && u < (min((uint32_t)kTF, a.T - tb * kTF) - 1) * hop + kN;
                off[i] = v[i] ? (int64_t)tb * a.span + u : 0;
            }
            for (uint32_t b0 = 0; b0 < a.batch; b0 += 4) {
                float p[4][2];
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    const float* pb = a.part + (int64_t)min(b0 + k, a.batch - 1) * a.ntb * a.span;
                    p[k][0] = gld<MBRT_NT_ISTFT & 1>(pb + off[0]);
                    p[k][1] = gld<MBRT_NT_ISTFT & 1>(pb + off[1]);
                }
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    if (b0 + k >= a.batch) break;
                    float acc = 0.0f;
                    if (v[0]) acc += p[k][0];
                    if (v[1]) acc += p[k][1];
                    gst<(MBRT_NT_ISTFT & 4) ? 2 : 0>(a.out + (int64_t)(b0 + k) * a.out_len + so, ws > 1.0e-8f ? acc * a.scale / ws : acc * a.scale);
                }
            }
            continue;
        }
#pragma unroll 4
        for (uint32_t b = 0; b < a.batch; ++b) {
            const float* pb = a.part + (int64_t)b * a.ntb * a.span;
            float acc = 0.0f;
            for (uint32_t tb = blo; tb <= bhi; ++tb) {
                const uint32_t u = s - tb * bhop;
                const uint32_t nf = min((uint32_t)kTF, a.T - tb * kTF);
                if (u < (nf - 1) * hop + kN) acc += gld<MBRT_NT_ISTFT & 1>(pb + (int64_t)tb * a.span + u);
            }
            gst<(MBRT_NT_ISTFT & 4) ? 2 : 0>(a.out + (int64_t)b * a.out_len + so, ws > 1.0e-8f ? acc * a.scale / ws : acc * a.scale);
        }
    }
}

__global__ __launch_bounds__(256) void hann_kernel(float* out, int64_t size) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= size) return;
    const float phase = (float)i * (6.28318530717958647692f / (float)size);
    out[i] = 0.5f * (1.0f - cosf(phase));
}

int check_fixed_size(const char* op, int64_t n_fft, int64_t win_length, int64_t window_numel) {
    MBRT_REQUIRE(n_fft == kN && win_length == kN && window_numel == kN, MBRT_E_SHAPE,
                 "%s: only n_fft=2048, win_length=2048 with a 2048-sample window is supported "
                 "(got n_fft=%lld, win_length=%lld, window %lld)", op, (long long)n_fft,
                 (long long)win_length, (long long)window_numel);
    return MBRT_OK;
}

constexpr int64_t kMaxHop = int64_t(1) << 20;  // keeps block spans and sample indices in 32 bits

int64_t grid_for(int64_t work, int64_t per_block) {
    return std::min<int64_t>(ceil_div(work, per_block), int64_t(1) << 20);
}

}  // namespace
}  // namespace mbrt

using namespace mbrt;

extern "C" {

int64_t mbrt_stft_num_frames(int64_t length, int64_t hop, int center) {
    if (length < 0 || hop < 1) return -1;
    const int64_t padded = length + (center ? kN : 0);
    if (padded < kN) return 0;
    return (padded - kN) / hop + 1;
}

int mbrt_hann_window(float* out, int64_t size, mbrt_stream_t stream) {
    const char* op = "mbrt_hann_window";
    MBRT_REQUIRE(size >= 0 && size < (int64_t(1) << 31), MBRT_E_SHAPE, "%s: bad size %lld", op, (long long)size);
    if (size == 0) return MBRT_OK;
    MBRT_REQUIRE(out != nullptr, MBRT_E_INVALID_ARG, "%s: NULL pointer", op);
    if (size == 1) return mbrt_fill(out, F32, 1, 1.0, stream);
    hipLaunchKernelGGL(hann_kernel, dim3((unsigned)ceil_div(size, 256)), dim3(256), 0, as_stream(stream), out, size);
    return check_launch(op);
}

int mbrt_stft(const float* signal, const float* window, float* out, int64_t batch, int64_t length, int64_t n_fft,
              int64_t hop, int64_t win_length, int64_t window_numel, int center, int normalized,
              mbrt_stream_t stream) {
    const char* op = "mbrt_stft";
    int s = check_fixed_size(op, n_fft, win_length, window_numel);
    if (s != MBRT_OK) return s;
    MBRT_REQUIRE(batch >= 0 && length >= 1 && hop >= 1 && hop < (1 << 30), MBRT_E_SHAPE,
                 "%s: bad shape (batch %lld, length %lld, hop %lld)", op, (long long)batch, (long long)length,
                 (long long)hop);
    const int64_t T = mbrt_stft_num_frames(length, hop, center);
    MBRT_REQUIRE(T >= 1, MBRT_E_SHAPE, "%s: signal of %lld samples is shorter than n_fft=2048", op,
                 (long long)length);
    MBRT_REQUIRE(length <= (1 << 30) && batch * T < (int64_t(1) << 31), MBRT_E_SHAPE, "%s: too many samples or frames",
                 op);
    if (batch == 0) return MBRT_OK;
    MBRT_REQUIRE(signal && window && out, MBRT_E_INVALID_ARG, "%s: NULL pointer", op);
    MBRT_REQUIRE(aligned(out, 8), MBRT_E_ALIGN, "%s: out must be 8-byte aligned", op);
    StftArgs a{};
    a.x = signal;
    a.w = window;
    a.out = reinterpret_cast<float2*>(out);
    a.L = (int)length;
    a.T = (uint32_t)T;
    const int64_t ntb = ceil_div(T, kTF);
    a.ntb = make_fastdiv((uint32_t)ntb);
    a.hop = (int)hop;
    a.offset = center ? kN / 2 : 0;
    a.scale = normalized ? 0.5f / std::sqrt((float)kN) : 0.5f;
    // the kTF frame slots hold the window and the span (hops up to 658), or each wave reads its
    // frame from memory.  (Staging the span alone, which fits up to 950, and reading the window from
    // memory ran [8, 352800] with a hop of 700 in 18.4 us instead of 15.2, [2, 352800] in 14.2
    // instead of 10.5; whole complex slots, staged up to 1910, 15.7 and 10.9.)
    a.staged = kN + (kTF - 1) * hop + kN <= kTF * kSlot ? 1 : 0;
    const int64_t groups = batch * ntb;
    MBRT_REQUIRE(groups < kMaxGridX, MBRT_E_SHAPE, "%s: too many frames", op);
    // A CU that gets one group more than the others sets the time, so the groups left over after
    // every CU has the same number are taken by two workgroups each, four frames apiece, when
    // they would fill at most half of the CUs (beyond that the halves cost more than the even
    // spread gives: each stages 3/4 of the whole group's samples).  Chunk of 808 groups, 40 left over:
    // 22.1 -> 20.8 us; 7 groups (0.5 s of mono) 7.4 -> 6.5; 632 groups, hop 1000: 13.5 -> 13.0.
    // Parts of 2 and 1 frames: 21.0 and 23.2 on the chunk.
    const int64_t cus = cu_count(), rem = groups % cus;
    const int64_t parts = 2 * rem <= cus ? rem : 0;
    a.whole = (uint32_t)(groups - parts);
    const int64_t blocks = a.whole + parts * (kTF / kSub);
    hipLaunchKernelGGL(stft_kernel, dim3((unsigned)blocks), dim3(kNT), 0, as_stream(stream), a);
    return check_launch(op);
}

int64_t mbrt_istft_output_length(int64_t frames, int64_t hop, int center, int64_t length) {
    if (frames < 1 || hop < 1) return -1;
    if (length > 0) return length;
    const int64_t full = kN + (frames - 1) * hop;
    return center ? full - kN : full;
}

int64_t mbrt_istft_workspace_bytes(int64_t batch, int64_t frames, int64_t hop) {
    if (batch < 0 || frames < 0 || hop < 1 || hop > kMaxHop) return -1;
    return batch * ceil_div(frames, kTF) * ((kTF - 1) * hop + kN) * (int64_t)sizeof(float);
}

}  // extern "C"

namespace {

// Scratch of the allocation-free iSTFT (mbrt_istft_noalloc): the block partials of one
// call.  A file-scope device array of MBRT_ISTFT_SCRATCH_BYTES, allocated on every GPU
// that loads the library's code object and held until the process ends; all calls on one
// GPU share it, so calls that overlap there race.  Nothing in it needs clearing: the block
// pass writes every partial sample the final pass reads.  In host code `scratch` names a
// host-side stand-in, not device memory: its device address on the current GPU is taken
// once per device with hipGetSymbolAddress, and only that pointer reaches the kernels.
__device__ __align__(256) float scratch[MBRT_ISTFT_SCRATCH_BYTES / sizeof(float)];

constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch[kMaxDevices];

int scratch_ptr(const char* op, void** ptr) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    MBRT_REQUIRE(e == hipSuccess, MBRT_E_HIP, "%s: hipGetDevice: %s", op, hipGetErrorString(e));
    MBRT_REQUIRE(dev >= 0 && dev < kMaxDevices, MBRT_E_HIP, "%s: device %d beyond %d", op, dev, kMaxDevices);
    void* p = g_scratch[dev].load(std::memory_order_acquire);
    if (p == nullptr) {
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        MBRT_REQUIRE(e == hipSuccess && p != nullptr, MBRT_E_HIP, "%s: hipGetSymbolAddress: %s", op,
                     hipGetErrorString(e));
        g_scratch[dev].store(p, std::memory_order_release);
    }
    *ptr = p;
    return MBRT_OK;
}

// The two iSTFT passes over a workspace of block partials; `workspace` is NULL for the
// allocation-free entry point, which then uses this GPU's scratch array.
int istft_impl(const char* op, const void* spec, int spec_dtype, const float* window, float* out, int64_t batch,
               int64_t freq_bins, int64_t frames, int64_t n_fft, int64_t hop, int64_t win_length,
               int64_t window_numel, int center, int normalized, int64_t length, void* workspace,
               int64_t workspace_bytes, mbrt_stream_t stream) {
    const bool scratch = workspace == nullptr;
    int s = check_fixed_size(op, n_fft, win_length, window_numel);
    if (s != MBRT_OK) return s;
    MBRT_REQUIRE(freq_bins == kBins, MBRT_E_SHAPE, "%s: %lld frequency bins (expected 1025)", op,
                 (long long)freq_bins);
    MBRT_REQUIRE(spec_dtype == F32 || spec_dtype == BF16, MBRT_E_UNSUPPORTED_DTYPE,
                 "%s: spectrum must be F32 or BF16", op);
    MBRT_REQUIRE(batch >= 0 && frames >= 1 && frames < (1 << 30) && hop >= 1 && hop <= kMaxHop, MBRT_E_SHAPE,
                 "%s: bad shape (batch %lld, frames %lld, hop %lld)", op, (long long)batch, (long long)frames,
                 (long long)hop);
    const int64_t out_len = mbrt_istft_output_length(frames, hop, center, length);
    if (batch == 0 || out_len == 0) return MBRT_OK;
    MBRT_REQUIRE(spec && window && out, MBRT_E_INVALID_ARG, "%s: NULL pointer", op);
    const int64_t need = mbrt_istft_workspace_bytes(batch, frames, hop);
    if (scratch) {
        MBRT_REQUIRE(need <= MBRT_ISTFT_SCRATCH_BYTES, MBRT_E_SHAPE,
                     "%s: needs %lld bytes of scratch, more than the %lld the library holds per GPU (use mbrt_istft "
                     "with a workspace)",
                     op, (long long)need, (long long)MBRT_ISTFT_SCRATCH_BYTES);
        s = scratch_ptr(op, &workspace);
        if (s != MBRT_OK) return s;
        workspace_bytes = MBRT_ISTFT_SCRATCH_BYTES;
    }
    MBRT_REQUIRE(workspace_bytes >= need, MBRT_E_INVALID_ARG, "%s: workspace of %lld bytes, %lld needed", op,
                 (long long)workspace_bytes, (long long)need);
    MBRT_REQUIRE(aligned(workspace, 4) && aligned(spec, spec_dtype == F32 ? 8 : 4), MBRT_E_ALIGN,
                 "%s: spectrum and workspace must be aligned to their element", op);
    const int64_t full = kN + (frames - 1) * hop;
    const int64_t ntb = ceil_div(frames, kTF);
    MBRT_REQUIRE(batch * ntb < (int64_t(1) << 31) && batch * out_len < (int64_t(1) << 31) &&
                     full + kN < (int64_t(1) << 31),
                 MBRT_E_SHAPE, "%s: signal too long", op);
    hipStream_t st = as_stream(stream);
    IstftBlockArgs ba{};
    ba.spec = spec;
    ba.w = window;
    ba.part = static_cast<float*>(workspace);
    ba.T = (uint32_t)frames;
    ba.ntb = make_fastdiv((uint32_t)ntb);
    ba.hop = make_fastdiv((uint32_t)hop);
    ba.span = (uint32_t)((kTF - 1) * hop + kN);
    ba.blocks = (uint32_t)(batch * ntb);
    if (spec_dtype == F32) hipLaunchKernelGGL(istft_block_kernel<F32>, dim3(ba.blocks), dim3(kNT), 0, st, ba);
    else hipLaunchKernelGGL(istft_block_kernel<BF16>, dim3(ba.blocks), dim3(kNT), 0, st, ba);
    s = check_launch(op);
    if (s != MBRT_OK) return s;
    IstftFinalArgs fa{};
    fa.part = ba.part;
    fa.w = window;
    fa.out = out;
    fa.batch = (uint32_t)batch;
    fa.out_len = (uint32_t)out_len;
    fa.hop = make_fastdiv((uint32_t)hop);
    fa.bhop = make_fastdiv((uint32_t)(kTF * hop));
    fa.span = ba.span;
    fa.ntb = (uint32_t)ntb;
    fa.T = (uint32_t)frames;
    fa.valid = (uint32_t)std::min<int64_t>(out_len, center ? full - kN : full);
    fa.offset = center ? kN / 2 : 0;
    fa.scale = (normalized ? std::sqrt((float)kN) : 1.0f) / (float)kN;
    hipLaunchKernelGGL(istft_final_kernel, dim3((unsigned)grid_for(out_len, 256)), dim3(256), 0, st, fa);
    return check_launch(op);
}

}  // namespace

extern "C" {

int mbrt_istft(const void* spec, int spec_dtype, const float* window, float* out, int64_t batch,
               int64_t freq_bins, int64_t frames, int64_t n_fft, int64_t hop, int64_t win_length,
               int64_t window_numel, int center, int normalized, int64_t length, void* workspace,
               int64_t workspace_bytes, mbrt_stream_t stream) {
    if (workspace == nullptr) return set_error(MBRT_E_INVALID_ARG, "mbrt_istft: NULL workspace");
    return istft_impl("mbrt_istft", spec, spec_dtype, window, out, batch, freq_bins, frames, n_fft, hop, win_length,
                      window_numel, center, normalized, length, workspace, workspace_bytes, stream);
}

int mbrt_istft_noalloc(const void* spec, int spec_dtype, const float* window, float* out, int64_t batch,
                       int64_t freq_bins, int64_t frames, int64_t n_fft, int64_t hop, int64_t win_length,
                       int64_t window_numel, int center, int normalized, int64_t length, mbrt_stream_t stream) {
    return istft_impl("mbrt_istft_noalloc", spec, spec_dtype, window, out, batch, freq_bins, frames, n_fft, hop,
                      win_length, window_numel, center, normalized, length, nullptr, 0, stream);
}

}  // extern "C"

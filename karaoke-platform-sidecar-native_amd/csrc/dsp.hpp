// STFT / iSTFT for the separation front and back end.
//
// Numerics follow native/vocalarc_separation.c:993-1136: float samples times
// the float periodic Hann window, a radix-2 FFT in double precision, results
// rounded to float; the inverse applies the complex mask in float, fills the
// Hermitian half, inverse-FFTs in double, and the overlap-add accumulates
// (float)(x * w) in frame order and divides by the float sum of w^2.
//
// n_fft = 2048 (both models): one wave per frame, the real transform as one
// complex transform of half its length (rfft2048 below).  Any other n_fft: one
// workgroup transforms one frame in LDS (n_fft complex doubles); its FFT
// is the reference's radix-2 decimation in time with its butterflies grouped
// three stages at a time: a thread loads the 8 points {base + k + j*h} that
// stages h, 2h and 4h combine only among themselves, applies those 12
// butterflies in registers and writes them back -- the same operations on
// every point as stage-by-stage radix-2, in 4 LDS passes (and 4 barriers)
// instead of 11 for n = 2048, with points skewed in LDS (fft_slot) so their
// accesses do not collide on banks.  The overlap-add
// is a gather (each output sample sums the frames that cover it in ascending
// frame order), so no atomics are needed and the summation order is the
// reference's.
#pragma once

#include "common.hpp"

namespace vh {

struct double2_t {
    double x, y;
};

VH_DEVICE int reflect_index_dev(int index, int length) {
    if (length <= 1) return 0;
    while (index < 0 || index >= length) {
        if (index < 0) index = -index;
        else index = 2 * length - 2 - index;
    }
    return index;
}

// LDS slot of point i.  A 16-byte point covers 4 of the 64 banks, so point
// slot q uses bank quad q % 16; the skews i/8 and i/256 give 8 consecutive
// lanes distinct quads in every access pattern of the transform: the
// bit-reversed scatter (points 256 apart), the first pass (8 apart), the
// second (stride-1 within 8-lane groups) and the stride-1 passes.
VH_DEVICE int fft_slot(int i) { return i + (i >> 3) + (i >> 8); }
// Radix-2 butterfly of the decimation-in-time FFT: (a, b) -> (a + w b, a - w b).
VH_DEVICE void fft_bfly(double2_t &a, double2_t &b, double2_t w) {
    const double rr = b.x * w.x - b.y * w.y;
    const double ri = b.x * w.y + b.y * w.x;
    b = {a.x - rr, a.y - ri};
    a = {a.x + rr, a.y + ri};
}

// W_M^x, M = 2^lm, from tw[j] = exp(-2*pi*i*j/n) (conjugated for the inverse).
VH_DEVICE double2_t fft_tw(const double2_t *__restrict__ tw, int x, int lm, int log2n, bool inverse) {
    double2_t w = tw[x << (log2n - lm)];
    if (inverse) w.y = -w.y;
    return w;
}

// In-place FFT of buf (n = 2^log2n points, slot fft_slot(i), input in
// bit-reversed order); every thread of the block takes part.
VH_DEVICE void fft_lds(double2_t *buf, const double2_t *__restrict__ tw, int log2n, bool inverse) {
    const int n = 1 << log2n;
    const int tid = (int)threadIdx.x, nt = (int)blockDim.x;
    for (int s = 0; s < log2n;) {
        const int r = min(3, log2n - s);  // stages merged in this pass
        const int h = 1 << s;
        for (int g = tid; g < (n >> r); g += nt) {
            const int k = g & (h - 1);
            const int base = (g >> s) << (s + r);
            if (r == 3) {
                double2_t p[8];
#pragma unroll
                for (int j = 0; j < 8; j++) p[j] = buf[fft_slot(base + k + j * h)];
                const double2_t w1 = fft_tw(tw, k, s + 1, log2n, inverse);
                const double2_t w2a = fft_tw(tw, k, s + 2, log2n, inverse);
                const double2_t w2b = fft_tw(tw, k + h, s + 2, log2n, inverse);
                fft_bfly(p[0], p[1], w1);
                fft_bfly(p[2], p[3], w1);
                fft_bfly(p[4], p[5], w1);
                fft_bfly(p[6], p[7], w1);
                fft_bfly(p[0], p[2], w2a);
                fft_bfly(p[1], p[3], w2b);
                fft_bfly(p[4], p[6], w2a);
                fft_bfly(p[5], p[7], w2b);
#pragma unroll
                for (int j = 0; j < 4; j++) fft_bfly(p[j], p[j + 4], fft_tw(tw, k + j * h, s + 3, log2n, inverse));
#pragma unroll
                for (int j = 0; j < 8; j++) buf[fft_slot(base + k + j * h)] = p[j];
            } else if (r == 2) {
                double2_t p[4];
#pragma unroll
                for (int j = 0; j < 4; j++) p[j] = buf[fft_slot(base + k + j * h)];
                const double2_t w1 = fft_tw(tw, k, s + 1, log2n, inverse);
                fft_bfly(p[0], p[1], w1);
                fft_bfly(p[2], p[3], w1);
                fft_bfly(p[0], p[2], fft_tw(tw, k, s + 2, log2n, inverse));
                fft_bfly(p[1], p[3], fft_tw(tw, k + h, s + 2, log2n, inverse));
#pragma unroll
                for (int j = 0; j < 4; j++) buf[fft_slot(base + k + j * h)] = p[j];
            } else {
                double2_t a = buf[fft_slot(base + k)], b = buf[fft_slot(base + k + h)];
                fft_bfly(a, b, fft_tw(tw, k, s + 1, log2n, inverse));
                buf[fft_slot(base + k)] = a;
                buf[fft_slot(base + k + h)] = b;
            }
        }
        __syncthreads();
        s += r;
    }
}

// LDS bytes of one padded n-point transform (slots up to fft_slot(n - 1)).
inline size_t fft_lds_bytes(int n) { return (size_t)(n + n / 8 + n / 256 + 1) * sizeof(double2_t); }

VH_DEVICE int bitrev_dev(int i, int log2n) { return (int)(__brev((unsigned)i) >> (32 - log2n)); }

// The STFT / iSTFT kernels run 256 threads per frame; their global loads are
// issued DSP_UNROLL per thread at a time so a frame waits on memory once per
// 2048 elements rather than once per element.
constexpr int DSP_THREADS = 256, DSP_UNROLL = 8;

// One frame of the STFT of one signal.  Signal `sig` = chunk * C + c reads
// samples audio[c][start_k + j] (zero beyond `audio_len`), j in
// [0, sig_len), with centre reflect padding inside the window of the chunk.
// Output: bins (chunk, f, c, t) of `source` in layout `out`.
struct StftArgs {
    const float *audio;
    int64_t audio_len;       // samples per channel of the audio buffer
    const int64_t *starts;   // chunk start sample per chunk (device), or null = 0
    int sig_len;             // window (chunk) length
    int C, T, F, n_fft, log2n, hop;
    const float *window;     // [n_fft]
    const double2_t *tw;     // [n_fft/2]
    float *source;
    SpecLayout out;
};

static __global__ __launch_bounds__(256) void stft_kernel(StftArgs a) {
    extern __shared__ double2_t sbuf[];
    const int t = (int)blockIdx.x;
    const int sig = (int)blockIdx.y;
    const int chunk = sig / a.C, c = sig % a.C;
    const int64_t start = a.starts ? a.starts[chunk] : 0;
    const float *src = a.audio + (size_t)c * a.audio_len;
    const int base = t * a.hop - a.n_fft / 2;
    const int tid = (int)threadIdx.x;
    for (int i0 = 0; i0 < a.n_fft; i0 += DSP_THREADS * DSP_UNROLL) {
        float xv[DSP_UNROLL], wv[DSP_UNROLL];
#pragma unroll
        for (int u = 0; u < DSP_UNROLL; u++) {
            const int i = i0 + tid + DSP_THREADS * u;
            xv[u] = 0.0f;
            wv[u] = 0.0f;
            if (i < a.n_fft) {
                const int64_t g = start + reflect_index_dev(base + i, a.sig_len);
                xv[u] = g < a.audio_len ? src[g] : 0.0f;
                wv[u] = a.window[i];
            }
        }
#pragma unroll
        for (int u = 0; u < DSP_UNROLL; u++) {
            const int i = i0 + tid + DSP_THREADS * u;
            if (i < a.n_fft) sbuf[fft_slot(bitrev_dev(i, a.log2n))] = {(double)(xv[u] * wv[u]), 0.0};
        }
    }
    __syncthreads();
    fft_lds(sbuf, a.tw, a.log2n, false);
    for (int f = (int)threadIdx.x; f < a.F; f += (int)blockDim.x) {
        const double2_t z = sbuf[fft_slot(f)];
        *reinterpret_cast<float2 *>(a.source + 2 * spec_at(a.out, chunk, f, c, t)) = float2{(float)z.x, (float)z.y};
    }
}

// Complex mask multiply + Hermitian fill + inverse FFT + window for one
// frame; frames[sig][T][n_fft] = (float)(x * w).
struct IstftArgs {
    const float *source;  // bins (chunk, f, c, t) in layout `in`
    const float *mask;    // same layout
    SpecLayout in;
    int C, T, F, n_fft, log2n;
    const float *window;
    const double2_t *tw;
    float *frames;        // [sig][T][n_fft]
};

static __global__ __launch_bounds__(256) void istft_frames_kernel(IstftArgs a) {
    extern __shared__ double2_t sbuf[];
    const int t = (int)blockIdx.x;
    const int sig = (int)blockIdx.y;
    const int chunk = sig / a.C, c = sig % a.C;
    const int n = a.n_fft;
    const int tid = (int)threadIdx.x;
    for (int f0 = 0; f0 < a.F; f0 += DSP_THREADS * DSP_UNROLL) {
        float2 sv[DSP_UNROLL], mv[DSP_UNROLL];
#pragma unroll
        for (int u = 0; u < DSP_UNROLL; u++) {
            const int f = f0 + tid + DSP_THREADS * u;
            if (f < a.F) {
                const int64_t e = 2 * spec_at(a.in, chunk, f, c, t);
                sv[u] = *reinterpret_cast<const float2 *>(a.source + e);
                mv[u] = *reinterpret_cast<const float2 *>(a.mask + e);
            }
        }
#pragma unroll
        for (int u = 0; u < DSP_UNROLL; u++) {
            const int f = f0 + tid + DSP_THREADS * u;
            if (f < a.F) {
                const float re = sv[u].x * mv[u].x - sv[u].y * mv[u].y;
                const float im = sv[u].x * mv[u].y + sv[u].y * mv[u].x;
                sbuf[fft_slot(bitrev_dev(f, a.log2n))] = {(double)re, (double)im};
                if (f >= 1 && f < a.F - 1) sbuf[fft_slot(bitrev_dev(n - f, a.log2n))] = {(double)re, -(double)im};
            }
        }
    }
    __syncthreads();
    fft_lds(sbuf, a.tw, a.log2n, true);
    const double scale = 1.0 / n;
    float *dst = a.frames + ((size_t)sig * a.T + t) * n;
    for (int i0 = 0; i0 < n; i0 += DSP_THREADS * DSP_UNROLL) {
        float wv[DSP_UNROLL];
#pragma unroll
        for (int u = 0; u < DSP_UNROLL; u++) {
            const int i = i0 + tid + DSP_THREADS * u;
            wv[u] = i < n ? a.window[i] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < DSP_UNROLL; u++) {
            const int i = i0 + tid + DSP_THREADS * u;
            if (i < n) dst[i] = (float)((sbuf[fft_slot(i)].x * scale) * (double)wv[u]);
        }
    }
}

// ---- n_fft = 2048: one wave per frame ---------------------------------------
// A frame's 2048 real samples are 1024 complex points z[m] = x[2m] + i x[2m+1];
// Z = FFT_1024(z) gives X[k] = e + W^k o, X[1024-k] = conj(e - W^k o) with
// e = (Z[k] + conj Z[1024-k]) / 2, o = (Z[k] - conj Z[1024-k]) / 2i, W = W_2048
// (the inverse the other way round).  So a frame costs half the points, and an
// exact zero frame stays exactly zero: frames do not share a transform.
//
// A lane holds 16 points at a time.  Forward (decimation in time): lane u loads
// z[u + 64 j] from memory -- a group of the bit-reversed order's first four
// stages -- transforms them in registers and writes 16 consecutive points to
// LDS; three more stages on two groups of 8 points, through LDS; and the last
// three on groups k and 128 - k (lane k; lane 0: 0 and 64), whose outputs
// k + 128 j and 1024 - (k + 128 j) are exactly the pairs the formula above
// combines, so the spectrum leaves from registers.  The inverse is the mirror
// (decimation in frequency).  The frame crosses LDS twice each way (64 KB of
// LDS traffic; radix-2 stages of the full-length complex transform in four
// passes took 311 KB) and nothing waits for another wave: no barriers.
// Twiddles: one table load per group, its square and fourth power computed.
// 60 s of stereo, 12002 frames: STFT 54 us (163 as 2048-point complex
// transforms, one 256-thread workgroup each), iSTFT 77 (189).
constexpr int RF_N = 2048, RF_H = RF_N / 2;
constexpr int RF_FRAMES = 4;  // frames (waves) per workgroup: 65 KB of LDS, eight waves per CU
// LDS slot of point i: sixteen lanes writing points 64 apart, or consecutive
// ones, touch sixteen distinct bank quads
VH_DEVICE int rf_slot(int i) { return i + (i >> 6); }
constexpr int RF_SLOTS = RF_H + RF_H / 64;

VH_DEVICE double2_t cadd(double2_t a, double2_t b) { return {a.x + b.x, a.y + b.y}; }
VH_DEVICE double2_t csub(double2_t a, double2_t b) { return {a.x - b.x, a.y - b.y}; }
VH_DEVICE double2_t cmul(double2_t a, double2_t b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
VH_DEVICE double2_t conj2(double2_t a) { return {a.x, -a.y}; }
// a times W_4 (-i; i for the inverse) and a times W_8
template <bool INV>
VH_DEVICE double2_t mul_w4(double2_t a) {
    return INV ? double2_t{-a.y, a.x} : double2_t{a.y, -a.x};
}
template <bool INV>
VH_DEVICE double2_t mul_w8(double2_t a) {
    constexpr double c = 0.70710678118654752440;
    return INV ? double2_t{(a.x - a.y) * c, (a.x + a.y) * c} : double2_t{(a.x + a.y) * c, (a.y - a.x) * c};
}
// Three stages of 8 points: W_2h^k = w1, W_4h^k = w2, W_8h^k = w3 (all 1 when
// UNIT), the other twiddles of a stage these times powers of W_8.
template <bool INV, bool UNIT>
VH_DEVICE void radix8_dit(double2_t *p, double2_t w1, double2_t w2, double2_t w3) {
    auto tw = [](double2_t v, double2_t w) { return UNIT ? v : cmul(v, w); };
    auto bfly = [&](int i, int j, double2_t t) {
        p[j] = csub(p[i], t);
        p[i] = cadd(p[i], t);
    };
#pragma unroll
    for (int i = 0; i < 8; i += 2) bfly(i, i + 1, tw(p[i + 1], w1));
#pragma unroll
    for (int i = 0; i < 8; i += 4) {
        bfly(i, i + 2, tw(p[i + 2], w2));
        bfly(i + 1, i + 3, mul_w4<INV>(tw(p[i + 3], w2)));
    }
    bfly(0, 4, tw(p[4], w3));
    bfly(1, 5, mul_w8<INV>(tw(p[5], w3)));
    bfly(2, 6, mul_w4<INV>(tw(p[6], w3)));
    bfly(3, 7, mul_w4<INV>(mul_w8<INV>(tw(p[7], w3))));
}
template <bool INV, bool UNIT>
VH_DEVICE void radix8_dif(double2_t *p, double2_t w1, double2_t w2, double2_t w3) {
    auto tw = [](double2_t v, double2_t w) { return UNIT ? v : cmul(v, w); };
    auto diff = [&](int i, int j) {
        const double2_t t = csub(p[i], p[j]);
        p[i] = cadd(p[i], p[j]);
        return t;
    };
    p[4] = tw(diff(0, 4), w3);
    p[5] = tw(mul_w8<INV>(diff(1, 5)), w3);
    p[6] = tw(mul_w4<INV>(diff(2, 6)), w3);
    p[7] = tw(mul_w4<INV>(mul_w8<INV>(diff(3, 7))), w3);
#pragma unroll
    for (int i = 0; i < 8; i += 4) {
        p[i + 2] = tw(diff(i, i + 2), w2);
        p[i + 3] = tw(mul_w4<INV>(diff(i + 1, i + 3)), w2);
    }
#pragma unroll
    for (int i = 0; i < 8; i += 2) p[i + 1] = tw(diff(i, i + 1), w1);
}
// W_16^j, j = 0..7 (conjugated for the inverse)
template <bool INV>
VH_DEVICE double2_t w16(int j) {
    constexpr double c1 = 0.92387953251128675613, s1 = 0.38268343236508977173, c2 = 0.70710678118654752440;
    const double c[8] = {1.0, c1, c2, s1, 0.0, -s1, -c2, -c1}, sn[8] = {0.0, s1, c2, c1, 1.0, c1, c2, s1};
    return {c[j], INV ? sn[j] : -sn[j]};
}
// The points a group's lane k (groups k and 128 - k; lane 0: 0 and 64) holds,
// a[j] = point k + 128 j (128 j) and b[j] = point 128 - k + 128 j (64 + 128 j),
// as eight pairs lo[j] = point i, hi[j] = point 1024 - i, i = rf_pair(lane, j),
// and point 512 beside them (lane 0; its pair 0 holds point 0 twice), and back.
VH_DEVICE int rf_pair(int lane, int j) { return lane ? lane + 128 * j : (j < 4 ? 128 * j : 64 + 128 * (j - 4)); }
VH_DEVICE double2_t sel(bool c, double2_t a, double2_t b) { return {c ? a.x : b.x, c ? a.y : b.y}; }
VH_DEVICE void rf_to_pairs(int lane, const double2_t *a, const double2_t *b, double2_t *lo, double2_t *hi) {
    const bool z = lane == 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        lo[j] = a[j];
        hi[j] = sel(z, j == 0 ? a[0] : a[8 - j], b[7 - j]);
        lo[4 + j] = sel(z, b[j], a[4 + j]);
        hi[4 + j] = sel(z, b[7 - j], b[3 - j]);
    }
}
VH_DEVICE void rf_from_pairs(int lane, const double2_t *lo, const double2_t *hi, double2_t mid, double2_t *a,
                             double2_t *b) {
    const bool z = lane == 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        a[j] = lo[j];
        b[7 - j] = sel(z, hi[4 + j], hi[j]);
        a[4 + j] = sel(z, j == 0 ? mid : hi[4 - j], lo[4 + j]);
        b[3 - j] = sel(z, lo[7 - j], hi[4 + j]);
    }
}
// LDS written by the wave's lanes is read by others of the same wave: its LDS
// operations complete in order, the compiler must keep them so.
VH_DEVICE void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
template <bool INV>
VH_DEVICE void rf_twiddles(const double2_t *__restrict__ tw, int i, double2_t &w1, double2_t &w2, double2_t &w3) {
    w3 = tw[i];
    if (INV) w3.y = -w3.y;
    w2 = cmul(w3, w3);
    w1 = cmul(w2, w2);
}
VH_DEVICE int brev4(int j) { return (j & 1) << 3 | (j & 2) << 1 | (j & 4) >> 1 | (j & 8) >> 3; }

static __global__ __launch_bounds__(64 * RF_FRAMES, 2) void stft2048_kernel(StftArgs a) {
    __shared__ double2_t lds[RF_FRAMES][RF_SLOTS];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    const int t = (int)blockIdx.x * RF_FRAMES + wave;
    if (t >= a.T) return;
    double2_t *buf = lds[wave];
    const int sig = (int)blockIdx.y;
    const int chunk = sig / a.C, c = sig % a.C;
    const int64_t start = a.starts ? a.starts[chunk] : 0;
    const float *src = a.audio + (size_t)c * a.audio_len;
    const int base = t * a.hop - RF_H;
    double2_t p[16];
    {
        // a frame inside the signal: 4-byte aligned pairs of samples (any hop)
        struct __attribute__((packed, aligned(4))) Pair { float x, y; };
        float2 xv[16];
        if (base >= 0 && base + RF_N <= a.sig_len && start + base + RF_N <= a.audio_len) {
            const float *f = src + start + base;
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const Pair v = *reinterpret_cast<const Pair *>(f + 2 * (lane + 64 * j));
                xv[j] = make_float2(v.x, v.y);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const int i = base + 2 * (lane + 64 * j);
                const int64_t g0 = start + reflect_index_dev(i, a.sig_len);
                const int64_t g1 = start + reflect_index_dev(i + 1, a.sig_len);
                xv[j].x = g0 < a.audio_len ? src[g0] : 0.0f;
                xv[j].y = g1 < a.audio_len ? src[g1] : 0.0f;
            }
        }
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const float2 w = *reinterpret_cast<const float2 *>(a.window + 2 * (lane + 64 * j));
            p[brev4(j)] = {(double)(xv[j].x * w.x), (double)(xv[j].y * w.y)};
        }
    }
    double2_t w1{}, w2{}, w3{};
    radix8_dit<false, true>(p, w1, w2, w3);
    radix8_dit<false, true>(p + 8, w1, w2, w3);
    const int group = 16 * bitrev_dev(lane, 6);
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const double2_t v = cmul(p[8 + j], w16<false>(j));
        buf[rf_slot(group + j)] = cadd(p[j], v);
        buf[rf_slot(group + 8 + j)] = csub(p[j], v);
    }
    wave_lds_order();
    rf_twiddles<false>(a.tw, 16 * (lane & 15), w1, w2, w3);
#pragma unroll
    for (int g = 0; g < 2; g++) {
        const int at = (((lane + 64 * g) >> 4) << 7) + (lane & 15);
#pragma unroll
        for (int j = 0; j < 8; j++) p[j] = buf[rf_slot(at + 16 * j)];
        radix8_dit<false, false>(p, w1, w2, w3);
#pragma unroll
        for (int j = 0; j < 8; j++) buf[rf_slot(at + 16 * j)] = p[j];
    }
    wave_lds_order();
#pragma unroll
    for (int g = 0; g < 2; g++) {
        const int k = g == 0 ? lane : (lane ? 128 - lane : 64);
#pragma unroll
        for (int j = 0; j < 8; j++) p[8 * g + j] = buf[rf_slot(k + 128 * j)];
        rf_twiddles<false>(a.tw, 2 * k, w1, w2, w3);
        radix8_dit<false, false>(p + 8 * g, w1, w2, w3);
    }
    double2_t lo[8], hi[8];
    rf_to_pairs(lane, p, p + 8, lo, hi);
    auto put = [&](int f, double2_t z) {
        *reinterpret_cast<float2 *>(a.source + 2 * spec_at(a.out, chunk, f, c, t)) = float2{(float)z.x, (float)z.y};
    };
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int i = rf_pair(lane, j);
        const double2_t e = {0.5 * (lo[j].x + hi[j].x), 0.5 * (lo[j].y - hi[j].y)};
        const double2_t o = {0.5 * (lo[j].y + hi[j].y), -0.5 * (lo[j].x - hi[j].x)};
        const double2_t v = cmul(a.tw[i], o);
        put(i, cadd(e, v));
        put(RF_H - i, conj2(csub(e, v)));
    }
    if (lane == 0) put(RF_H / 2, conj2(p[4]));
}

static __global__ __launch_bounds__(64 * RF_FRAMES, 2) void istft2048_frames_kernel(IstftArgs a) {
    __shared__ double2_t lds[RF_FRAMES][RF_SLOTS];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    const int t = (int)blockIdx.x * RF_FRAMES + wave;
    if (t >= a.T) return;
    double2_t *buf = lds[wave];
    const int sig = (int)blockIdx.y;
    const int chunk = sig / a.C, c = sig % a.C;
    // masked bins, the complex product in fp32
    float2 sv[17], mv[17];
    auto load = [&](int n, int f) {
        const int64_t e = 2 * spec_at(a.in, chunk, f, c, t);
        sv[n] = *reinterpret_cast<const float2 *>(a.source + e);
        mv[n] = *reinterpret_cast<const float2 *>(a.mask + e);
    };
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int i = rf_pair(lane, j);
        load(2 * j, i);
        load(2 * j + 1, RF_H - i);
    }
    load(16, RF_H / 2);
    auto bin = [&](int n) {
        return double2_t{(double)(sv[n].x * mv[n].x - sv[n].y * mv[n].y), (double)(sv[n].x * mv[n].y + sv[n].y * mv[n].x)};
    };
    // twice the half-length spectrum: the scale 1 / 2048 below halves it
    double2_t lo[8], hi[8], p[16];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        double2_t y = bin(2 * j), yc = conj2(bin(2 * j + 1));
        if (j == 0 && lane == 0) {  // bins 0 and 1024 are real: their imaginary parts reach no sample
            y = {y.x + 0.0 * y.y, 0.0};
            yc = {yc.x + 0.0 * yc.y, 0.0};
        }
        const double2_t e = cadd(y, yc), o = cmul(csub(y, yc), conj2(a.tw[rf_pair(lane, j)]));
        lo[j] = {e.x - o.y, e.y + o.x};   // e + i o
        hi[j] = {e.x + o.y, o.x - e.y};   // conj(e) + i conj(o)
    }
    const double2_t ym = bin(16);
    rf_from_pairs(lane, lo, hi, double2_t{2.0 * ym.x, -2.0 * ym.y}, p, p + 8);
    double2_t w1{}, w2{}, w3{};
#pragma unroll
    for (int g = 0; g < 2; g++) {
        const int k = g == 0 ? lane : (lane ? 128 - lane : 64);
        rf_twiddles<true>(a.tw, 2 * k, w1, w2, w3);
        radix8_dif<true, false>(p + 8 * g, w1, w2, w3);
#pragma unroll
        for (int j = 0; j < 8; j++) buf[rf_slot(k + 128 * j)] = p[8 * g + j];
    }
    wave_lds_order();
    rf_twiddles<true>(a.tw, 16 * (lane & 15), w1, w2, w3);
#pragma unroll
    for (int g = 0; g < 2; g++) {
        const int at = (((lane + 64 * g) >> 4) << 7) + (lane & 15);
#pragma unroll
        for (int j = 0; j < 8; j++) p[j] = buf[rf_slot(at + 16 * j)];
        radix8_dif<true, false>(p, w1, w2, w3);
#pragma unroll
        for (int j = 0; j < 8; j++) buf[rf_slot(at + 16 * j)] = p[j];
    }
    wave_lds_order();
    const int group = 16 * bitrev_dev(lane, 6);
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const double2_t u = buf[rf_slot(group + j)], v = buf[rf_slot(group + 8 + j)];
        p[j] = cadd(u, v);
        p[8 + j] = cmul(csub(u, v), w16<true>(j));
    }
    radix8_dif<true, true>(p, w1, w2, w3);
    radix8_dif<true, true>(p + 8, w1, w2, w3);
    const double scale = 1.0 / RF_N;
    float *dst = a.frames + ((size_t)sig * a.T + t) * RF_N;
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const float2 w = *reinterpret_cast<const float2 *>(a.window + 2 * (lane + 64 * j));
        const double2_t z = p[brev4(j)];
        *reinterpret_cast<float2 *>(dst + 2 * (lane + 64 * j)) =
            float2{(float)((z.x * scale) * (double)w.x), (float)((z.y * scale) * (double)w.y)};
    }
}

// Gather overlap-add: out[sig][s] = sum_t frames[sig][t][s - t*hop + n/2] /
// sum_t w^2, ascending t; 0 where the envelope is <= 1e-12.
struct OlaArgs {
    const float *frames;
    const float *window;
    int T, n_fft, hop, length;
    float *out;            // [sig][out_pitch]
    int64_t out_pitch;
};

static __global__ __launch_bounds__(256) void ola_kernel(OlaArgs a) {
    const int sig = (int)blockIdx.y;
    const int s = (int)(blockIdx.x * 256 + threadIdx.x);
    if (s >= a.length) return;
    const int half = a.n_fft / 2;
    // frames t with 0 <= s - (t*hop - half) < n_fft
    int t_lo = s + half - a.n_fft + 1;
    t_lo = t_lo <= 0 ? 0 : (t_lo + a.hop - 1) / a.hop;
    int t_hi = (s + half) / a.hop;
    if (t_hi > a.T - 1) t_hi = a.T - 1;
    float acc = 0.0f, norm = 0.0f;
    const float *fr = a.frames + (size_t)sig * a.T * a.n_fft;
    for (int t0 = t_lo; t0 <= t_hi; t0 += DSP_UNROLL) {
        float fv[DSP_UNROLL], wv[DSP_UNROLL];
#pragma unroll
        for (int u = 0; u < DSP_UNROLL; u++) {
            const int t = t0 + u, i = s - t * a.hop + half;
            fv[u] = t <= t_hi ? fr[(size_t)t * a.n_fft + i] : 0.0f;
            wv[u] = t <= t_hi ? a.window[i] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < DSP_UNROLL; u++)  // ascending frame order, as the reference
            if (t0 + u <= t_hi) {
                acc += fv[u];
                norm += wv[u] * wv[u];
            }
    }
    a.out[(size_t)sig * a.out_pitch + s] = norm > 1.0e-12f ? acc / norm : 0.0f;
}

// Cross-fade of chunk outputs: chunks[k][C][chunk] -> out[C][length],
// out = sum_k w_k * y_k / sum_k w_k over the chunks covering each sample, in
// ascending k.  Fade-in over the first (chunk-step) samples of every chunk
// but the first, fade-out over the last (chunk-step) of every chunk but the
// last: w = (i + 0.5)/overlap and ((chunk - i) - 0.5)/overlap.
struct FadeArgs {
    const float *chunks;
    int count, chunk, step, C;
    int64_t length;
    float *out;
    const float *mix;    // input audio [C][length] (for the instrumental)
    float *instrumental; // may be null
};

VH_DEVICE float fade_weight(int i, int k, int count, int chunk, int step) {
    const int overlap = chunk - step;
    float v = 1.0f;
    if (k > 0 && i < overlap) v = ((float)i + 0.5f) / (float)overlap;
    if (k + 1 < count && i >= chunk - overlap) v = ((float)(chunk - i) - 0.5f) / (float)overlap;
    return v;
}

static __global__ __launch_bounds__(256) void crossfade_kernel(FadeArgs a) {
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int c = (int)blockIdx.y;
    if (s >= a.length) return;
    int k_hi = (int)(s / a.step);
    if (k_hi > a.count - 1) k_hi = a.count - 1;
    int64_t lo = s - a.chunk + 1;
    int k_lo = lo <= 0 ? 0 : (int)((lo + a.step - 1) / a.step);
    float acc = 0.0f, ws = 0.0f;
    for (int k = k_lo; k <= k_hi; k++) {
        const int i = (int)(s - (int64_t)k * a.step);
        const float w = fade_weight(i, k, a.count, a.chunk, a.step);
        acc += w * a.chunks[((size_t)k * a.C + c) * a.chunk + i];
        ws += w;
    }
    const float v = acc / ws;
    a.out[(size_t)c * a.length + s] = v;
    if (a.instrumental) a.instrumental[(size_t)c * a.length + s] = a.mix[(size_t)c * a.length + s] - v;
}

// instrumental = mix - vocals (native/vocalarc_separation.c:1589-1591)
static __global__ __launch_bounds__(256) void subtract_kernel(const float *__restrict__ mix,
                                                              const float *__restrict__ vocals,
                                                              float *__restrict__ inst, int64_t n) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e < n) inst[e] = mix[e] - vocals[e];
}

}  // namespace vh

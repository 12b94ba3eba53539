// The band split in one pass (native/vocalarc_separation.c:887-912): a
// workgroup takes RT spectrogram rows of one band, gathers their bins from the
// spectrum, RMSNorms them, splits them into fp16 pieces in LDS and multiplies
// them with the band's weight pieces on the fp16 matrix cores (three piece
// products per fp32 product, gemm_h2.hpp), all output features at once.  The
// normalised band inputs never reach memory, and no call uploads a table.
//
// Bound by writing the features: 4 D bytes per row and band (571 MB for 60 s at
// D = 384, against 98 MB read and 57 GFLOP of piece products).  Gathering into
// memory and a batched fp32 MFMA GEMM took 144 + 367 us for those 6001 rows; this
// kernel 260, one launch per class of padded inputs (44 bands of 8-48 inputs 120,
// 16 of 96 and 192 98, two of 512 and 516 42; the narrow ones in the launch of
// the middle ones 220 + 47).  Rows per workgroup: 64 up to 192 inputs, so that a
// band's pieces are read once per 98 KB written; 32 and four waves up to 64
// inputs, 10 KB of LDS, so that many workgroups' gathers are in flight; 32 up to
// 528, where 64 rows would not leave two workgroups' worth of LDS; up to 640
// inputs 32 rows take 82 KB, one workgroup per CU.
//
// Precision: 22 bits of each operand, the products exact, their sums in fp32
// over 16 inputs at a time.  2-norm error against 64 bits 1.9e-7 where the fp32
// MFMA GEMM has 2.7e-7 (normal spectra, audio, pure tones, bins over six
// decades; both models).  Where a row has a single nonzero bin, so that nothing
// is summed, the operands show: 1.07e-7 against 6.7e-8.
//
// Rows stay in LDS as h2 rows (h2.hpp) made in place of the gathered fp32
// values, pitch 16 bytes over a multiple of 64 so that lanes reading one chunk
// of consecutive rows touch distinct banks.
#pragma once

#include "runtime.hpp"

#include "gemm_h2.hpp"

namespace vh {

struct BandSplitDesc {
    const void *W;       // pieces of [D][kpad] (columns past the band's zero)
    const float *gamma;  // [kpad], zero past the band's inputs
    const float *bias;   // [D]
    int first_freq, width;
    int kpad;  // the band's inputs 2 C width rounded up to 16
    int ea;    // h2_exponent of the bound sqrt(K) max|gamma| on a normalised row's elements
};

struct BandSplitArgs {
    const float *source;
    SpecLayout lay;
    const BandSplitDesc *bands;
    const int *list;  // the launch's bands
    int count;
    float *out;  // band b's row m at out + b * band_stride + m * ldo
    int64_t band_stride, ldo;
    int M, T, C, D;
};

// RT rows, KMAX padded inputs at most, J column tiles at a time per wave,
// BS_BATCH gather loads in flight per thread (enough for a tile's bins at once
// up to 528 inputs: a tile waits on memory once).
template <int RT, int KMAX, int J, int BS_THREADS, int BS_BATCH>
__global__ __launch_bounds__(BS_THREADS, BS_THREADS == 256 ? 3 : 4) void band_split_kernel(BandSplitArgs a) {
    static_assert(RT == 32 || RT == 64, "one or two 32-row blocks");
    constexpr int PARTS = BS_THREADS / RT;
    __shared__ __attribute__((aligned(16))) unsigned char rows[RT * (KMAX * 4 + 16)];
    __shared__ float part[PARTS][RT];
    __shared__ float rinv[RT];
    // a row tile's bands on one XCD: they share the spectrum's cache lines
    const int id = xcd_swizzle((int)blockIdx.x, (int)gridDim.x);
    const int b = a.list[id % a.count];
    const int m0 = id / a.count * RT;
    const BandSplitDesc d = a.bands[b];
    const int tid = (int)threadIdx.x;
    const int pitch = d.kpad * 4 + 16;
    const int pairs = d.width * a.C;

    // wave: 32 of the rows and, of the column tiles of 32, every CG-th
    constexpr int RB = RT / 32, CG = BS_THREADS / 64 / RB;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const int r0 = 32 * (wave % RB);
    const int nct = (a.D + 31) / 32, nk = d.kpad / GS_BK;
    const int eu = -(d.ea + h2_exponent(*static_cast<const float *>(d.W)));
    const char *const planes = static_cast<const char *>(d.W) + H2_HEADER;
    const char *wp[J];
    float bias[J];
    halfx8 wh[J], wm[J];
    auto fetch = [&](int k, halfx8 (&h)[J], halfx8 (&m)[J]) {
#pragma unroll
        for (int j = 0; j < J; j++) {
            h[j] = *reinterpret_cast<const halfx8 *>(wp[j] + k * (H2_WBLOCK * 2));
            m[j] = *reinterpret_cast<const halfx8 *>(wp[j] + k * (H2_WBLOCK * 2) + GS_BN * GS_BK * 2);
        }
    };
    // the column tiles ct0, ct0 + CG, ...: their biases and first pieces
    auto begin = [&](int ct0) {
#pragma unroll
        for (int j = 0; j < J; j++) {
            const int n = 32 * min(ct0 + CG * j, nct - 1), r = n % GS_BN + li;  // past the last tile: not stored
            wp[j] = planes + (size_t)(n / GS_BN) * nk * (H2_WBLOCK * 2) + r * 32 + 16 * (lh ^ ((r >> 3) & 1));
            bias[j] = n + li < a.D ? d.bias[n + li] : 0.0f;
        }
        fetch(0, wh, wm);
    };
    if (wave / RB < nct) begin(wave / RB);  // on their way while the rows are gathered

    // gather: consecutive threads along the spectrum's contiguous direction
    const int ch0 = m0 / a.T, t0 = m0 - ch0 * a.T;
    const bool f_fast = a.lay.f_s == 1;
    for (int i0 = 0; i0 < RT * pairs; i0 += BS_THREADS * BS_BATCH) {
        float2 v[BS_BATCH];
        int at[BS_BATCH];
#pragma unroll
        for (int u = 0; u < BS_BATCH; u++) {
            const int i = i0 + tid + BS_THREADS * u;
            at[u] = -1;
            if (i < RT * pairs) {
                int row, f, c;
                if (f_fast) {
                    const int q = i / d.width;
                    f = i - q * d.width;
                    row = q / a.C;
                    c = q - row * a.C;
                } else {
                    row = i % RT;
                    f = i / RT / a.C;
                    c = i / RT - f * a.C;
                }
                int t = t0 + min(row, a.M - 1 - m0), ch = ch0;
                while (t >= a.T) {
                    t -= a.T;
                    ch++;
                }
                at[u] = row * pitch + (f * a.C + c) * 8;
                v[u] = *reinterpret_cast<const float2 *>(a.source + 2 * spec_at(a.lay, ch, d.first_freq + f, c, t));
            }
        }
#pragma unroll
        for (int u = 0; u < BS_BATCH; u++)
            if (at[u] >= 0) *reinterpret_cast<float2 *>(rows + at[u]) = v[u];
    }
    const int pad = d.kpad - 2 * pairs;  // even
    for (int i = tid; i < RT * (pad / 2); i += BS_THREADS) {
        const int row = i % RT, p = i / RT;
        *reinterpret_cast<float2 *>(rows + row * pitch + (pairs + p) * 8) = make_float2(0.0f, 0.0f);
    }
    __syncthreads();

    const int row = tid % RT, pt = tid / RT;
    unsigned char *const rp = rows + row * pitch;
    float ss = 0.0f;
    for (int k = pt; k < nk; k += PARTS) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const floatx4 x = *reinterpret_cast<const floatx4 *>(rp + 64 * k + 16 * q);
#pragma unroll
            for (int e = 0; e < 4; e++) ss = fmaf(x[e], x[e], ss);
        }
    }
    part[pt][row] = ss;
    __syncthreads();
    if (tid < RT) {
        float s = 0.0f;
#pragma unroll
        for (int p = 0; p < PARTS; p++) s += part[p][tid];
        rinv[tid] = sqrtf((float)(2 * pairs)) / sqrtf(s + 1.0e-12f);
    }
    __syncthreads();
    {
        const float inv = rinv[row], scale = ldexpf(1.0f, d.ea);
        for (int k = pt; k < nk; k += PARTS) {
            floatx4 y[4];
#pragma unroll
            for (int q = 0; q < 4; q++)
                y[q] = (*reinterpret_cast<const floatx4 *>(rp + 64 * k + 16 * q) * inv) * ld4(d.gamma + 16 * k + 4 * q);
            halfx8 h0, m0_, h1, m1;
            split8_h2(y[0], y[2], scale, h0, m0_);
            split8_h2(y[1], y[3], scale, h1, m1);
            *reinterpret_cast<halfx8 *>(rp + 64 * k) = h0;
            *reinterpret_cast<halfx8 *>(rp + 64 * k + 16) = h1;
            *reinterpret_cast<halfx8 *>(rp + 64 * k + 32) = m0_;
            *reinterpret_cast<halfx8 *>(rp + 64 * k + 48) = m1;
        }
    }
    __syncthreads();

    const unsigned char *const ar = rows + (r0 + li) * pitch + 16 * lh;
    float *const out = a.out + (int64_t)b * a.band_stride + (int64_t)(m0 + r0) * a.ldo;
    for (int ct0 = wave / RB; ct0 < nct; ct0 += CG * J) {
        if (ct0 != wave / RB) begin(ct0);
        floatx16 acc[J];
#pragma unroll
        for (int j = 0; j < J; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[j][r] = 0.0f;
        // the pieces of chunk k + 1 are on their way while chunk k is
        // multiplied (the last chunk's are read twice)
        for (int k = 0; k < nk; k++) {
            halfx8 nh[J], nm[J];
            fetch(min(k + 1, nk - 1), nh, nm);
            const halfx8 ah = *reinterpret_cast<const halfx8 *>(ar + 64 * k);
            const halfx8 am = *reinterpret_cast<const halfx8 *>(ar + 64 * k + 32);
#pragma unroll
            for (int j = 0; j < J; j++) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(am, wh[j], acc[j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < J; j++) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, wm[j], acc[j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < J; j++) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, wh[j], acc[j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < J; j++) {
                wh[j] = nh[j];
                wm[j] = nm[j];
            }
        }
#pragma unroll
        for (int j = 0; j < J; j++) {
            const int col = 32 * (ct0 + CG * j) + li;
            if (col >= a.D) continue;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = 8 * (r >> 2) + 4 * lh + (r & 3);
                if (m0 + r0 + m < a.M)
                    __builtin_nontemporal_store(ldexpf(acc[j][r], eu) + bias[j], out + (int64_t)m * a.ldo + col);
            }
        }
    }
}

}  // namespace vh

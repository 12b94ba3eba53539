// fp32 token-wise linear on fp16 matrix cores by two-piece operand splitting:
// C[M][N] (op)= A[M][K] * W[N][K]^T with fp32 inputs, fp32 accumulation and
// the fused epilogues of the fp32 GEMM (gemm.hpp).  The default fp32 path's
// transformer and mask-estimator linears.
//
// Splitting.  Each operand is first scaled by a power of two 2^e (exact), so
// that everything it can hold lies below 2^14; then every scaled value y is
// split into two fp16 values (round to nearest even)
//   h = fp16(y),  m = fp16(y - h)
// y - h is exact in fp32 (Sterbenz) and |m| <= 2^-11 |y|, so h + m carries 22
// significant bits; where m is an fp16 subnormal (|y| < 2^-3, i.e. below
// 2^-17 of the operand's bound) the pair is exact to 2^-25 absolute.  The
// kernel accumulates the three products hh, hm, mh -- each exact in fp32
// (11 x 11 bits) -- and drops mm (<= 2^-22 |a||w|) and the pieces' rounding
// (<= 2^-22 each): per product term about 2^-21 relative, which the fp32
// accumulation over K (16 terms per MFMA, K/16 x 3 roundings) already
// exceeds.  Measured against fp64 on the transformer shapes, the result is
// 1.5-2 dB more accurate than the three-piece bf16 split (gemm_split.hpp,
// six products) and as accurate as a sequential fp32 FMA chain, at half its
// matrix-core work.
//
// Scales.  W's exponent comes from its absolute maximum, found on the device
// when the pieces are made and kept in their 256-byte header.  A's comes
// from a bound the caller supplies -- a value or a device float -- that every
// |A| element respects; the model derives exact bounds from the producers'
// weights (operand_bounds_kernel): an RMSNorm output obeys
// |y_i| <= ||y||_2 <= sqrt(D) max|gamma|, a linear of it obeys
// |W y + b|_n <= sqrt(D) max|gamma| ||W_n||_2 + |b_n|, an attention output
// (a convex combination of value rows times a gate in (0, 1)) obeys the
// value bound, a GELU-GLU output the square of its pre-activation bound
// (|gelu(g)| <= |g|), a tanh output 1.  The bound only has to hold: a loose
// one costs precision only for elements more than 2^17 below it.
//
// Block tiles (H2Tile) of 256x128 and 128x128 (waves of 32x128) where a launch
// fills the chip's 256 CUs several times over, of 64x128 and 64x64 where it
// does not (the launcher's rule says which; all give the same bits).
// Operands and pipeline as gemm_split.hpp (for 256x128: 8 waves of 32x128,
// K chunks of 16 in a global->LDS DMA ring, A fp32 in LDS split by each wave
// in registers, or h2 rows read as they are): W's pieces are two fp16 planes
// per tile-major block (8 KB per 128 rows x 16 k, the same row/slot
// permutation), one 1 KB load per wave per chunk; a 3-chunk ring (two chunks
// in flight while one is multiplied: 72 KB of LDS, two workgroups per CU;
// 0-2.4% faster than two chunks, bit-identical); per wave and chunk 12 MFMAs
// (v_mfma_f32_32x32x16_f16) and, for fp32 A, 4 VALU per A value for the scale
// and split.
#pragma once

#include "attention.hpp"
#include "gemm_split.hpp"
#include "h2.hpp"

namespace vh {

struct GemmDescH2 {
    const float *A;  // fp32 [M][lda]
    const void *W;   // pieces (split_weight_h2_kernel): 256-byte header, then the planes
    const float *bias;
    float *C;
    int M, N, K;
    int lda, ldc;
    // Null for none.  zero_slot: a device float the kernel sets to 0 (the bound
    // slot a later residual GEMM raises); amax: raised to max |C| by the
    // residual epilogue (gemm_bf16_epilogue).
    float *zero_slot;
    float *amax;
    // kv_inner > 0: C holds a fused q|k|v|gates projection with k in columns
    // [kv_inner, 2 kv_inner) and v in [2 kv_inner, 3 kv_inner); those are
    // written times 2^ek and 2^ev (att_h2_exponents of *kv_bound), the scales
    // the fp16 two-piece attention would otherwise apply as it stages them
    const float *kv_bound;
    int kv_inner;
    // kv_pieces (with kv_inner): k, rotated, and v are written as the fp16
    // pieces of those scaled values (kv_pieces_epilogue), the rotary position
    // of row r being (r / rope_period) % rope_len -- rope_period >= 32: rows
    // ordered [chunk][position][sequence], rope_period sequences per position
    // (the time axis of [chunk][frame][band], the band axis of [band][frame]);
    // 1: consecutive rows are consecutive positions, rope_len >= 32 of them --
    // its (cos, sin) at rope[(position * 32 + pair) * 2]
    int kv_pieces;
    const float *rope;
    int rope_period, rope_len;
    // EPI_MASK_GLU: the band's first frequency and its inputs
    int mask_f0, mask_dim;
};
// EPI_MASK_GLU: where the mask goes.
struct H2MaskOut {
    float *mask;
    SpecLayout lay;
    int T, C;
};

// The mask estimator's GLU and bin scatter on a wave's 32 x 32 NJ tile of its
// second layer, whose columns come in (16 value, 16 gate) groups.  Of two
// accumulator rows r, r + 1 v_permlane16_swap leaves the values of r in lanes
// 0-15 and of r + 1 in lanes 16-31 of one register, their gates in the other:
// every lane then holds one output.  The projection (twice the mask's bytes)
// is no longer written, read back and scattered by a pass of its own (36 us of
// 474 on an 8 s window).
template <int NJ>
VH_DEVICE void mask_glu_epilogue(const GemmDescH2 &d, const H2MaskOut &o, int row0, int col0, int li, int lh,
                                 const floatx16 (&acc)[1][NJ], const float *bpre) {
    const int ch0 = row0 / o.T, t0 = row0 - ch0 * o.T;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int i = (col0 + 32 * j) / 2 + (li & 15);
        const int pair = i >> 1, f = pair / o.C, c = pair - f * o.C;
        const int64_t at = spec_at(o.lay, 0, d.mask_f0 + f, c, 0);
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
            typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
            const u32x2 vg = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[0][j][r] + bpre[j]),
                                                              __float_as_uint(acc[0][j][r + 1] + bpre[j]), false, false);
            const float v = __uint_as_float(vg[0]) * sigmoid_dev(__uint_as_float(vg[1]));
            const int off = 8 * (r >> 2) + 4 * lh + (r & 3) + (li >> 4);
            int t = t0 + off, ch = ch0;
            while (t >= o.T) {
                t -= o.T;
                ch++;
            }
            if (i < d.mask_dim && row0 + off < d.M)
                o.mask[2 * (at + ch * o.lay.chunk_s + t * o.lay.t_s) + (i & 1)] = v;
        }
    }
}


// The fused projection's k or v column tile (32 x 32 NJ per wave, n0 inside
// [kv_inner, 3 kv_inner)) written as fp16 pieces instead of fp32: the head's
// 64 columns of a row occupy its 256 bytes of the region -- 64 h halves, then
// 64 m halves, dim order -- where h + m is the value y scaled by 2^ek (2^ev),
// h = fp16(y), m = fp16(y - h) (exact difference): the pieces the two-piece
// attention's staging forms, so the attention copies them into LDS as they
// are.  k is rotated first (rope_own: each lane swaps its value with the
// lane of the pair's other dimension), by the (cos, sin) of the row's
// position; a wave's 32 consecutive rows span at most two positions, or
// (rope_period 1) 32 of them, whose entries the lane loads four rows at a
// time (cache hits; eight at a time took the kernel past 128 VGPRs).  Each value is first
// formed as the plain epilogue forms it: acc times the row's norm scale plus
// the bias in one fused multiply-add.
// tv: the rotary table entry (cos, sin) of position f0 (lanes 0-31) or f1
// (lanes 32-63) and pair lane % 32, loaded before the K loop (k tiles only,
// rope_period > 1).
// Stores.  A register quad holds four consecutive rows of the lane's column:
// the four lanes of a quad swap halves (transpose4_f16) so that each holds
// four consecutive columns of one row, and the wave lays a head's two column
// tiles out in LDS (its own part of the ring, which the K loop no longer reads)
// to leave as 16-byte stores of whole 256-byte rows.  Stored from registers the
// two tiles each wrote 64 bytes of every 128-byte line, in 2-byte (248 us) or
// 8-byte (276) pieces, against 243 now (an 8 s window's QKV GEMM, 49662 x 1568 x
// 384 on consecutive rows; eight windows' time axis 1694 -> 1655).
VH_DEVICE uint32_t dpp_quad_xor1(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false);
}
VH_DEVICE uint32_t dpp_quad_xor2(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, false);
}
typedef uint32_t kvp_u32x2 __attribute__((ext_vector_type(2)));
// a: fp16 rows 0 (low half) and 1 of the lane's column, b: rows 2 and 3; the
// result: row lane % 4, columns 0-3 of the lane's quad.
VH_DEVICE kvp_u32x2 transpose4_f16(uint32_t a, uint32_t b, int quad) {
    const uint32_t sel = quad & 1 ? 0x03020706u : 0x05040100u;
    const uint32_t ca = __builtin_amdgcn_perm(dpp_quad_xor1(a), a, sel);  // row quad & 1, the lane pair's columns
    const uint32_t cb = __builtin_amdgcn_perm(dpp_quad_xor1(b), b, sel);  // row 2 + (quad & 1)
    const uint32_t got = dpp_quad_xor2(quad & 2 ? ca : cb);
    return quad & 2 ? kvp_u32x2{got, cb} : kvp_u32x2{ca, got};
}
template <int NJ>
VH_DEVICE void kv_pieces_epilogue(const GemmDescH2 &d, int row0, int n0, int li, int lh, float2 tv,
                                  const floatx16 (&acc)[1][NJ], floatx16 rs, floatx4 bpre, unsigned char *stage) {
    const bool is_k = n0 < 2 * d.kv_inner;
    const int region = is_k ? d.kv_inner : 2 * d.kv_inner;  // first column of the k (v) region
    const int quad = li & 3, lane = 32 * lh + li;
    const bool even = (li & 1) == 0;
    // column tiles per pass (a head's two, or the wave's one), the bytes of a
    // row's h or m piece of them and of a staged row, 16-byte slots per row
    constexpr int TP = NJ >= 2 ? 2 : 1, PIECE = 64 * TP, SPITCH = 2 * PIECE + 16, SLOTS = 2 * PIECE / 16;
    constexpr int RP = 64 / SLOTS;  // rows per store
    const float one = opaque_one();
    char *const rbase = reinterpret_cast<char *>(d.C) + (size_t)row0 * d.ldc * 4u;
    const uint32_t pitch = (uint32_t)d.ldc * 4u;
    const int p0 = row0 % d.rope_len;  // rope_period 1: the first row's position
    // rope_period > 1: first row (within the wave's 32) of the second position
    // the rows span; its table entries are those tv holds in lanes 32-63
    const int off_b = d.rope_period - row0 % d.rope_period;
    const int slot = lane % SLOTS, rsub = lane / SLOTS;
    // one pass at a time: nothing of the next is hoisted into this one (the
    // registers the K loop needs bound the epilogue's)
#pragma unroll
    for (int jb = 0; jb < NJ; jb += TP) {
        __builtin_amdgcn_sched_barrier(0);
        float y[TP][16];
#pragma unroll
        for (int jj = 0; jj < TP; jj++)
#pragma unroll
            for (int r = 0; r < 16; r++) y[jj][r] = fmaf(acc[0][jb + jj][r], rs[r], bpre[jb + jj]);
        if (is_k) {
#pragma unroll
            for (int jj = 0; jj < TP; jj++) {
                const int pr = ((n0 + 32 * (jb + jj) + li - region) & 63) >> 1;  // the lane's pair
                auto turn = [&](int r, float c, float sn) {
                    const float other =
                        __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(y[jj][r]), 0xB1, 0xF, 0xF, false));
                    y[jj][r] = rope_own(y[jj][r], other, c, even ? -sn : sn);
                };
                if (d.rope_period == 1) {
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        __builtin_amdgcn_sched_barrier(0);
                        float2 cs[4];
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            int p = p0 + 8 * q + 4 * lh + e;
                            if (p >= d.rope_len) p -= d.rope_len;
                            cs[e] = *reinterpret_cast<const float2 *>(d.rope + 2 * (p * 32 + pr));
                        }
#pragma unroll
                        for (int e = 0; e < 4; e++) turn(4 * q + e, cs[e].x, cs[e].y);
                    }
                } else {
                    // the pair's entries from the lanes holding them
                    const float c0 = __shfl(tv.x, pr, 64), s0 = __shfl(tv.y, pr, 64);
                    const float c1 = __shfl(tv.x, 32 + pr, 64), s1 = __shfl(tv.y, 32 + pr, 64);
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const bool nxt = 8 * (r >> 2) + 4 * lh + (r & 3) >= off_b;
                        turn(r, nxt ? c1 : c0, nxt ? s1 : s0);
                    }
                }
            }
        }
#pragma unroll
        for (int jj = 0; jj < TP; jj++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                __builtin_amdgcn_sched_barrier(0);
                // rows in pairs: one v_cvt_pk_f16_f32 makes both h, one
                // v_fma_mix_f32 per value and one v_cvt_pk_f16_f32 both m
                const float *v = &y[jj][4 * q];
                const uint32_t ha = pack_f16x2(v[0], v[1]), hb = pack_f16x2(v[2], v[3]);
                const uint32_t ma = m_pair_f16(v[0], v[1], one, ha), mb = m_pair_f16(v[2], v[3], one, hb);
                unsigned char *const at = stage + (8 * q + 4 * lh + quad) * SPITCH + 64 * jj + 2 * (li & ~3);
                *reinterpret_cast<kvp_u32x2 *>(at) = transpose4_f16(ha, hb, quad);
                *reinterpret_cast<kvp_u32x2 *>(at + PIECE) = transpose4_f16(ma, mb, quad);
            }
        // the wave's own LDS operations complete in order
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int kc = n0 + 32 * jb - region;
        const uint32_t off = 4u * (uint32_t)region + 256u * (uint32_t)(kc >> 6) + 2u * (uint32_t)(kc & 63) +
                             (slot < SLOTS / 2 ? 16u * (uint32_t)slot : 128u + 16u * (uint32_t)(slot - SLOTS / 2)) +
                             (uint32_t)rsub * pitch;
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int i = 0; i < 32 / RP; i++) {
            if (i % 2 == 0) __builtin_amdgcn_sched_barrier(0);  // two reads in flight
            const u32x4 v = *reinterpret_cast<const u32x4 *>(stage + (RP * i + rsub) * SPITCH + 16 * slot);
            if (row0 + RP * i + rsub < d.M)
                __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(rbase + (uint32_t)(RP * i) * pitch + off));
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}
// Bound on |A|: *ptr when ptr is set (a device float), else value.
struct H2Bound {
    const float *ptr;
    float value;
};

// A workgroup's tile: WR x WC waves of 32 rows x 32 NJ_ columns; a ring of
// RING_ stages in LDS, each KS_ chunks of 16 of K, RING_ - 1 of them in flight
// while one is multiplied; OCC_ waves per SIMD the register count must allow.
template <int WR, int WC_, int NJ_, int KS_, int RING_, int OCC_>
struct H2Tile {
    static constexpr int WC = WC_, NJ = NJ_, KS = KS_, RING = RING_, OCC = OCC_;
    static constexpr int WAVES = WR * WC, THREADS = 64 * WAVES;
    static constexpr int BM = 32 * WR, BN = 32 * NJ * WC;
    static_assert(BN <= GS_BN && GS_BN % BN == 0, "a tile's columns lie in one 128-row tile of the pieces");
};
using H2Tile256 = H2Tile<8, 1, 4, 1, 3, 4>;  // 256 x 128, 72 KB LDS: two workgroups per CU
using H2Tile128 = H2Tile<4, 1, 4, 1, 3, 3>;  // 128 x 128, 48 KB: three
// The small tiles take K 32 at a time (half the barriers: at one wave of work
// per SIMD between them, they and the LDS latency are the time), which leaves
// room for one stage in flight (a third stage, fewer workgroups per CU: +3-10%).
using H2Tile64 = H2Tile<2, 2, 2, 2, 2, 3>;   // 64 x 128, 48 KB: three
using H2Tile64n = H2Tile<2, 2, 1, 2, 2, 4>;  // 64 x 64, 32 KB: five

constexpr int H2_HEADER = 256;                // bytes before the planes: float max|W|
constexpr int H2_WBLOCK = 2 * GS_BN * GS_BK;  // fp16 per (row tile, K chunk) block of W pieces

// A_H2: A arrives as h2 rows (h2.hpp) scaled by 2^h2_exponent(a_bound) -- its
// producer split it -- and the K loop only reads the pieces.
// T: the block tile (H2Tile).  Every tile forms each output by the same
// products in the same order: the results are the same bits.
// NORM (fp32 A): the GEMM of an RMSNorm of A's rows, W holding the norm's gain
// folded in (W[n][k] gamma[k]): each accumulator row is multiplied by its row's
// sqrt(K) / sqrt(sum_k A^2 + 1e-12) (the RMSNorm kernels' expression), the
// sum taken from the fp32 values the K loop splits anyway, before bias and
// activation.  So the normalised rows are never written: the RMSNorm pass and
// its 2 x 4 bytes per element of traffic go, and A is the residual stream
// itself, bounded by the max |x| its producer's epilogue recorded.
// KVS: the k and v columns scaled (GemmDescH2::kv_inner), compiled only into
// the fused projection's instantiations, and with kv_pieces written as their
// fp16 pieces (k rotated).
template <int EPI, bool A_H2, class T, bool NORM = false, bool KVS = false>
__device__ __forceinline__ void gemm_h2_body(const GemmDescH2 &d, float a_bound, int tile,
                                             const H2MaskOut *mo = nullptr) {
    static_assert(!(NORM && A_H2), "the row norm needs the fp32 rows");
    static_assert(EPI != EPI_GEGLU || T::NJ % 2 == 0, "a wave holds the value and the gate columns");
    constexpr int NJW = T::NJ, RING = T::RING, KS = T::KS;
    constexpr int A_BYTES = T::BM * GS_BK * 4;  // fp32 rows of 64 B
    constexpr int P_BYTES = T::BN * GS_BK * 2;  // per W plane: fp16 rows of 32 B
    constexpr int SUB_BYTES = A_BYTES + 2 * P_BYTES;
    constexpr int STAGE_BYTES = KS * SUB_BYTES;
    // 1 KB loads of A and W per wave and chunk
    constexpr int UA = T::BM / 16 / T::WAVES, UW = T::BN / 16 / T::WAVES;
    static_assert(UA * T::WAVES * 16 == T::BM && UW * T::WAVES * 16 == T::BN, "whole 1 KB loads per wave");
    constexpr int LOADS = KS * (UA + UW);  // per wave and stage
    __shared__ __attribute__((aligned(1024))) unsigned char ring[RING * STAGE_BYTES];

    const int tiles_n = (d.N + T::BN - 1) / T::BN;
    const int tiles_m = (d.M + T::BM - 1) / T::BM;
    if (d.zero_slot && tile == 0 && threadIdx.x == 0) *d.zero_slot = 0.0f;
    if (tile >= tiles_m * tiles_n) return;
    // column-fastest order within groups of row tiles (see gemm.hpp)
    // groups of 1024 rows for the wide GEMMs (256-row tiles: 4 measured
    // against 1, 2, 8, 16, best by 0.3-1.3% on N = 1568 and 3072), one row
    // tile for N = 384
    const int gsz = d.N >= 1024 ? 1024 / T::BM : 1;
    const int group = tile / (gsz * tiles_n);
    const int in_group = tile % (gsz * tiles_n);
    const int group_rows = min(gsz, tiles_m - group * gsz);
    const int m0 = (group * gsz + in_group % group_rows) * T::BM;
    const int n0 = (in_group / group_rows) * T::BN;

    const int ea = h2_exponent(a_bound);
    const int ew = h2_exponent(*static_cast<const float *>(d.W));
    const float a_scale = ldexpf(1.0f, ea);

    const int tid = (int)threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const int wr = wave / T::WC, wc = wave % T::WC;  // the wave's 32 rows and 32 NJ columns
    const int row0 = m0 + 32 * wr, col0 = n0 + 32 * NJW * wc;
    const uint32_t ring_base = (uint32_t)(uintptr_t)ring;
    auto swz_a = [](int r) { return (r >> 2) & 3; };
    auto swz_w = [](int r) { return (r >> 3) & 1; };

    // the bias of the lane's column in each 32-column tile (0 past N), loaded
    // before the K loop so that its latency is spent there, not in the
    // epilogue
    float bpre[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < NJW; j++) {
        const int col = col0 + 32 * j + li;
        bpre[j] = d.bias && col < d.N ? d.bias[col] : 0.0f;
    }
    // each 32-column tile's extra power of two: ek for k columns, ev for v
    // (kv_inner is a multiple of 32, so a tile is all q, k, v or gates)
    int ekv[4] = {0, 0, 0, 0};
    if (KVS && d.kv_inner > 0) {
        int ek, eq, ev;
        att_h2_exponents(*d.kv_bound, 1.0f, ek, eq, ev);
#pragma unroll
        for (int j = 0; j < NJW; j++) {
            const int c = col0 + 32 * j;
            ekv[j] = c < d.kv_inner ? 0 : c < 2 * d.kv_inner ? ek : c < 3 * d.kv_inner ? ev : 0;
        }
    }

    // A: 1 KB loads of 16 rows each, wave w loads blocks w, w + WAVES, ...
    // from the tile's first row (scalar base) plus its lane offset (below
    // 2^32: at most 256 rows of lda <= 2^21 floats).  W: the tile's rows of
    // each plane of the chunk's 128-row tile-major image, consecutive there:
    // blocks w, w + WAVES, ... of 1 KB, the h plane's first.
    const float *a_base = d.A + (size_t)m0 * d.lda;
    uint32_t a_voff[UA];
#pragma unroll
    for (int j = 0; j < UA; j++) {
        const int r = 16 * (wave + T::WAVES * j) + (lane >> 2);
        a_voff[j] = (uint32_t)(min(m0 + r, d.M - 1) - m0) * (uint32_t)d.lda * 4u + 16u * ((lane & 3) ^ swz_a(r));
    }
    const _Float16 *w_base = reinterpret_cast<const _Float16 *>(static_cast<const char *>(d.W) + H2_HEADER) +
                             (size_t)(n0 / GS_BN) * (d.K / GS_BK) * H2_WBLOCK + (n0 % GS_BN) * GS_BK;
    const uint32_t w_voff = 16 * lane;
    auto issue = [&](int st) {
#pragma unroll
        for (int u = 0; u < KS; u++) {
            const int kt = st * KS + u;
            const uint32_t sb = ring_base + (st % RING) * STAGE_BYTES + u * SUB_BYTES;
            const float *ab = a_base + kt * GS_BK;
#pragma unroll
            for (int j = 0; j < UA; j++) lds_dma16s(a_voff[j], ab, sb + (wave + T::WAVES * j) * 1024);
#pragma unroll
            for (int j = 0; j < UW; j++) {
                const int i = wave + T::WAVES * j;
                const int plane = i / (T::BN / 32), blk = i % (T::BN / 32);
                lds_dma16s(w_voff, w_base + (size_t)kt * H2_WBLOCK + plane * (GS_BN * GS_BK) + blk * 512,
                           sb + A_BYTES + i * 1024);
            }
        }
    };

    floatx16 acc[1][NJW];
#pragma unroll
    for (int j = 0; j < NJW; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[0][j][r] = 0.0f;

    // k/v pieces: the rotary table entries the epilogue of a k tile needs,
    // loaded now so that their latency is spent in the K loop (two registers)
    float2 tv = make_float2(1.0f, 0.0f);
    if constexpr (KVS && EPI == EPI_STORE) {
        if (d.kv_pieces && d.rope_period > 1 && col0 >= d.kv_inner && col0 < 2 * d.kv_inner) {
            const int f0 = (row0 / d.rope_period) % d.rope_len;
            const int f = lane < 32 ? f0 : (f0 + 1 == d.rope_len ? 0 : f0 + 1);
            tv = *reinterpret_cast<const float2 *>(d.rope + 2 * (f * 32 + (lane & 31)));
        }
    }
    const int ns = d.K / (GS_BK * KS);  // stages (KS > 1: the launcher checked K)
    float ss = 0.0f;  // NORM: sum of squares of this lane's half of row 32 wr + li
#pragma unroll
    for (int i = 0; i < RING - 1; i++)
        if (i < ns) issue(i);
    // stage 0 has landed once at most the stages issued after it are in flight
    if (ns >= RING - 1) wait_vmcnt<LOADS *(RING - 2)>();
    else wait_vmcnt<0>();
    __syncthreads();
    // NJ live 32-column accumulators, chosen once per tile (as gemm_split_body)
    auto k_loop = [&](auto nj_c) {
        constexpr int NJ = decltype(nj_c)::value;
        for (int st = 0; st < ns; st++) {
            // stage st+RING-1 goes to the slot stage st-1 used: every wave
            // finished reading it before the barrier that ended the previous
            // iteration
            if (st + RING - 1 < ns) issue(st + RING - 1);
#pragma unroll
            for (int u = 0; u < KS; u++) {
                const unsigned char *sbuf = ring + (st % RING) * STAGE_BYTES + u * SUB_BYTES;
                const int r = wr * 32 + li;
                const unsigned char *ar = sbuf + r * 64;
                halfx8 ah, am;
                if constexpr (A_H2) {
                    ah = *reinterpret_cast<const halfx8 *>(ar + 16 * (lh ^ swz_a(r)));
                    am = *reinterpret_cast<const halfx8 *>(ar + 16 * ((2 + lh) ^ swz_a(r)));
                } else {
                    const floatx4 lo = *reinterpret_cast<const floatx4 *>(ar + 16 * (lh ^ swz_a(r)));
                    const floatx4 hi = *reinterpret_cast<const floatx4 *>(ar + 16 * ((2 + lh) ^ swz_a(r)));
                    split8_h2(lo, hi, a_scale, ah, am);
                    if constexpr (NORM) {
#pragma unroll
                        for (int e = 0; e < 4; e++) ss = fmaf(hi[e], hi[e], fmaf(lo[e], lo[e], ss));
                    }
                }
                // W column tiles two at a time: their pieces, then (m,h) (h,m) (h,h)
#pragma unroll
                for (int jp = 0; jp < (NJ + 1) / 2; jp++) {
                    constexpr int NJJ = NJ == 1 ? 1 : 2;
                    halfx8 wh[NJJ], wm[NJJ];
#pragma unroll
                    for (int jj = 0; jj < NJJ; jj++) {
                        const int rw = 32 * (NJW * wc + 2 * jp + jj) + li;
                        const unsigned char *wp = sbuf + A_BYTES + rw * 32 + 16 * (lh ^ swz_w(rw));
                        wh[jj] = *reinterpret_cast<const halfx8 *>(wp);
                        wm[jj] = *reinterpret_cast<const halfx8 *>(wp + P_BYTES);
                    }
#pragma unroll
                    for (int jj = 0; jj < NJJ; jj++)
                        acc[0][2 * jp + jj] =
                            __builtin_amdgcn_mfma_f32_32x32x16_f16(am, wh[jj], acc[0][2 * jp + jj], 0, 0, 0);
#pragma unroll
                    for (int jj = 0; jj < NJJ; jj++)
                        acc[0][2 * jp + jj] =
                            __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, wm[jj], acc[0][2 * jp + jj], 0, 0, 0);
#pragma unroll
                    for (int jj = 0; jj < NJJ; jj++)
                        acc[0][2 * jp + jj] =
                            __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, wh[jj], acc[0][2 * jp + jj], 0, 0, 0);
                }
            }
            // stage st+1 has landed (LOADS loads per wave and stage; later stages may fly)
            if (st + RING - 1 < ns) wait_vmcnt<LOADS *(RING - 2)>();
            else wait_vmcnt<0>();
            __syncthreads();
        }
    };
    if constexpr (T::WC == 1 && NJW == 4) {
        const int live = d.N - n0;
        if (live > 64) k_loop(std::integral_constant<int, 4>());
        else if (live > 32) k_loop(std::integral_constant<int, 2>());
        else k_loop(std::integral_constant<int, 1>());
    } else {
        k_loop(std::integral_constant<int, NJW>());
    }
    // both scales undone at once: acc 2^-(ea+ew) by one v_ldexp_f32 (exact, as
    // the two power-of-two multiplies it replaces were where their product
    // is a normal float, and correctly rounded where it is not)
    const int eu = -(ea + ew);
#pragma unroll
    for (int j = 0; j < NJW; j++) {
#pragma unroll
        for (int r = 0; r < 16; r++) acc[0][j][r] = ldexpf(acc[0][j][r], eu + ekv[j]);
        bpre[j] = ldexpf(bpre[j], ekv[j]);  // (acc + b) 2^e exactly, with the row norm too
    }
    float rs[16];  // NORM: the scale of each accumulator row, applied with the bias
    if constexpr (NORM) {
        // lanes li and li + 32 summed the two halves of row 32 wr + li;
        // register 4q + e of a lane holds row 8q + 4lh + e of the wave's 32
        __shared__ float rscale[T::WAVES][32];
        const float tot = ss + __shfl_xor(ss, 32, 64);
        if (lh == 0) rscale[wave][li] = sqrtf((float)d.K) / sqrtf(tot + 1.0e-12f);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const floatx4 r4 = *reinterpret_cast<const floatx4 *>(&rscale[wave][8 * q + 4 * lh]);
#pragma unroll
            for (int e = 0; e < 4; e++) rs[4 * q + e] = r4[e];
        }
    }
    if constexpr (KVS && EPI == EPI_STORE) {
        if (d.kv_pieces && col0 >= d.kv_inner && col0 < 3 * d.kv_inner) {
            // the plain epilogue's value of each element (bias and row norm in
            // one fused multiply-add), formed in place first so the row
            // scales and biases are dead before the rotation and the split
            // the row scales and biases as vector values (not arrays), which
            // keeps them in registers across the epilogue's variants
            floatx16 rsv;
#pragma unroll
            for (int r = 0; r < 16; r++) rsv[r] = NORM ? rs[r] : 1.0f;  // x 1 + b: one rounding, as x + b
            static_assert(RING * STAGE_BYTES / T::WAVES >= 32 * (128 * (NJW >= 2 ? 2 : 1) + 16), "staged rows");
            kv_pieces_epilogue<NJW>(d, row0, col0, li, lh, tv, acc, rsv, floatx4{bpre[0], bpre[1], bpre[2], bpre[3]},
                                    ring + wave * (RING * STAGE_BYTES / T::WAVES));
            return;
        }
    }
    if constexpr (EPI == EPI_MASK_GLU) {
        mask_glu_epilogue<NJW>(d, *mo, row0, col0, li, lh, acc, bpre);
        return;
    }
    GemmDescBF16 e{};
    e.bias = d.bias; e.C = d.C; e.M = d.M; e.N = d.N; e.K = d.K; e.ldc = d.ldc;
    float mx = 0.0f;
    gemm_bf16_epilogue<EPI, float, 1, NJW>(e, acc, row0, col0, li, lh, &mx, bpre, NORM ? rs : nullptr);
    if constexpr (EPI == EPI_RESIDUAL) {
        if (d.amax) {
            // one atomic per workgroup (one per wave, all on one address,
            // cost 17 us per launch of 4656 tiles); non-negative floats
            // order as their bit patterns
            __shared__ float wmax[T::WAVES];
            mx = wave_max(mx);
            if (lane == 0) wmax[wave] = mx;
            __syncthreads();
            if (tid == 0) {
#pragma unroll
                for (int w = 1; w < T::WAVES; w++) mx = fmaxf(mx, wmax[w]);
                atomicMax(reinterpret_cast<unsigned int *>(d.amax), __float_as_uint(mx));
            }
        }
    }
}

template <int EPI, bool A_H2, class T, bool NORM = false, bool KVS = false>
__global__ __launch_bounds__(T::THREADS, T::OCC) void gemm_h2_kernel(GemmDescH2 d, H2Bound b) {
    gemm_h2_body<EPI, A_H2, T, NORM, KVS>(d, b.ptr ? *b.ptr : b.value, xcd_swizzle((int)blockIdx.x, (int)gridDim.x));
}

// Ragged batch (the mask estimator's per-band linears): problem blockIdx.z,
// one bound for all problems; as kernel arguments, 64 bytes each, so that both
// models' bands fit one launch (the 90-band model's second launch waited for
// the whole of the first: its mask on 1 s 108 -> 77 us).
constexpr int H2_MAX_BATCH = 96;
struct GemmBatchItemH2 {
    const float *A;
    const void *W;
    const float *bias;
    float *C;
    int M, N, K, lda, ldc;
    int mask_f0, mask_dim;  // EPI_MASK_GLU
};
struct GemmBatchH2 {
    GemmBatchItemH2 d[H2_MAX_BATCH];
    H2Bound b;
    H2MaskOut mo;  // EPI_MASK_GLU
};

template <int EPI, class T>
__global__ __launch_bounds__(T::THREADS, T::OCC) void gemm_h2_batched_kernel(GemmBatchH2 b) {
    const GemmBatchItemH2 &i = b.d[blockIdx.z];
    GemmDescH2 d{};
    d.A = i.A; d.W = i.W; d.bias = i.bias; d.C = i.C;
    d.M = i.M; d.N = i.N; d.K = i.K; d.lda = i.lda; d.ldc = i.ldc;
    d.mask_f0 = i.mask_f0; d.mask_dim = i.mask_dim;
    gemm_h2_body<EPI, false, T>(d, b.b.ptr ? *b.b.ptr : b.b.value, (int)blockIdx.x, &b.mo);
}

// max |W| over W [N][ldw] (first K columns) into out[0]; one workgroup of
// 1024 threads, no atomics.
static __global__ __launch_bounds__(1024) void absmax_kernel(const float *__restrict__ W, int N, int K, int ldw,
                                                            float *__restrict__ out) {
    __shared__ float red[16];
    float mx = 0.0f;
    const int64_t n = (int64_t)N * K;
    for (int64_t i = threadIdx.x; i < n; i += 1024) mx = fmaxf(mx, fabsf(W[(i / K) * ldw + i % K]));
    mx = wave_max(mx);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; w++) mx = fmaxf(mx, red[w]);
        out[0] = mx;
    }
}

// max |W| over W [N][ldw] (first K columns) raised into *out, which the
// stream zeroed before (zero_float_kernel): grid-stride over the matrix, one
// atomic max per workgroup (non-negative floats order as their bit
// patterns).  The weights' maxima at model load: one workgroup per matrix
// took 83 us each, 25 ms for a 16-layer model's 309 matrices.
static __global__ __launch_bounds__(256) void absmax_rows_kernel(const float *__restrict__ W, int N, int K, int ldw,
                                                                 float *__restrict__ out) {
    __shared__ float red[4];
    float mx = 0.0f;
    const int64_t n = (int64_t)N * K;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        mx = fmaxf(mx, fabsf(W[(i / K) * ldw + i % K]));
    mx = wave_max(mx);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0)
        atomicMax(reinterpret_cast<unsigned int *>(out),
                  __float_as_uint(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]))));
}

static __global__ void zero_float_kernel(float *out) { *out = 0.0f; }

// Per-workgroup max |x| over x[n] (grid-stride, 256 threads) into
// partial[blockIdx.x]; absmax_kernel over the partials finishes the reduction.
static __global__ __launch_bounds__(256) void absmax_partial_kernel(const float *__restrict__ x, int64_t n,
                                                                   float *__restrict__ partial) {
    __shared__ float red[4];
    float mx = 0.0f;
    const int64_t n4 = ((uintptr_t)x & 15) ? 0 : n / 4;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)gridDim.x * 256) {
        const floatx4 v = ld4(x + 4 * i);
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
    }
    for (int64_t i = 4 * n4 + (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        mx = fmaxf(mx, fabsf(x[i]));
    mx = wave_max(mx);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// fp32 W [N][ldw_in] (K a multiple of 16) scaled by 2^h2_exponent(max|W|)
// (max|W| read from the header) -> its h, m fp16 pieces, tile-major: element
// (n, k) of piece p at H2_HEADER bytes plus, in fp16 units,
//   ((n/128 * K/16 + k/16) * 2 + p) * 2048 + (n%128) * 16 + 8 * (s ^ (n/8)%2) + e
// with slot s and element e from split_k_slot(k) % 16 = 8 s + e (the layout
// of split_weight_kernel with two planes).  Rows past N are zero.
static __global__ __launch_bounds__(256) void split_weight_h2_kernel(const float *__restrict__ W, int N, int K,
                                                                    int ldw_in, void *__restrict__ pieces) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int rows = (N + GS_BN - 1) / GS_BN * GS_BN;
    if (idx >= (int64_t)rows * K) return;
    const float s = ldexpf(1.0f, h2_exponent(*static_cast<const float *>(pieces)));
    const int n = (int)(idx / K), k = (int)(idx % K);
    _Float16 h = (_Float16)0.0f, m = (_Float16)0.0f;
    if (n < N) {
        const float y = W[(size_t)n * ldw_in + k] * s;
        h = (_Float16)y;
        m = (_Float16)(y - (float)h);
    }
    const int r = n % GS_BN, pos = split_k_slot(k) & 15;
    const int phys = (pos >> 3) ^ ((r >> 3) & 1);
    const size_t o = ((size_t)(n / GS_BN) * (K / GS_BK) + k / GS_BK) * H2_WBLOCK + (size_t)r * GS_BK + 8 * phys + (pos & 7);
    _Float16 *planes = reinterpret_cast<_Float16 *>(static_cast<char *>(pieces) + H2_HEADER);
    planes[o] = h;
    planes[o + GS_BN * GS_BK] = m;
}

// Bounds on the operands downstream of an RMSNorm with gain gamma[D]:
//   out[0] = sqrt(D) max|gamma|                  (|y_i| <= ||y||_2 <= out[0])
//   out[1] = t or t^2 (square), t = out[0] max_n ||W_n||_2 + max_n |b_n|
//            (a bound on every output of the linear W y + b, W [N][D]; its
//            square bounds a GELU-GLU of two such outputs); 0 without W.
// One workgroup of 1024 threads: one wave per row of W at a time.
static __global__ __launch_bounds__(1024) void operand_bounds_kernel(const float *__restrict__ gamma, int D,
                                                                    const float *__restrict__ W, int N,
                                                                    const float *__restrict__ b, int square,
                                                                    float *__restrict__ out) {
    __shared__ float red[2][16];
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float g = 0.0f, nrm = 0.0f, bm = 0.0f;
    for (int i = tid; i < D; i += 1024) g = fmaxf(g, fabsf(gamma[i]));
    if (W) {
        for (int n = wave; n < N; n += 16) {
            float ss = 0.0f;
            for (int k = lane; k < D; k += 64) ss = fmaf(W[(size_t)n * D + k], W[(size_t)n * D + k], ss);
            nrm = fmaxf(nrm, sqrtf(wave_sum(ss)));
        }
        if (b)
            for (int n = tid; n < N; n += 1024) bm = fmaxf(bm, fabsf(b[n]));
    }
    g = wave_max(g);
    bm = wave_max(bm);
    if (lane == 0) {
        red[0][wave] = fmaxf(g, 0.0f);
        red[1][wave] = bm;
    }
    __shared__ float red_n[16];
    if (lane == 0) red_n[wave] = nrm;
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 16; w++) {
            red[0][0] = fmaxf(red[0][0], red[0][w]);
            red[1][0] = fmaxf(red[1][0], red[1][w]);
            red_n[0] = fmaxf(red_n[0], red_n[w]);
        }
        // 1 + 2^-10 covers the rounding of the sums above
        const float in = sqrtf((float)D) * red[0][0] * (1.0f + 0x1p-10f);
        out[0] = in;
        float t = W ? (in * red_n[0] + red[1][0]) * (1.0f + 0x1p-10f) : 0.0f;
        out[1] = square ? t * t : t;
    }
}

}  // namespace vh

// Fused axial attention on bf16 matrix cores: the bf16 variant of
// attention_kernel (attention.hpp), same task decomposition, layout and
// online softmax, with q, k, v and the probabilities as bf16 MFMA operands
// and fp32 accumulation, statistics and normalisation.
//
// q/k/v/gates come from the bf16 fused projection (rows as in attention.hpp).
// q and k are rotated in fp32 (host-built cos/sin table) and rounded to bf16;
// q is also scaled by scale*log2(e) before rounding.
//
// Per wavefront: 32 queries.  Per block of 32 keys:
//   S^T = K * Q^T: 4 x v_mfma_f32_32x32x16_bf16 over the 64 head dims (A = K
//     rows from LDS, B = the wave's Q held in registers).  Lane (li, lh)
//     receives the scores of query li for keys 8*(r/4) + 4*lh + r%4.
//   O^T += V^T * P^T: per 16-key step st the lane's own registers
//     8st .. 8st+7 are the probabilities of keys {16st + 4lh + 0..3,
//     16st + 8 + 4lh + 0..3}: converted to bf16 they are the B operand as
//     they stand, and the A operand (V^T rows from LDS) is read in the same
//     key order (two 8-byte reads).
#pragma once

#include "attention.hpp"
#include "gemm_bf16.hpp"
#include "common.hpp"

namespace vh {

constexpr int ATB_KPITCH = ATT_DH + 8;  // K tile row pitch (bf16): 144 B, conflict-free 16-byte reads
constexpr int ATB_VPITCH = ATT_KB + 8;  // V^T tile row pitch (bf16)

template <int WAVES, typename TO>
__global__ __launch_bounds__(64 * WAVES, 4) void attention_bf16_kernel(AttnArgs a) {
    constexpr int NT = 64 * WAVES;
    constexpr int CHUNKS = ATT_KB * ATT_DH / 8;  // 16-byte chunks per K (or V) tile: 256
    constexpr int PER_T = CHUNKS / NT;
    static_assert(CHUNKS % NT == 0, "tile must divide evenly");
    __shared__ __attribute__((aligned(16))) bf16 Ks[2][ATT_KB][ATB_KPITCH];
    __shared__ __attribute__((aligned(16))) bf16 Vt[2][ATT_DH][ATB_VPITCH];

    const bf16 *qkv = static_cast<const bf16 *>(a.qkv);
    const int qgroups = (a.L + 32 * WAVES - 1) / (32 * WAVES);
    const int task = xcd_swizzle((int)blockIdx.x, (int)gridDim.x);  // neighbouring tasks share K/V rows: same XCD
    const int qg = task % qgroups;
    const int sh = task / qgroups;
    const int h = sh % a.H;
    const int s = sh / a.H;

    const int tid = (int)threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int li = lane & 31, lh = lane >> 5;
    const int q0 = (qg * WAVES + wave) * 32;
    const bool wave_active = q0 < a.L;

    const int kcol = a.inner + h * ATT_DH;
    const int vcol = 2 * a.inner + h * ATT_DH;

    // Q of query q0+li, dims 16g + 8lh .. +7, rotated and scaled (log2 domain).
    bf16x8 qb[4];
    float gate_logit = 0.0f;  // loaded with Q so the store does not wait on it
    {
        const int q = min(q0 + li, a.L - 1);
        const bf16 *qp = qkv + (size_t)attn_row(a, s, q) * a.ld + h * ATT_DH;
        if (a.gate_col >= 0) gate_logit = (float)qkv[(size_t)attn_row(a, s, q) * a.ld + a.gate_col + h];
        const float qs = a.scale * 1.4426950408889634f;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int d0 = 16 * g + 8 * lh;
            qb[g] = rope8_bf16(*reinterpret_cast<const bf16x8 *>(qp + d0), a.rope, q, d0, qs);
        }
    }

    // Staging: chunk c of the K tile is key c/8, dims 8*(c%8) (8 threads read
    // one key's 128 contiguous bytes); chunk c of the V tile is key c%32, dims
    // 8*(c/32), so a wave's V^T column writes spread over the banks.
    bf16x8 kreg[PER_T], vreg[PER_T];
    auto load = [&](int kb) {
#pragma unroll
        for (int i = 0; i < PER_T; i++) {
            const int c = tid + NT * i;
            const int kk = c >> 3, kd = 8 * (c & 7);
            const int vk = c & 31, vd = 8 * (c >> 5);
            const int pk = kb * ATT_KB + kk, pv = kb * ATT_KB + vk;
            if (pk < a.L) {
                const bf16 *kp = qkv + (size_t)attn_row(a, s, pk) * a.ld + kcol + kd;
                kreg[i] = rope8_bf16(*reinterpret_cast<const bf16x8 *>(kp), a.rope, pk, kd, 1.0f);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) kreg[i][e] = (bf16)0.0f;
            }
            if (pv < a.L) {
                vreg[i] = *reinterpret_cast<const bf16x8 *>(qkv + (size_t)attn_row(a, s, pv) * a.ld + vcol + vd);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) vreg[i][e] = (bf16)0.0f;
            }
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PER_T; i++) {
            const int c = tid + NT * i;
            *reinterpret_cast<bf16x8 *>(&Ks[buf][c >> 3][8 * (c & 7)]) = kreg[i];
            const int vk = c & 31, vd = 8 * (c >> 5);
#pragma unroll
            for (int e = 0; e < 8; e++) Vt[buf][vd + e][vk] = vreg[i][e];
        }
    };

    floatx16 o[2];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[t][r] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;

    const int nkb = (a.L + ATT_KB - 1) / ATT_KB;
    load(0);
    store(0);
    __syncthreads();
    for (int kb = 0; kb < nkb; kb++) {
        const int buf = kb & 1;
        if (kb + 1 < nkb) load(kb + 1);
        if (wave_active) {
            floatx16 sc;
#pragma unroll
            for (int r = 0; r < 16; r++) sc[r] = 0.0f;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const bf16x8 kf = *reinterpret_cast<const bf16x8 *>(&Ks[buf][li][16 * g + 8 * lh]);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qb[g], sc, 0, 0, 0);
            }
            const int valid = a.L - kb * ATT_KB;
            if (valid < ATT_KB) {
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (8 * (r >> 2) + 4 * lh + (r & 3) >= valid) sc[r] = -INFINITY;
            }
            online_softmax_block(sc, m_run, l_run, o);
#pragma unroll
            for (int st = 0; st < 2; st++) {
                bf16x8 pb;
#pragma unroll
                for (int e = 0; e < 8; e++) pb[e] = (bf16)sc[8 * st + e];
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const bf16 *vr = &Vt[buf][32 * t + li][16 * st + 4 * lh];
                    const bf16x4 v0 = *reinterpret_cast<const bf16x4 *>(vr);
                    const bf16x4 v1 = *reinterpret_cast<const bf16x4 *>(vr + 8);
                    const bf16x8 va = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                    o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, pb, o[t], 0, 0, 0);
                }
            }
        }
        if (kb + 1 < nkb) store(buf ^ 1);
        __syncthreads();
    }

    if (!wave_active) return;
    const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
    const int q = q0 + li;
    if (q >= a.L) return;
    const float inv = 1.0f / l_tot;
    const int row = attn_row(a, s, q);
    const float gate = a.gate_col >= 0 ? sigmoid_dev(gate_logit) : 1.0f;
    TO *op = static_cast<TO *>(a.out) + (size_t)row * a.ld_out + h * ATT_DH;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int rq = 0; rq < 4; rq++) {
            floatx4 v;
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = (o[t][4 * rq + r] * inv) * gate;
            st4(op + 32 * t + 8 * rq + 4 * lh, v);
        }
}

// The same on k that the fused projection has already rotated
// (GemmDescBF16::rope): nothing is computed while staging.  A 32-key block of K
// or V is 4 KB, copied global -> LDS by one 1 KB global_load_lds_dwordx4 per
// wave; V stays key-major and its transposed operand comes from
// ds_read_b64_tr_b16, swizzles and read orders as attention_h2_kvp_kernel's, the
// key blocks' pipeline too.  The register-staged kernel rotates every key once
// per 128 queries and transposes V by 2-byte LDS writes: 62 x 801 x 8 heads
// 220 us, this kernel 158.  Bound by the softmax's VALU work (some 110
// instructions beside 8 MFMAs per wave and block).  Same bits as
// attention_bf16_kernel.
constexpr int KVB_ROW = 128;                 // bytes of a key's 64 dims
constexpr int KVB_TILE = ATT_KB * KVB_ROW;   // 4 KB
template <typename TO>
__global__ __launch_bounds__(256, 4) void attention_bf16_kvp_kernel(AttnArgs a) {
    constexpr int WAVES = 4;
    __shared__ __attribute__((aligned(1024))) unsigned char Ks[2][KVB_TILE];
    __shared__ __attribute__((aligned(1024))) unsigned char Vs[2][KVB_TILE];
    auto swz_k = [](int r) { return (r >> 1) & 7; };
    auto swz_v = [](int r) { return 4 * ((r >> 1) & 1); };

    const bf16 *qkv = static_cast<const bf16 *>(a.qkv);
    const int qgroups = (a.L + 32 * WAVES - 1) / (32 * WAVES);
    const int task = xcd_swizzle((int)blockIdx.x, (int)gridDim.x);  // neighbouring tasks share K/V rows: same XCD
    const int qg = task % qgroups;
    const int sh = task / qgroups;
    const int h = sh % a.H;
    const int s = sh / a.H;
    const int tid = (int)threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const int q0 = (qg * WAVES + wave) * 32;

    bf16x8 qb[4];
    float gate_logit = 0.0f;
    {
        const int q = min(q0 + li, a.L - 1);
        const bf16 *qp = qkv + (size_t)attn_row(a, s, q) * a.ld + h * ATT_DH;
        if (a.gate_col >= 0) gate_logit = (float)qkv[(size_t)attn_row(a, s, q) * a.ld + a.gate_col + h];
        const float qs = a.scale * 1.4426950408889634f;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int d0 = 16 * g + 8 * lh;
            qb[g] = rope8_bf16(*reinterpret_cast<const bf16x8 *>(qp + d0), a.rope, q, d0, qs);
        }
    }

    // wave w copies keys 8 w .. +7 of a block: lane l key 8 w + l / 8, slot
    // l % 8, from that key's chunk (l % 8) ^ swz.  Keys past L load the row of
    // key L - 1 (masked scores: their probabilities are exactly 0).  32-bit
    // offsets from the sequence's first row (the launcher checks they fit).
    const char *seq_base = reinterpret_cast<const char *>(qkv) + (size_t)attn_row(a, s, 0) * a.ld * 2u;
    const uint32_t pos_bytes = (uint32_t)a.pos_stride * (uint32_t)a.ld * 2u;
    const int kr = 8 * wave + (lane >> 3);
    const uint32_t k_off = 2u * (uint32_t)a.inner + 128u * (uint32_t)h + 16u * (uint32_t)((lane & 7) ^ swz_k(kr));
    const uint32_t v_off = 4u * (uint32_t)a.inner + 128u * (uint32_t)h + 16u * (uint32_t)((lane & 7) ^ swz_v(kr));
    const uint32_t ks_base = (uint32_t)(uintptr_t)&Ks[0][0], vs_base = (uint32_t)(uintptr_t)&Vs[0][0];
    auto issue_k = [&](int kb) {
        lds_dma16s((uint32_t)min(kb * ATT_KB + kr, a.L - 1) * pos_bytes + k_off, seq_base,
                   ks_base + (uint32_t)((kb & 1) * KVB_TILE + 1024 * wave));
    };
    auto issue_v = [&](int kb) {
        lds_dma16s((uint32_t)min(kb * ATT_KB + kr, a.L - 1) * pos_bytes + v_off, seq_base,
                   vs_base + (uint32_t)((kb & 1) * KVB_TILE + 1024 * wave));
    };
    auto qk = [&](int buf) {
        floatx16 sc;
#pragma unroll
        for (int r = 0; r < 16; r++) sc[r] = 0.0f;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const bf16x8 kf =
                *reinterpret_cast<const bf16x8 *>(&Ks[buf][0] + li * KVB_ROW + 16 * ((2 * g + lh) ^ swz_k(li)));
            sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qb[g], sc, 0, 0, 0);
        }
        return sc;
    };
    floatx16 o[2];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[t][r] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;
    typedef __fp16 fp16x4 __attribute__((ext_vector_type(4)));
    const int tr_j = lane & 15, tr_dhalf = (lane >> 4) & 1;
    auto soft_pv = [&](floatx16 &sc, int kb) {
        const int valid = a.L - kb * ATT_KB;
        if (valid < ATT_KB) {
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (8 * (r >> 2) + 4 * lh + (r & 3) >= valid) sc[r] = -INFINITY;
        }
        online_softmax_block(sc, m_run, l_run, o);
#pragma unroll
        for (int st = 0; st < 2; st++) {
            bf16x8 pb;
#pragma unroll
            for (int e = 0; e < 8; e++) pb[e] = (bf16)sc[8 * st + e];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int key = 16 * st + 4 * lh + (tr_j >> 2);
                const int chunk = 4 * t + 2 * tr_dhalf + ((tr_j & 3) >> 1);
                const unsigned char *base = &Vs[kb & 1][0] + 8 * (tr_j & 1);
                const unsigned char *a0 = base + key * KVB_ROW + 16 * (chunk ^ swz_v(key));
                const unsigned char *a1 = base + (key + 8) * KVB_ROW + 16 * (chunk ^ swz_v(key + 8));
                // 16-bit elements moved as they are (the type only names their size)
                const fp16x4 r0 = __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) fp16x4 *)(a0));
                const fp16x4 r1 = __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) fp16x4 *)(a1));
                typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
                const u32x2 w0 = __builtin_bit_cast(u32x2, r0), w1 = __builtin_bit_cast(u32x2, r1);
                const bf16x8 va = __builtin_bit_cast(bf16x8, u32x4{w0[0], w0[1], w1[0], w1[1]});
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, pb, o[t], 0, 0, 0);
            }
        }
    };

    // entering iteration kb, Ks[(kb + 1) % 2] holds K(kb + 1) and Vs[kb % 2]
    // V(kb); it issues K(kb + 2) into Ks[kb % 2] (last read for block kb's
    // scores, before the barrier that ended the previous iteration) and V(kb + 1)
    // into Vs[(kb + 1) % 2] (last read before that barrier too)
    const int nkb = (a.L + ATT_KB - 1) / ATT_KB;
    issue_k(0);
    issue_v(0);
    issue_k(1);
    wait_vmcnt<0>();
    __syncthreads();
    const bool active = q0 < a.L;
    floatx16 sc;
    if (active) sc = qk(0);
    __syncthreads();  // every wave has read K(0): iteration 0 copies K(2) there
    for (int kb = 0; kb < nkb; kb++) {
        issue_k(kb + 2);
        issue_v(kb + 1);
        if (active) {
            const floatx16 next = qk((kb + 1) & 1);
            soft_pv(sc, kb);
            sc = next;
        }
        wait_vmcnt<0>();
        __syncthreads();
    }

    if (!active) return;
    const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
    const int q = q0 + li;
    if (q >= a.L) return;
    const float inv = 1.0f / l_tot;
    const int row = attn_row(a, s, q);
    const float gate = a.gate_col >= 0 ? sigmoid_dev(gate_logit) : 1.0f;
    TO *op = static_cast<TO *>(a.out) + (size_t)row * a.ld_out + h * ATT_DH;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int rq = 0; rq < 4; rq++) {
            floatx4 v;
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = (o[t][4 * rq + r] * inv) * gate;
            st4(op + 32 * t + 8 * rq + 4 * lh, v);
        }
}

}  // namespace vh

// q8_0_t.hip — Q8_0 x Q8_0 for several activation rows in the AVX1 tile order T
// (bench/bpd_gemm_q8_0_cpu.c:32-86), on f16 MFMA.
#include <algorithm>

#include "bpdq_device.h"
#include "bpdq_launch.h"
#include "bpdq_q8_0.h"

namespace bpdq {

// ----------------------------------------------------------------------------
// k_q8_0_gemm_TM.  Per cell and lane L = 0..7 of the reference's vector, over the
// blocks b in order:  acc_L = RN(RN(RN(Ad*Bd) * p_L) + acc_L), p_L the exact dot of
// elements 4L..4L+3 of the two blocks; the cell is
// ((a0+a4)+(a2+a6))+((a1+a5)+(a3+a7)).  The 16 fp32 operations per cell and block
// cannot be merged (each result is rounded), so the VALU bounds this product; the
// kernel gives it nothing else to do:
//  - v_mfma_f32_16x16x4_4b_f16 computes four independent 16x16 products of inner
//    length 4: with the quants as f16 (exact) its "block" k gives p_L of 16 rows x
//    16 tokens as the exact fp32 value (|p_L| <= 65,536), so there is no
//    int-to-float conversion.  Two of them (L = 2k, L = 2k+1) cover a Q8_0 block.
//  - the same instruction with the two f16 scales at inner index 0 and zeros
//    elsewhere gives RN(Ad*Bd) (exact: 11 x 11 bits) of both blocks of a stage at once.
// A workgroup owns R = 16 WRN weight rows x C = 16 WCN tokens; each of its WRN x
// WCN waves 16 rows x 16 tokens: 32 accumulators per lane.  A stage is 2 blocks
// (68 bytes of a row), staged by 4 threads per row: a thread loads half a block,
// turns its 16 quants to f16 (0x6400 | (q ^ 0x80) is 1152 + q) and writes 32 bytes.
// PF stages are in flight in registers, two LDS slots alternate, one barrier per
// stage (LDS only, so the loads stay in flight across it).
// LDS: [block][row][64 bytes]; the 16-byte chunk k of a row (quants 8k..8k+7) sits
// at k ^ ((row >> 2) & 3) and a block's plane is padded by 16 bytes, so that 16
// consecutive lanes reading (16 rows, one chunk) or writing (4 rows, two blocks, two
// chunks) touch 16 different 16-byte groups modulo 256.
// Blocks past the end of a row have zero scales: acc + 0 is acc (a chain that
// starts at +0.0 never is -0.0).  Rows and tokens past the end repeat the last one.
// ----------------------------------------------------------------------------
typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));
typedef float tf32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t tu32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t tu32x4_a1 __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t tu32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

template <int WRN, int WCN>
struct TmGeo {
    static constexpr int R = 16 * WRN, C = 16 * WCN, ROWS = R + C;
    static constexpr int NT = 64 * WRN * WCN, UNITS = 4 * ROWS;  // staging threads (UNITS % 64 == 0)
    static constexpr int PASSES = (UNITS + NT - 1) / NT;
    static constexpr int PLANE = ROWS * 64 + 16;                 // bytes of one block's quants
    static constexpr int SLOT = 2 * PLANE + 2 * ROWS * 4;        // quants, then the scales [block][row]
};

struct TmRaw {
    tu32x4 q;    // AL: the dwords at the half block's (aligned) start; else its 16 quants
    uint32_t e;  // AL: the dword after them; else the block's scale
};

// 4 int8 quants -> 4 f16.
__device__ __forceinline__ uint2 tm_f16(uint32_t q) {
    const uint32_t u = q ^ 0x80808080u;  // q + 128 per byte
    const h16x2 bias = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    const h16x2 lo = __builtin_bit_cast(h16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + bias;
    const h16x2 hi = __builtin_bit_cast(h16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + bias;
    return make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
}

// AL: W, X 4-byte aligned and nb even: part p of a stage's 68 bytes is loaded from
// dword offset {0, 16, 36, 52} (block 0's quants start 2 bytes into a dword).
template <bool AL>
__device__ __forceinline__ void tm_load(TmRaw& t, const uint8_t* __restrict__ src, int p, int st, int nst, int nb) {
    if constexpr (AL) {
        const uint8_t* s = src + (int64_t)min(st, nst - 1) * (2 * kQ80Bytes) + 16 * p + (p >= 2 ? 4 : 0);
        t.q = *reinterpret_cast<const tu32x4_a4*>(s);
        t.e = *reinterpret_cast<const uint32_t*>(s + (p >= 2 ? 12 : 16));
    } else {
        const uint8_t* s = src + (int64_t)min(2 * st + (p >> 1), nb - 1) * kQ80Bytes;
        t.q = *reinterpret_cast<const tu32x4_a1*>(s + 2 + 16 * (p & 1));
        t.e = ld_u16(s);
    }
}

// Stage st of one staging thread into a slot; returns the OR of has_m128 of its quants.
template <bool AL, int ROWS, int PLANE>
__device__ __forceinline__ uint32_t tm_store(uint8_t* slot, const TmRaw& t, int row, int p, int st, int nb, bool want) {
    uint32_t q[4], d;
    if constexpr (AL) {
        const uint32_t sh = p >= 2 ? 0u : 16u;
        q[0] = __builtin_amdgcn_alignbit(t.q[1], t.q[0], sh);
        q[1] = __builtin_amdgcn_alignbit(t.q[2], t.q[1], sh);
        q[2] = __builtin_amdgcn_alignbit(t.q[3], t.q[2], sh);
        q[3] = __builtin_amdgcn_alignbit(t.e, t.q[3], sh);
        d = p == 0 ? (t.q[0] & 0xFFFFu) : (t.e >> 16);  // block 1's scale: high half of part 1's last dword
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = t.q[i];
        d = t.e;
    }
    const int u = p >> 1, h = p & 1, swz = (row >> 2) & 3;
    uint8_t* base = slot + u * PLANE + row * 64;
    const uint2 a = tm_f16(q[0]), b = tm_f16(q[1]), c = tm_f16(q[2]), e = tm_f16(q[3]);
    *reinterpret_cast<uint4*>(base + 16 * ((2 * h) ^ swz)) = make_uint4(a.x, a.y, b.x, b.y);
    *reinterpret_cast<uint4*>(base + 16 * ((2 * h + 1) ^ swz)) = make_uint4(c.x, c.y, e.x, e.y);
    uint32_t* sc = reinterpret_cast<uint32_t*>(slot + 2 * PLANE);
    if constexpr (AL) {
        if (p < 2) sc[p * ROWS + row] = d;
    } else {
        if (h == 0) sc[u * ROWS + row] = 2 * st + u < nb ? d : 0u;
    }
    if (!want) return 0u;
    return has_m128(q[0]) | has_m128(q[1]) | has_m128(q[2]) | has_m128(q[3]);
}

template <int WRN, int WCN, int PF, bool AL>
__global__ __launch_bounds__(64 * WRN * WCN) void k_q8_0_gemm_TM(GemmW gw, const uint8_t* __restrict__ X, int m_tokens,
                                                                 int nb) {
    using G = TmGeo<WRN, WCN>;
    static_assert(PF % 2 == 0, "slot parity");
    __shared__ __align__(16) uint8_t lds[2 * G::SLOT];
    __shared__ uint32_t m128[G::C];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / WCN, wc = wave % WCN;
    int bx, by;
    sh_tile(blockIdx.x, gw.first[kGemmMulti], (m_tokens + G::C - 1) / G::C, bx, by);
    const int mi = (bx >= gw.first[1]) + (bx >= gw.first[2]);
    const uint8_t* __restrict__ W = gw.w[mi];
    float* __restrict__ out = gw.out[mi];
    const int m_weight = gw.m[mi];
    const int m0 = (bx - gw.first[mi]) * G::R, n0 = by * G::C;
    const int64_t bpr = (int64_t)nb * kQ80Bytes;
    const int nst = (nb + 1) / 2;

    // staging: unit tid + ps * NT is part p of staged row (the R weight rows, then the C tokens)
    const uint8_t* src[G::PASSES];
    int srow[G::PASSES];
    const int p = tid & 3;
#pragma unroll
    for (int ps = 0; ps < G::PASSES; ps++) {
        const int row = min((tid + ps * G::NT) >> 2, G::ROWS - 1);
        srow[ps] = row;
        src[ps] = row < G::R ? W + (int64_t)min(m0 + row, m_weight - 1) * bpr
                             : X + (int64_t)min(n0 + row - G::R, m_tokens - 1) * bpr;
    }
    for (int i = tid; i < G::C; i += G::NT) m128[i] = 0u;

    TmRaw raw[PF][G::PASSES];
    uint32_t bad[G::PASSES] = {};
    const auto load = [&](TmRaw (&r)[G::PASSES], int st) {
#pragma unroll
        for (int ps = 0; ps < G::PASSES; ps++)
            if ((ps + 1) * G::NT <= G::UNITS || tid + ps * G::NT < G::UNITS) tm_load<AL>(r[ps], src[ps], p, st, nst, nb);
    };
    const auto store = [&](const TmRaw (&r)[G::PASSES], int slot, int st) {
#pragma unroll
        for (int ps = 0; ps < G::PASSES; ps++)
            if ((ps + 1) * G::NT <= G::UNITS || tid + ps * G::NT < G::UNITS)
                bad[ps] |= tm_store<AL, G::ROWS, G::PLANE>(lds + slot * G::SLOT, r[ps], srow[ps], p, st, nb,
                                                           srow[ps] >= G::R);
    };
#pragma unroll
    for (int i = 0; i < PF; i++) load(raw[i], i);
    store(raw[0], 0, 0);
    load(raw[0], PF);
    lds_barrier();

    float acc[8][4];
#pragma unroll
    for (int L = 0; L < 8; L++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[L][r] = 0.0f;

    const int j = lane & 15, k = lane >> 4;
    const int frag = j * 64 + 16 * (k ^ (j >> 2));  // this lane's chunk in a 16-row tile
    const int arow = wr * 16, brow = G::R + wc * 16;
    // scale operands: lane group k gives block k & 1
    const int asc = (k & 1) * G::ROWS + arow + j, bsc = (k & 1) * G::ROWS + brow + j;
    const tf32x16 zero = {0.0f};

    for (int s0 = 0; s0 < nst; s0 += PF) {
#pragma unroll
        for (int i = 0; i < PF; i++) {
            const int st = s0 + i;
            if (st >= nst) break;
            if (st + 1 < nst) {  // the other slot was last read before the previous barrier
                store(raw[(i + 1) % PF], (i + 1) & 1, st + 1);
                load(raw[(i + 1) % PF], st + 1 + PF);
            }
            const uint8_t* slot = lds + (i & 1) * G::SLOT;
            const uint32_t* sc = reinterpret_cast<const uint32_t*>(slot + 2 * G::PLANE);
            const h16x4 sa = __builtin_bit_cast(h16x4, make_uint2(sc[asc], 0u));
            const h16x4 sb = __builtin_bit_cast(h16x4, make_uint2(sc[bsc], 0u));
            const tf32x16 delta = __builtin_amdgcn_mfma_f32_16x16x4f16(sa, sb, zero, 0, 0, 0);
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const uint4 fa = *reinterpret_cast<const uint4*>(slot + u * G::PLANE + arow * 64 + frag);
                const h16x4 a0 = __builtin_bit_cast(h16x4, make_uint2(fa.x, fa.y));
                const h16x4 a1 = __builtin_bit_cast(h16x4, make_uint2(fa.z, fa.w));
                const uint4 fb = *reinterpret_cast<const uint4*>(slot + u * G::PLANE + brow * 64 + frag);
                const h16x4 b0 = __builtin_bit_cast(h16x4, make_uint2(fb.x, fb.y));
                const h16x4 b1 = __builtin_bit_cast(h16x4, make_uint2(fb.z, fb.w));
                const tf32x16 p0 = __builtin_amdgcn_mfma_f32_16x16x4f16(a0, b0, zero, 0, 0, 0);
                const tf32x16 p1 = __builtin_amdgcn_mfma_f32_16x16x4f16(a1, b1, zero, 0, 0, 0);
#pragma unroll
                for (int g = 0; g < 4; g++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float d = delta[4 * u + r];
                        acc[2 * g][r] = d * p0[4 * g + r] + acc[2 * g][r];
                        acc[2 * g + 1][r] = d * p1[4 * g + r] + acc[2 * g + 1][r];
                    }
            }
            lds_barrier();
        }
    }

#pragma unroll
    for (int ps = 0; ps < G::PASSES; ps++)
        if (bad[ps] != 0) m128[srow[ps] - G::R] = 1u;
    __syncthreads();
    // register r of lane l: row 4 (l / 16) + r of the wave's 16, token l % 16
    const int tl = wc * 16 + j, tok = n0 + tl, r0 = m0 + arow + 4 * k;
    if (tok >= m_tokens) return;
    float y[4];
    bool odd = m128[tl] != 0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        y[r] = ((acc[0][r] + acc[4][r]) + (acc[2][r] + acc[6][r])) + ((acc[1][r] + acc[5][r]) + (acc[3][r] + acc[7][r]));
        odd |= __builtin_isnan(y[r]);
    }
    if (odd) {  // the reference's own arithmetic: NaN bits, -128 activation quants
        for (int r = 0; r < 4; r++)
            if (r0 + r < m_weight && (m128[tl] != 0 || __builtin_isnan(y[r])))
                y[r] = t_order_cell(W + (r0 + r) * bpr, kQ80Bytes, 2, X + tok * bpr, nb, r0 + r, tok, m_weight, m_tokens);
    }
    float* o = out + (int64_t)tok * m_weight + r0;
    if ((reinterpret_cast<uintptr_t>(o) & 15) == 0 && r0 + 4 <= m_weight) {
        *reinterpret_cast<float4*>(o) = make_float4(y[0], y[1], y[2], y[3]);
    } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (r0 + r < m_weight) o[r] = y[r];
    }
}

// ----------------------------------------------------------------------------
// k_q8_0_gemm_TQ: the same cells on v_mfma_f32_4x4x4_16b_f16, 16 independent 4x4
// products of inner length 4, for few tokens.  A wave owns 8 rows; "block" L + 8 rg
// of the instruction gives p_L of rows 4 rg .. 4 rg + 3 x 4 tokens, so a lane holds
// the chains of 4 rows for one (L, token), and the accumulators of 4 NQ tokens are
// 4 NQ registers.  Each wave streams its own rows in chunks of CB blocks through
// registers (two chunks in flight) and its own LDS slot as 16-byte pieces; the
// workgroup shares only the activation chunk (f16, two slots), so there is one
// barrier per CB blocks.  Any K and alignment: the pieces are 16-byte loads at any address,
// and zero blocks fill the last chunk.  (4096x8 at K = 4128: 34.5 us in per-token GEMVs,
// 15.8 here; at K = 4096 the alignment is worth less than the runs differ.)
// LDS: rows at an odd multiple of 8 dwords (8 rows x 8 quant dwords of a block touch
// 64 different banks); the quants of 4 tokens of a block are 256 contiguous bytes.
// ----------------------------------------------------------------------------
typedef float tf32x4 __attribute__((ext_vector_type(4)));

template <int NQ, int NW>
struct TqGeo {
    static constexpr int C = 4 * NQ, R = 8 * NW, NT = 64 * NW, CB = kChunkBlocks;
    static constexpr int PLANE = C * 64 + 32;             // one block's activation quants
    static constexpr int XSLOT = CB * PLANE + CB * C * 4;  // quants, then the scales [block pair][token][2]
    static constexpr int UX = C * CB * 2, XP = (UX + NT - 1) / NT;
    static constexpr int LDS = 2 * XSLOT + NW * 8 * kChunkPitch;
    static_assert((kChunkPitch / 32) % 2 == 1 && kChunkPitch % 32 == 0 && XSLOT % 16 == 0, "LDS geometry");
};

struct TqX {
    tu32x4 q;
    uint32_t d;
};

// The operands of blocks 2t and 2t + 1 of a chunk: this lane's weight dwords, the
// scales of its row, and per 4 tokens the quants and both scales.
template <int NQ>
struct TqOps {
    uint32_t lo, hi, q1, d0, d1;
    uint2 b0[NQ], b1[NQ];
    float2 s[NQ];
};

template <int NQ, int C, int PLANE>
__device__ __forceinline__ void tq_read(TqOps<NQ>& o, const uint8_t* wq, const uint8_t* wd, const uint8_t* xq,
                                        const float2* xd, int t) {
    o.lo = *reinterpret_cast<const uint32_t*>(wq + 68 * t);  // block 2t: quants 2 bytes into a dword
    o.hi = *reinterpret_cast<const uint32_t*>(wq + 68 * t + 4);
    o.q1 = *reinterpret_cast<const uint32_t*>(wq + 68 * t + 36);
    o.d0 = *reinterpret_cast<const uint16_t*>(wd + 68 * t);
    o.d1 = *reinterpret_cast<const uint16_t*>(wd + 68 * t + 34);
#pragma unroll
    for (int n = 0; n < NQ; n++) {
        o.b0[n] = *reinterpret_cast<const uint2*>(xq + 2 * t * PLANE + 256 * n);
        o.b1[n] = *reinterpret_cast<const uint2*>(xq + (2 * t + 1) * PLANE + 256 * n);
        o.s[n] = xd[t * C + 4 * n];
    }
}

template <int NQ>
__device__ __forceinline__ void tq_pair(const TqOps<NQ>& o, float (&acc)[NQ][4]) {
    const tf32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const h16x4 a0 = __builtin_bit_cast(h16x4, tm_f16(__builtin_amdgcn_alignbit(o.hi, o.lo, 16)));
    const h16x4 a1 = __builtin_bit_cast(h16x4, tm_f16(o.q1));
    const float d0 = f16_ieee(o.d0), d1 = f16_ieee(o.d1);
    tf32x4 p0[NQ], p1[NQ], e0[NQ], e1[NQ];
#pragma unroll
    for (int n = 0; n < NQ; n++) {
        e0[n] = __builtin_amdgcn_mfma_f32_4x4x1f32(d0, o.s[n].x, zero, 0, 0, 0);
        p0[n] = __builtin_amdgcn_mfma_f32_4x4x4f16(a0, __builtin_bit_cast(h16x4, o.b0[n]), zero, 0, 0, 0);
        e1[n] = __builtin_amdgcn_mfma_f32_4x4x1f32(d1, o.s[n].y, zero, 0, 0, 0);
        p1[n] = __builtin_amdgcn_mfma_f32_4x4x4f16(a1, __builtin_bit_cast(h16x4, o.b1[n]), zero, 0, 0, 0);
    }
#pragma unroll
    for (int n = 0; n < NQ; n++) {
#pragma unroll
        for (int r = 0; r < 4; r++) acc[n][r] = e0[n][r] * p0[n][r] + acc[n][r];
    }
#pragma unroll
    for (int n = 0; n < NQ; n++) {
#pragma unroll
        for (int r = 0; r < 4; r++) acc[n][r] = e1[n][r] * p1[n][r] + acc[n][r];
    }
}

template <int NQ, int NW>
__global__ __launch_bounds__(64 * NW) void k_q8_0_gemm_TQ(GemmW gw, const uint8_t* __restrict__ X, int m_tokens, int nb) {
    using G = TqGeo<NQ, NW>;
    constexpr int CB = G::CB;
    __shared__ __align__(16) uint8_t lds[G::LDS];
    __shared__ uint32_t m128[G::C];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int bx, by;
    sh_tile(blockIdx.x, gw.first[kGemmMulti], (m_tokens + G::C - 1) / G::C, bx, by);
    const int mi = (bx >= gw.first[1]) + (bx >= gw.first[2]);
    const uint8_t* __restrict__ W = gw.w[mi];
    float* __restrict__ out = gw.out[mi];
    const int m_weight = gw.m[mi];
    const int row0 = (bx - gw.first[mi]) * G::R + wave * 8, n0 = by * G::C;
    const int64_t bpr = (int64_t)nb * kQ80Bytes;
    const int nch = (nb + CB - 1) / CB;
    const RowChunks<8> rows(W, row0, m_weight, nb);
    uint8_t* slot = lds + 2 * G::XSLOT + wave * 8 * kChunkPitch;
    // activations: unit i is half i & 1 of block (i / 2) % CB of token i / (2 CB)
    TqX xr[G::XP];
    const auto xload = [&](int c) {
#pragma unroll
        for (int u = 0; u < G::XP; u++) {
            const int i = min(tid + u * G::NT, G::UX - 1), t = i / (2 * CB), b = (i >> 1) % CB;
            const uint8_t* s = X + (int64_t)min(n0 + t, m_tokens - 1) * bpr + (int64_t)min(c * CB + b, nb - 1) * kQ80Bytes;
            xr[u].q = *reinterpret_cast<const tu32x4_a1*>(s + 2 + 16 * (i & 1));
            xr[u].d = ld_u16(s);
        }
    };
    uint32_t bad[G::XP] = {};
    const auto xstore = [&](int xs, int c) {
        uint8_t* x = lds + xs * G::XSLOT;
#pragma unroll
        for (int u = 0; u < G::XP; u++) {
            const int i = tid + u * G::NT, t = i / (2 * CB), b = (i >> 1) % CB;
            if (G::UX % G::NT != 0 && i >= G::UX) continue;
            if (c * CB + b >= nb) xr[u] = TqX{{0, 0, 0, 0}, 0};  // a zero block adds +0
            const uint2 q0 = tm_f16(xr[u].q[0]), q1 = tm_f16(xr[u].q[1]), q2 = tm_f16(xr[u].q[2]), q3 = tm_f16(xr[u].q[3]);
            uint4* d = reinterpret_cast<uint4*>(x + b * G::PLANE + t * 64 + 32 * (i & 1));
            d[0] = make_uint4(q0.x, q0.y, q1.x, q1.y);
            d[1] = make_uint4(q2.x, q2.y, q3.x, q3.y);
            if ((i & 1) == 0)
                reinterpret_cast<float*>(x + CB * G::PLANE)[2 * ((b >> 1) * G::C + t) + (b & 1)] = f16_ieee(xr[u].d);
            bad[u] |= has_m128(xr[u].q[0]) | has_m128(xr[u].q[1]) | has_m128(xr[u].q[2]) | has_m128(xr[u].q[3]);
        }
    };

    RowChunks<8>::V wv[2];
    xload(0);
    rows.load(wv[0], 0);
    rows.load(wv[1], 1);
    for (int i = tid; i < G::C; i += G::NT) m128[i] = 0u;
    xstore(0, 0);
    lds_barrier();

    float acc[NQ][4];
#pragma unroll
    for (int q = 0; q < NQ; q++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[q][r] = 0.0f;
    const int j = lane & 3, L = (lane >> 2) & 7, rg = lane >> 5;
    const uint8_t* wq = slot + (4 * rg + j) * kChunkPitch + 4 * L;   // this lane's row, dword L
    const uint8_t* wd = slot + (4 * rg + j) * kChunkPitch;

    const auto step = [&](RowChunks<8>::V& v, int xs, int c) {
        if (c == nch - 1) rows.end(v);
        rows.store(slot, v);
        xload(min(c + 1, nch - 1));  // before the weights: loads return in order
        rows.load(v, c + 2);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        const uint8_t* x = lds + xs * G::XSLOT;
        const uint8_t* xq = x + j * 64 + 8 * L;
        const float2* xd = reinterpret_cast<const float2*>(x + CB * G::PLANE) + j;
        // pairs of blocks, the next pair's operands read before this one's arithmetic
        TqOps<NQ> o[2];
        tq_read<NQ, G::C, G::PLANE>(o[0], wq, wd, xq, xd, 0);
        if ((c + 1) * CB <= nb) {
#pragma unroll
            for (int t = 0; t < CB / 2; t++) {
                if (t + 1 < CB / 2) tq_read<NQ, G::C, G::PLANE>(o[(t + 1) & 1], wq, wd, xq, xd, t + 1);
                __builtin_amdgcn_sched_barrier(0);
                tq_pair<NQ>(o[t & 1], acc);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            const int npair = (nb - c * CB + 1) / 2;
#pragma unroll 1
            for (int t = 0; t < npair; t++) {
                tq_read<NQ, G::C, G::PLANE>(o[0], wq, wd, xq, xd, t);
                tq_pair<NQ>(o[0], acc);
            }
        }
        xstore(xs ^ 1, c + 1);  // last read before the previous barrier
        lds_barrier();
    };
    int c0 = 0;
    for (; c0 + 1 < nch; c0 += 2) {
        step(wv[0], 0, c0);
        step(wv[1], 1, c0 + 1);
    }
    if (c0 < nch) step(wv[0], 0, c0);

#pragma unroll
    for (int u = 0; u < G::XP; u++) {
        const int t = min(tid + u * G::NT, G::UX - 1) / (2 * CB);
        if (bad[u] != 0) m128[t] = 1u;
    }
    __syncthreads();
    // the 8 lanes L of a cell all hold its sum; lane L takes row L % 4 of its four and token
    // L / 4 of its NQ, so the cells that t_order_cell recomputes, one chain over the row each,
    // run side by side (14336x2 with a -128 in every block 420 us; 1,810 where the lanes L = 0 took
    // them four by four, 1,520 in the GEMVs)
    const int n = L >> 2, r = L & 3, tl = 4 * n + j, tok = n0 + tl, row = row0 + 4 * rg + r;
    float y = 0.0f;
#pragma unroll
    for (int i = 0; i < 4 * NQ; i++) {
        float a = acc[i >> 2][i & 3];
        a = a + xor_f(a, 16);
        a = a + xor_f(a, 8);
        a = a + xor_f(a, 4);
        y = L == i ? a : y;
    }
    if (n >= NQ || tok >= m_tokens || row >= m_weight) return;
    if (m128[tl] != 0 || __builtin_isnan(y))
        y = t_order_cell(W + row * bpr, kQ80Bytes, 2, X + tok * bpr, nb, row, tok, m_weight, m_tokens);
    out[(int64_t)tok * m_weight + row] = y;
}

template <int WRN, int WCN, int PF, bool AL>
static void launch_tm(const uint8_t* const* W, float* const* out, const int* M, int n, const uint8_t* Xq, int m_tokens,
                      int nb, hipStream_t s) {
    using G = TmGeo<WRN, WCN>;
    const GemmW g = gemm_args<G::R>(W, out, M, n);
    hipLaunchKernelGGL((k_q8_0_gemm_TM<WRN, WCN, PF, AL>), dim3(g.first[kGemmMulti] * ((m_tokens + G::C - 1) / G::C)),
                       dim3(G::NT), 0, s, g, Xq, m_tokens, nb);
}

template <int NQ, int NW>
static void launch_tq(const uint8_t* const* W, float* const* out, const int* M, int n, const uint8_t* Xq, int m_tokens,
                      int nb, hipStream_t s) {
    using G = TqGeo<NQ, NW>;
    const GemmW g = gemm_args<G::R>(W, out, M, n);
    hipLaunchKernelGGL((k_q8_0_gemm_TQ<NQ, NW>), dim3(g.first[kGemmMulti] * ((m_tokens + G::C - 1) / G::C)),
                       dim3(G::NT), 0, s, g, Xq, m_tokens, nb);
}

// Which kernel: the least of the estimated times (ns) of the per-token GEMVs and the four
// forms here.  A launch's workgroups run in n = ceil(workgroups / 256) per CU, whether their
// rows and tokens are real or padding, and its time is close to fixed + step * n + K * g(n),
// g the ns per element of K:
//   TQ<1> 32 rows x 4 tokens    g = max(1.22 + 1.38 n, 1.85 n)
//   TQ<2> 32 rows x 8 tokens    g = max(1.5 + 1.95 n, 3.3 n - 1.9)
//   TM    32 rows x 64 tokens   g = 2 + 9 n
//   TM    64 rows x 64 tokens   g = 16.6 n - 2; not without 4-byte alignment, where 23 n - 2 is
//                               more than twice the n of 32 rows cost
// (a first wave per SIMD waits for memory, so the small forms cost more at n = 1 than their
// share).  The GEMVs (launch_wide) take time by cells: rows * tokens * (0.04 + 1.6e-4 K), less
// where the rows stay in the L2s between tokens, more where launch_wide does not run.  Fitted
// to 1,200 shapes on MI355X, weights beyond the MALL (512 to 128256 rows, 2 to 256 tokens,
// K 1024 to 14336, 1440, 4128 and 8032): the choice is on the average 0.4 % and at most 16 %
// over the best form, and no shape is slower than the GEMVs.  us, K = 4096, the GEMVs / TQ<1>
// / TQ<2> / TM 32 / TM 64:
//   4096x2 8.7 / 14.3 / 17.8; 4096x4 14.1 / 14.5 / 17.9; 4096x8 22.4 / 14.6 / 18.0
//   8192x2 14.8 / 15.2 / 18.7; 11008x2 18.7 / 20.6 / 26.6; 14336x2 22.3 / 20.6 / 26.9
//   14336x8 74 / 34 / 30; 32000x2 44 / 37 / 55; 32000x9 184 / 85 / 97 / - / 157
//   128256x2 175 / 132 / 224 / - / 579; 4096x33 77 / - / 44 / 54 / 61; 14336x33 286 / - / 119 / 86 / 70
//   4096x512 1,360 / - / - / - / 125;  14336x512 4,890 / - / - / - / 434 (88 % of it the 382 us that 16
//   VALU operations per cell and block take)
// Below 16,384 cells the GEMVs stay: 1024x8 7.8 against 14.2.
// 4 waves of 16-block chunks per workgroup; with 2 waves, 8 waves, 8-block chunks (whole
// calls, us): 14336x8 30.5 against 32.5, 29.8, 32.5; 8192x8 20.6 against 26.1, 26.5, 22.9;
// 4096x16 19.7 against 25.5, 26.1, 22.6; 14336x16 53.3 against 55.5, 53.1, 53.0.
bool launch_q8_0_gemm_T_multi(const uint8_t* const* W, float* const* out, const int* M, int n, const uint8_t* Xq,
                              int m_tokens, int K, hipStream_t s) {
    const int nb = K / 32;
    bool al4 = nb % 2 == 0 && (reinterpret_cast<uintptr_t>(Xq) & 3) == 0;
    bool wide = nb % 32 == 0;  // launch_wide takes every matrix
    int64_t rows = 0;
    for (int i = 0; i < n; i++) {
        rows += M[i];
        al4 = al4 && (reinterpret_cast<uintptr_t>(W[i]) & 3) == 0;
        wide = wide && (reinterpret_cast<uintptr_t>(W[i]) & 15) == 0;
    }
    const int64_t cells = rows * m_tokens;
    if (nb == 0 || m_tokens < 2 || cells < 16384) return false;
    // workgroups of R rows x C tokens per CU
    const auto per_cu = [&](int R, int C) {
        int64_t b = 0;
        for (int i = 0; i < n; i++) b += (M[i] + R - 1) / R;
        return (double)((b * ((m_tokens + C - 1) / C) + 255) / 256);
    };
    const double k = K, n1 = per_cu(32, 4), n2 = per_cu(32, 8), n3 = per_cu(32, 64), n4 = per_cu(64, 64);
    const double gemv = 2600.0 * n + (double)cells * (!wide ? 0.08 + 2.5e-4 * k : rows <= 2048 ? 0.03 + 1.35e-4 * k : 0.04 + 1.6e-4 * k);
    const double tq1 = 3300 + 600 * n1 + k * std::max(1.22 + 1.38 * n1, 1.85 * n1);
    const double tq2 = 3500 + 600 * n2 + k * std::max(1.5 + 1.95 * n2, 3.3 * n2 - 1.9);
    const double tm32 = 3000 + 300 * n3 + k * (2 + 9 * n3);
    const double tm64 = 3000 + 300 * n4 + k * (16.6 * n4 - 2);
    double least = std::min(std::min(tq1, tq2), tm32);
    if (al4) least = std::min(least, tm64);
    if (gemv <= least) return false;
    if (least == tq1)
        launch_tq<1, 4>(W, out, M, n, Xq, m_tokens, nb, s);
    else if (least == tq2)
        launch_tq<2, 4>(W, out, M, n, Xq, m_tokens, nb, s);
    else if (least == tm32 && al4)
        launch_tm<2, 4, 4, true>(W, out, M, n, Xq, m_tokens, nb, s);
    else if (least == tm32)
        launch_tm<2, 4, 4, false>(W, out, M, n, Xq, m_tokens, nb, s);
    else
        launch_tm<4, 4, 4, true>(W, out, M, n, Xq, m_tokens, nb, s);
    return true;
}

}  // namespace bpdq

// bpdq_q8_0.h — device helpers shared by the Q8_0 product kernels (q8_0.hip, q8_0_t.hip, q8_0_s.hip).
#pragma once
#include "bpdq_device.h"

namespace bpdq {

__device__ __forceinline__ uint32_t ld_u16(const uint8_t* p) {
    uint16_t v;
    __builtin_memcpy(&v, p, 2);
    return v;
}

// ----------------------------------------------------------------------------
// Cells of the AVX1 tile order T (bench/bpd_gemm_q8_0_cpu.c:32-86) that the fast
// kernels below cannot give bit for bit are recomputed by one lane in the
// reference's own arithmetic (t_order_cell): NaN cells, and every cell of an
// activation row holding a -128 quant (where SSSE3's sign/maddubs wrap: -(-128)
// is -128 against a negative weight; the kernels use the exact dot, which the
// Q8_0 quantizers' [-127, 127] output always gives).  NaN bits: the reference build
// on x86 gives a NaN operand back
// quieted (the first operand's when both are NaN) and Inf*0, Inf-Inf give the
// default NaN.  Which operand is first differs between the build's nine tile
// kernels, so a cell's bits depend on the tile that computes it
// (bench/bpd_gemm_q8_0_cpu.c:159-207: tiles of 4, then 2, then 1 rows and
// tokens).  Measured on that build, one probe per operand pair with NaNs of both
// signs: Ad and Bd come from the ldexpf decode of :13-26 (an f16 NaN becomes
// +/-0x7FC00000, no payload); scale = Bd*Ad with Bd first in every tile; lane L's
// product scale*float(p_L); its chain acc_L = prod + acc_L with the accumulator
// first in the 1x1 tile and the product first in the others; the hsum
// ((a0+a4)+(a2+a6))+((a1+a5)+(a3+a7)) with a per-cell mask of swapped additions
// (t_tile_mask).  Weight block b of the row is at wrow + b * bstride, its quants
// at +qoff.
// ----------------------------------------------------------------------------
__device__ __forceinline__ float x86_mul(float first, float second) {
    const float r = first * second;
    return __builtin_isnan(r) ? x86_nan_of(first, second) : r;
}
__device__ __forceinline__ float x86_add(float first, float second) {
    const float r = first + second;
    return __builtin_isnan(r) ? x86_nan_of(first, second) : r;
}
__device__ __forceinline__ float x86_add_sw(float a, float b, uint32_t sw) { return sw ? x86_add(b, a) : x86_add(a, b); }
__device__ __forceinline__ float f16_tile(uint32_t h) {
    if (!f16_is_nan(h)) return f16_ieee(h);
    return __uint_as_float(((h & 0x8000u) << 16) | 0x7FC00000u);
}

// The tile of cell (row r, token t) and its hsum mask: bits 0-3 swap the pairs
// (a0,a4), (a2,a6), (a1,a5), (a3,a7) (the right one first), bit 4 the left
// second-level sum, bit 5 the right one, bit 6 the top addition.  *acc_first:
// the 1x1 tile.
__device__ __forceinline__ uint32_t t_tile_mask(int r, int t, int m_weight, int m_tokens, bool* acc_first) {
    const int full_r = m_weight / 4 * 4, full_t = m_tokens / 4 * 4;
    const int RM = r < full_r ? 4 : (m_weight - full_r >= 2 && r < full_r + 2) ? 2 : 1;
    const int RN = t < full_t ? 4 : (m_tokens - full_t >= 2 && t < full_t + 2) ? 2 : 1;
    const int i = RM == 4 ? r % 4 : RM == 2 ? r - full_r : 0;
    const int j = RN == 4 ? t % 4 : RN == 2 ? t - full_t : 0;
    *acc_first = RM == 1 && RN == 1;
    if (RM == 4) return 0x12u;
    if (RM == 2) return (RN == 1 || i == 0) ? 0u : 0x12u;
    return RN == 4 ? 0x10u : RN == 2 ? (j == 0 ? 0x01u : 0x10u) : 0u;
}

__device__ __forceinline__ float t_order_cell(const uint8_t* __restrict__ wrow, int64_t bstride, int qoff,
                                             const uint8_t* __restrict__ xrow, int nb, int r, int t, int m_weight,
                                             int m_tokens) {
    bool acc_first;
    const uint32_t m = t_tile_mask(r, t, m_weight, m_tokens, &acc_first);
    float C[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    for (int b = 0; b < nb; b++) {
        const uint8_t* wb = wrow + (int64_t)b * bstride;
        const uint8_t* xb = xrow + (int64_t)b * kQ80Bytes;
        const uint32_t hw = (uint32_t)wb[0] | ((uint32_t)wb[1] << 8);
        const uint32_t hx = (uint32_t)xb[0] | ((uint32_t)xb[1] << 8);
        const float scale = x86_mul(f16_tile(hx), f16_tile(hw));
#pragma unroll
        for (int L = 0; L < 8; L++) {
            const int p = ssse3_quad_inl(ld_u32(wb + qoff + 4 * L), ld_u32(xb + 2 + 4 * L));
            const float prod = x86_mul(scale, (float)p);
            C[L] = acc_first ? x86_add(C[L], prod) : x86_add(prod, C[L]);
        }
    }
    const float l0 = x86_add_sw(C[0], C[4], m & 1u), l1 = x86_add_sw(C[2], C[6], m & 2u);
    const float l2 = x86_add_sw(C[1], C[5], m & 4u), l3 = x86_add_sw(C[3], C[7], m & 8u);
    return x86_add_sw(x86_add_sw(l0, l1, m & 16u), x86_add_sw(l2, l3, m & 32u), m & 64u);
}

// ROWS consecutive 34-byte rows of a wave in chunks of 16 blocks, each row's chunk as 34
// 16-byte pieces at any address: loaded into registers (piece lane + 64 k of the chunk per lane)
// and stored to the wave's LDS slot at a pitch of 544 bytes (136 dwords, 8 mod 64: the rows of a
// column of quants fall in different banks).  Rows past the matrix repeat its last one.  A piece
// past a row's end is the row's last 16 bytes; end() moves the last chunk's into place, zeros
// behind.
constexpr int kChunkBlocks = 16, kChunkPieces = 34, kChunkPitch = 16 * kChunkPieces;
typedef uint32_t cu32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t cu32x4_a1 __attribute__((ext_vector_type(4), aligned(1)));

template <int ROWS>
struct RowChunks {
    static constexpr int N = ROWS * kChunkPieces, PER = (N + 63) / 64;
    typedef cu32x4 V[PER];
    const uint8_t* base;
    uint32_t off[PER], dst[PER];
    int pc[PER], nch, last;  // this lane's pieces of a row; chunks; where a row's last 16 bytes start

    __device__ __forceinline__ RowChunks(const uint8_t* W, int row0, int m_weight, int nb) {
        const int64_t bpr = (int64_t)nb * kQ80Bytes;
        const int first = min(row0, m_weight - 1), lane = threadIdx.x & 63;
        base = W + first * bpr;
        nch = (nb + kChunkBlocks - 1) / kChunkBlocks;
        last = (int)bpr - 16;
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int f = min(lane + 64 * k, N - 1), r = f / kChunkPieces;
            pc[k] = f % kChunkPieces;
            off[k] = (uint32_t)((min(row0 + r, m_weight - 1) - first) * bpr);
            dst[k] = (uint32_t)(r * kChunkPitch + 16 * pc[k]);
        }
    }
    __device__ __forceinline__ void load(V& v, int c) const {  // chunks past the last: the last again
        const int at = min(c, nch - 1) * kChunkPitch;
#pragma unroll
        for (int k = 0; k < PER; k++)
            v[k] = *reinterpret_cast<const cu32x4_a1*>(base + (off[k] + (uint32_t)min(at + 16 * pc[k], last)));
    }
    __device__ __forceinline__ void end(V& v) const {  // v: chunk nch - 1
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int past = (nch - 1) * kChunkPitch + 16 * pc[k] - last;
            if (past <= 0) continue;
            const unsigned __int128 x = __builtin_bit_cast(unsigned __int128, v[k]);
            v[k] = __builtin_bit_cast(cu32x4, past >= 16 ? (unsigned __int128)0 : x >> (8 * past));
        }
    }
    __device__ __forceinline__ void store(uint8_t* slot, const V& v) const {
#pragma unroll
        for (int k = 0; k < PER; k++)
            if (k < PER - 1 || N % 64 == 0 || (int)(threadIdx.x & 63) + 64 * k < N)
                *reinterpret_cast<cu32x4*>(slot + dst[k]) = v[k];
    }
};

// Up to kGemmMulti weight matrices that share the activation rows X (a prefill's
// Q, K and V) in one launch: workgroup column bx takes row block bx - first[i]
// of matrix i.
constexpr int kGemmMulti = 3;
struct GemmW {
    const uint8_t* w[kGemmMulti];
    float* out[kGemmMulti];
    int m[kGemmMulti];
    int first[kGemmMulti + 1];  // row blocks before matrix i
    uint8_t* yq;                // SwiGLU pairs: Q8_0 rows of y = silu(gate) * up, m[0] / 32 blocks per token
};

// The launch arguments of n <= kGemmMulti matrices in row blocks of R.
template <int R>
static GemmW gemm_args(const uint8_t* const* W, float* const* out, const int* M, int n) {
    GemmW g{};
    int blocks = 0;
    for (int i = 0; i < kGemmMulti; i++) {
        const int q = i < n ? i : 0;
        g.first[i] = blocks;
        g.w[i] = W[q];
        g.out[i] = out[q];
        g.m[i] = M[q];
        if (i < n) blocks += (M[i] + R - 1) / R;
    }
    g.first[kGemmMulti] = blocks;
    return g;
}

// Workgroup b of nP * nT (row panels x token tiles) takes panel bx, token tile
// by.  Workgroups go to the 8 XCDs round robin (b % 8), each with its own L2:
// when nP divides into 8, panel p runs on XCD p % 8 and its nT token tiles are
// numbered within one run of 8 nT workgroups, so they run together and read the
// panel's weight rows from one L2 (numbered panel-major, tiles of one panel ran
// a whole grid row apart, and a launch of more workgroups than fit at once read
// each panel twice).
__device__ __forceinline__ void sh_tile(int b, int nP, int nT, int& bx, int& by) {
    if ((nP & 7) == 0) {
        const int g = b / (8 * nT), r = b % (8 * nT);
        by = r >> 3;
        bx = 8 * g + (r & 7);
    } else {
        bx = b % nP;
        by = b / nP;
    }
}

// ----------------------------------------------------------------------------
// NaN cells of the scalar order S.  The reference computes
//   acc = acc + float(S_b) * (Ad*Bd)   over blocks b in order
// on x86, where the first NaN of the chain sticks (acc + p keeps acc's NaN), a
// NaN factor comes out quieted (the first operand's when both are NaN) and
// Inf*0, Inf-Inf give the default NaN.  Two reference forms differ in their NaN
// bits:
//   kSNanTile (the scalar tiles, bench/bpd_gemm_q8_0_cpu.c:112-128): scales by
//     the ldexpf decode of :13-26 (an f16 NaN becomes +/-0x7FC00000, no payload);
//     the build puts Bd first in Ad*Bd;
//   kSNanQdot (bpd_qdot_q8_0_q8_0_cpu's scalar form, bench/bpd_cpu.c:4263-4280,
//     which the scalar build's llamafile entry uses): the magic-number decode
//     (payload kept); the weight scale first.
// A finite scale product keeps a finite accumulator finite (|S_b*Ad*Bd| < 2^51)
// and an infinite one unchanged, so only blocks with an Inf or NaN scale can
// change the state, and the first NaN event fixes the bits.  Called only for a
// cell whose sum came out NaN; NaN-ness itself is the same on every IEEE machine.
// ----------------------------------------------------------------------------
constexpr int kSNanTile = 0;
constexpr int kSNanQdot = 1;
static_assert(kSNanTile != kSNanQdot, "the two NaN forms");

__device__ __forceinline__ float f16_ref(uint32_t h, int mode) {
    if (!f16_is_nan(h)) return f16_ieee(h);
    return mode == kSNanTile ? __uint_as_float(((h & 0x8000u) << 16) | 0x7FC00000u) : f16_nan_x86(h);
}

__device__ __noinline__ inline float s_order_nan_bits(const uint8_t* __restrict__ wrow,
                                                      const uint8_t* __restrict__ xrow, int nb, int mode) {
    float acc = 0.0f;  // stands for any finite value
    for (int b = 0; b < nb; b++) {
        const uint8_t* wb = wrow + (int64_t)b * kQ80Bytes;
        const uint8_t* xb = xrow + (int64_t)b * kQ80Bytes;
        const uint32_t hw = (uint32_t)wb[0] | ((uint32_t)wb[1] << 8);
        const uint32_t hx = (uint32_t)xb[0] | ((uint32_t)xb[1] << 8);
        if (!f16_exp31(hw) && !f16_exp31(hx)) continue;
        const float fw = f16_ref(hw, mode), fx = f16_ref(hx, mode);
        const float first = mode == kSNanTile ? fx : fw, second = mode == kSNanTile ? fw : fx;
        const float delta = first * second;
        // a NaN product: p = float(S_b) * delta is delta's NaN, and acc + p is p's
        if (__builtin_isnan(delta)) return x86_nan_of(first, second);
        // delta is +/-Inf: p = +/-Inf, or the default NaN when S_b = 0
        int sumi = 0;
        for (int j = 0; j < 32; j++) sumi += (int)(int8_t)wb[2 + j] * (int)(int8_t)xb[2 + j];
        if (sumi == 0) return __uint_as_float(kX86NaN);
        const float p = sumi < 0 ? -delta : delta;
        if (__builtin_isinf(acc) && acc != p) return __uint_as_float(kX86NaN);  // Inf - Inf
        acc = p;
    }
    return acc;
}

}  // namespace bpdq

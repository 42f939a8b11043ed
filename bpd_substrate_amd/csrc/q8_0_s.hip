// q8_0_s.hip — Q8_0 x Q8_0 for few activation rows in the scalar order S
// (bench/bpd_gemm_q8_0_cpu.c:102-131, bench/bpd_cpu.c:4263-4280), on int8 MFMA.
#include <algorithm>
#include <mutex>

#include "bpdq_device.h"
#include "bpdq_launch.h"
#include "bpdq_q8_0.h"

namespace bpdq {

// ----------------------------------------------------------------------------
// k_q8_0_gemm_SQ.  Per cell  acc = RN(acc + RN(float(S_b) * RN(Ad_b * Bd_b)))  over the
// blocks in order, S_b the exact dot of the cell's two blocks.  k_q8_0_gemm_SH stages 128
// tokens for any token count and waits for one half-stage of 4 blocks at a time, so a few
// tokens cost what 128 do and every 4 blocks a memory round trip: 14336x8, K = 4096, 46 us
// there, 18 here (62 MB at 3.5 TB/s; 128256x1 230 and 103 us, 5.4 TB/s).  What bounds it: the
// memory where the launch fills the chip; with few rows, a wave's own instructions.  For any C a
// wave issues 57 VALU and MFMA instructions per 4 blocks (16 conversions, 16 multiplications, 16
// additions, 4 realignments, 5 MFMA), about 290 cycles at the 5 cycles that a wave alone on its
// SIMD needs for each; 4096x1 (64 workgroups, one wave per SIMD) takes 13.6 us with C = 4 and 17.6
// with C = 16, 660 and 960 cycles per 4 blocks beyond the launch and the staging: the rest is
// operand reads from LDS (lanes of equal tokens share them) and the staging of the next chunk,
// not taken apart further.  Here the workgroup puts
// its C activation rows into LDS once; after that barrier each wave runs by itself over its
// 16 rows: chunks of 16 blocks as 16-byte pieces, two chunks in flight in registers, through
// its own LDS slot (a wave's LDS operations execute in order, so the next chunk is written
// behind the last reads of this one without a wait).  One v_mfma_i32_16x16x32_i8 is one
// block of 16 rows x 16 tokens; the scale products of four blocks come from one
// v_mfma_f32_16x16x4_4b_f16 (scales at inner index 0, zeros elsewhere: exact), so a tile and
// block costs the 12 VALU operations of the order (convert, multiply, add for 4 cells per
// lane) and one realignment.  Any K and any alignment (the pieces
// are 16-byte loads at any address), as long as the activation fits in LDS.
// LDS: a weight row's chunk at an odd multiple of 8 dwords (16 rows x 4 eight-byte groups of
// a block meet each bank twice, the least for 512 bytes); the quants of C tokens of a block
// are contiguous.
// ----------------------------------------------------------------------------
typedef _Float16 sh16x4 __attribute__((ext_vector_type(4)));
typedef float sf32x16 __attribute__((ext_vector_type(16)));
typedef int si32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t su32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t su32x4_a1 __attribute__((ext_vector_type(4), aligned(1)));

constexpr int kSqSlot = 16 * kChunkPitch;  // a wave's 16 rows
constexpr int kSqMaxLds = 160 * 1024;

// blocks of the activation in LDS: whole groups of 4, zeros past the end (a zero block adds
// +0 to a sum that is never -0)
__host__ __device__ constexpr int sq_blocks(int nb) { return (nb + 3) / 4 * 4; }
// bytes of LDS: quants [blocks][C][32], f16 scales [blocks][C], the waves' slots
__host__ __device__ constexpr size_t sq_lds(int C, int nw, int nb) {
    return (size_t)sq_blocks(nb) * C * 34 + (size_t)nw * kSqSlot;
}

// The operands of blocks 4t .. 4t+3 of a chunk.
struct SqOps {
    uint32_t a[4][3];  // even blocks: 3 dwords from 2 bytes before the quants; odd ones: 2
    uint32_t da, db;   // the scales of block 4t + lane / 16: this lane's row, this lane's token
    uint2 b[4];
};

template <int C>
__device__ __forceinline__ void sq_read(SqOps& o, const uint8_t* wq, const uint8_t* wd, const uint8_t* xq,
                                        const uint16_t* xd, int t) {
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int off = 34 * (4 * t + u);
        if (u & 1) {
            o.a[u][0] = *reinterpret_cast<const uint32_t*>(wq + off + 2);
            o.a[u][1] = *reinterpret_cast<const uint32_t*>(wq + off + 6);
        } else {
#pragma unroll
            for (int i = 0; i < 3; i++) o.a[u][i] = *reinterpret_cast<const uint32_t*>(wq + off + 4 * i);
        }
        o.b[u] = *reinterpret_cast<const uint2*>(xq + (4 * t + u) * C * 32);
    }
    o.da = *reinterpret_cast<const uint16_t*>(wd + 136 * t);
    o.db = xd[4 * t * C];
}

__device__ __forceinline__ void sq_group(const SqOps& o, float (&acc)[4]) {
    const sf32x16 fzero = {0.0f};
    const si32x4 zero = {0, 0, 0, 0};
    const sf32x16 delta =
        __builtin_amdgcn_mfma_f32_16x16x4f16(__builtin_bit_cast(sh16x4, make_uint2(o.da, 0u)),
                                             __builtin_bit_cast(sh16x4, make_uint2(o.db, 0u)), fzero, 0, 0, 0);
    si32x4 s[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const uint2 w = u & 1 ? make_uint2(o.a[u][0], o.a[u][1])
                              : make_uint2(__builtin_amdgcn_alignbit(o.a[u][1], o.a[u][0], 16),
                                           __builtin_amdgcn_alignbit(o.a[u][2], o.a[u][1], 16));
        s[u] = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, w), __builtin_bit_cast(long, o.b[u]), zero,
                                                     0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[r] = acc[r] + (float)s[u][r] * delta[4 * u + r];
    // the group's arithmetic ends here (the compiler would move every group's to the end of
    // the unrolled chunk and spill)
    asm volatile("" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
}

template <int C, int NW>
__global__ __launch_bounds__(64 * NW) void k_q8_0_gemm_SQ(GemmW gw, const uint8_t* __restrict__ X, int m_tokens, int nb,
                                                          int nan_mode) {
    constexpr int R = 16 * NW, NT = 64 * NW;
    extern __shared__ __align__(16) uint8_t sqlds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int bx, by;
    sh_tile(blockIdx.x, gw.first[kGemmMulti], (m_tokens + C - 1) / C, bx, by);
    const int mi = (bx >= gw.first[1]) + (bx >= gw.first[2]);
    const uint8_t* __restrict__ W = gw.w[mi];
    float* __restrict__ out = gw.out[mi];
    const int m_weight = gw.m[mi];
    const int row0 = (bx - gw.first[mi]) * R + wave * 16, n0 = by * C;
    const int64_t bpr = (int64_t)nb * kQ80Bytes;
    const int nch = (nb + 15) / 16, nbp = sq_blocks(nb);
    const RowChunks<16> rows(W, row0, m_weight, nb);
    uint8_t* xs = sqlds;
    uint16_t* xsc = reinterpret_cast<uint16_t*>(sqlds + (size_t)nbp * C * 32);
    uint8_t* slot = sqlds + (size_t)nbp * C * 34 + wave * kSqSlot;
    const auto wstore = [&](const RowChunks<16>::V& v) {
        asm volatile("" ::: "memory");  // behind the reads of the previous chunk
        rows.store(slot, v);
        asm volatile("" ::: "memory");
    };

    // the activation: unit i is token i % C, half (i / C) & 1 of block i / (2 C); the first
    // batch is loaded before the weights (loads return in order)
    constexpr int XU = 4;
    su32x4 xv[XU];
    uint32_t xh[XU];
    const int nu = 2 * C * nb, nup = 2 * C * nbp;
    const auto xload = [&](int i0) {
#pragma unroll
        for (int u = 0; u < XU; u++) {
            const int i = min(i0 + u * NT, nu - 1);
            const uint8_t* s = X + (int64_t)min(n0 + i % C, m_tokens - 1) * bpr + (i / (2 * C)) * kQ80Bytes;
            xv[u] = *reinterpret_cast<const su32x4_a1*>(s + 2 + 16 * ((i / C) & 1));
            xh[u] = ld_u16(s);
        }
    };
    const auto xstore = [&](int i0) {
#pragma unroll
        for (int u = 0; u < XU; u++) {
            const int i = i0 + u * NT, t = i % C, h = (i / C) & 1, b = i / (2 * C);
            if (i >= nup) continue;
            *reinterpret_cast<su32x4*>(xs + ((size_t)b * C + t) * 32 + 16 * h) = i < nu ? xv[u] : su32x4{0, 0, 0, 0};
            if (h == 0) xsc[b * C + t] = i < nu ? (uint16_t)xh[u] : (uint16_t)0;
        }
    };
    RowChunks<16>::V wv[2];
    xload(tid);
    __builtin_amdgcn_sched_barrier(0);
    rows.load(wv[0], 0);
    rows.load(wv[1], 1);
    __builtin_amdgcn_sched_barrier(0);
    xstore(tid);
    for (int i0 = tid + XU * NT; i0 < nup; i0 += XU * NT) {
        xload(i0);
        xstore(i0);
    }
    lds_barrier();

    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const int j = lane & 15, k = lane >> 4;
    const uint8_t* wq = slot + j * kChunkPitch + 8 * k;   // this lane's row, eight quants from 8 k
    const uint8_t* wd = slot + j * kChunkPitch + 34 * k;  // the scale of block k of a group of four
    const uint8_t* xq = xs + (j % C) * 32 + 8 * k;     // columns past C repeat tokens (not stored)
    const uint16_t* xd = xsc + k * C + j % C;
    SqOps o[2];
    if (nch == 1) rows.end(wv[0]);
    wstore(wv[0]);
    rows.load(wv[0], 2);
    sq_read<C>(o[0], wq, wd, xq, xd, 0);
    // a whole chunk of 4 groups; the next chunk goes into the slot behind the last group's reads
    const auto step = [&](RowChunks<16>::V& next, int c) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if (t < 3) {
                sq_read<C>(o[(t + 1) & 1], wq, wd, xq, xd, t + 1);
            } else {
                xq += 16 * C * 32;
                xd += 16 * C;
                if (c + 2 == nch) rows.end(next);
                wstore(next);
                rows.load(next, c + 3);
                sq_read<C>(o[0], wq, wd, xq, xd, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            sq_group(o[t & 1], acc);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int c = 0;
    for (; c + 2 < nch; c += 2) {
        step(wv[1], c);
        step(wv[0], c + 1);
    }
    if (c + 1 < nch) {
        step(wv[1], c);
        c++;
    }
    // the last chunk: 1 to 4 groups, the first already read
    const int ng = (nb - 16 * c + 3) / 4;
#pragma unroll 1
    for (int t = 0; t < ng; t += 2) {
        sq_read<C>(o[1], wq, wd, xq, xd, min(t + 1, ng - 1));
        sq_group(o[0], acc);
        if (t + 1 == ng) break;
        sq_read<C>(o[0], wq, wd, xq, xd, min(t + 2, ng - 1));
        sq_group(o[1], acc);
    }

    // register r of lane l: row 4 (l / 16) + r of the wave's 16, token l % 16
    const int tok = n0 + j, r0 = row0 + 4 * k;
    if (j >= C || tok >= m_tokens) return;
#pragma unroll
    for (int r = 0; r < 4; r++)
        if (__builtin_isnan(acc[r]) && r0 + r < m_weight)
            acc[r] = s_order_nan_bits(W + (r0 + r) * bpr, X + tok * bpr, nb, nan_mode);
    float* o_ = out + (int64_t)tok * m_weight + r0;
    if ((reinterpret_cast<uintptr_t>(o_) & 15) == 0 && r0 + 4 <= m_weight) {
        *reinterpret_cast<float4*>(o_) = make_float4(acc[0], acc[1], acc[2], acc[3]);
    } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (r0 + r < m_weight) o_[r] = acc[r];
    }
}

template <int C, int NW>
static bool launch_sq(const uint8_t* const* W, float* const* out, const int* M, int n, const uint8_t* Xq, int m_tokens,
                      int nb, int nan_mode, hipStream_t s) {
    const size_t lds = sq_lds(C, NW, nb);
    if (lds > kSqMaxLds) return false;
    if (lds > 64 * 1024) {  // asked for once per process
        static std::once_flag once;
        static bool ok = false;
        std::call_once(once, [] {
            ok = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_q8_0_gemm_SQ<C, NW>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, kSqMaxLds) == hipSuccess;
            (void)hipGetLastError();
        });
        if (!ok) return false;
    }
    const GemmW g = gemm_args<16 * NW>(W, out, M, n);
    hipLaunchKernelGGL((k_q8_0_gemm_SQ<C, NW>), dim3(g.first[kGemmMulti] * ((m_tokens + C - 1) / C)), dim3(64 * NW), lds, s,
                       g, Xq, m_tokens, nb, nan_mode);
    return true;
}

// Estimated times (ns) of a launch over the rows and tokens of n matrices.  Its workgroups run
// in `per` = ceil(workgroups / 256) per CU however many of their rows and tokens are real, so
// it is fixed + step * per + K * g(per), g the ns per element of K: g1 for one workgroup per CU,
// else gs[o - 1] per workgroup where LDS lets o of them run at once (2.25 against 1.85 for 4
// tokens, 4.3 against 2.85 for 16, where one has the CU to itself).  An odd number of blocks
// leaves the rows off the 4-byte grid: `odd` times that.  Fitted to 950 shapes on MI355X, weights
// beyond the MALL (512 to 128256 rows, 1 to 512 tokens, K 1024 to 28672): the choice is on the
// average 0.2 % and at most 16 % over the best form, and no shape is more than 4 % slower than
// k_q8_0_gemm_SH and k_q8_0_gemm_S.  us, 4 / 8 / 16 tokens x 64 rows / 16 x 128 / those two:
//   K = 1024   32000x8 21 / 13 / 15 / 15 / 20; 32000x17 39 / 28 / 22 / 26 / 20
//   K = 1440   14336x64 74 / 43 / 32 / 32 / 57
//   K = 4096   14336x1 17 / 18 / 20 / 27 / 47; 14336x16 40 / 27 / 23 / 32 / 47; 14336x48 95 / 65 / 60 / 60 / 49
//              4096x64 40 / 27 / 22 / 30 / 43; 128256x1 103 / 108 / 140 / 123 / 230
//   K = 8192   8192x64 130 / 100 / - / - / 83; 32000x17 207 / 167 / - / - / 128
struct SqForm {
    int rows, tokens;
    double step, g1, gs[3], odd;
    bool (*launch)(const uint8_t* const*, float* const*, const int*, int, const uint8_t*, int, int, int, hipStream_t);
};
static constexpr SqForm kSqForms[] = {{64, 4, 800, 1.85, {2.25, 2.15, 1.85}, 1.55, launch_sq<4, 4>},
                                      {64, 8, 800, 2.1, {2.85, 2.15, 2.15}, 1.5, launch_sq<8, 4>},
                                      {64, 16, 800, 2.85, {4.3, 3.4, 2.85}, 1.25, launch_sq<16, 4>},
                                      {128, 16, 1600, 5.2, {6.5, 6.5, 6.5}, 1.35, launch_sq<16, 8>}};

static int64_t tiles(const int* M, int n, int m_tokens, int rows, int tokens) {
    int64_t b = 0;
    for (int i = 0; i < n; i++) b += (M[i] + rows - 1) / rows;
    return b * ((m_tokens + tokens - 1) / tokens);
}

static const SqForm* sq_best(const int* M, int n, int m_tokens, int K, double* ns) {
    const int nb = K / 32;
    const SqForm* best = nullptr;
    *ns = 0;
    for (const SqForm& f : kSqForms) {
        const size_t lds = sq_lds(f.tokens, f.rows / 16, nb);
        if (lds > kSqMaxLds) continue;
        const int at_once = std::min<int>((int)(kSqMaxLds / lds), 3);
        const double per = (double)((tiles(M, n, m_tokens, f.rows, f.tokens) + 255) / 256);
        const double g = (per == 1 ? f.g1 : f.gs[at_once - 1] * per) * (nb % 2 != 0 ? f.odd : 1.0);
        const double t = 4000 + f.step * per + K * g;
        if (best != nullptr && t >= *ns) continue;
        best = &f;
        *ns = t;
    }
    return best;
}

// k_q8_0_gemm_SH (staged) by its three forms, k_q8_0_gemm_S otherwise.
static double sh_ns(const int* M, int n, int m_tokens, int K, bool staged) {
    const auto wgs = [&](int rows) { return tiles(M, n, m_tokens, rows, 128); };
    if (!staged) {
        const double fixed = m_tokens <= 64 ? 4600 : 8600, g = m_tokens <= 64 ? 32.5 : 36.5;
        return fixed + K * std::max(g, 0.096 * (double)wgs(128));
    }
    const double g = wgs(128) >= 256 ? (wgs(128) <= 512 ? 27.0 : 28.0 * (double)((wgs(128) + 511) / 512))
                     : wgs(64) >= 256 ? 15.0
                     : wgs(32) > 256  ? 11.3
                                      : 9.4;
    return 3000 + K * g;
}

bool launch_q8_0_gemm_S_few(const uint8_t* const* W, float* const* out, const int* M, int n, const uint8_t* Xq,
                            int m_tokens, int K, bool staged, int nan_mode, hipStream_t s) {
    if (K / 32 == 0) return false;
    double ns;
    const SqForm* form = sq_best(M, n, m_tokens, K, &ns);
    if (form == nullptr || ns >= 0.97 * sh_ns(M, n, m_tokens, K, staged)) return false;
    return form->launch(W, out, M, n, Xq, m_tokens, K / 32, nan_mode, s);
}

// The epilogue form takes 64 rows of gate and of up x 128 tokens per workgroup, so a few tokens
// cost what 128 do: about 16.5 ns per element of K for up to 256 workgroups, 25.7 for each 512
// beyond; k_swiglu costs 2.5 us and 4.5 us per million values.  us, epilogue / apart, K = 4096:
// 4096x16 73 / 20, 14336x16 75 / 39, 14336x32 76 / 65, 14336x96 77 / 80, 28672x24 115 / 122;
// K = 1024: 14336x17 25 / 23, 28672x32 37 / 40; K = 8192: 4096x64 140 / 107, 14336x32 144 / 129.
bool q8_0_swiglu_S_apart(int F, int m_tokens, int K) {
    const int M[2] = {F, F};
    double ns;
    const bool few = K / 32 > 0 && sq_best(M, 2, m_tokens, K, &ns) != nullptr;
    const double sh = sh_ns(M, 2, m_tokens, K, true);
    const double apart = (few ? std::min(ns, sh) : sh) + 2500 + 4.5e-3 * (double)F * m_tokens;
    const int64_t wgs = tiles(M, 1, m_tokens, 64, 128);
    const double joint = wgs <= 256 ? 5200 + 0.2 * F + 16.5 * K : 10000 + 25.7 * K * (double)((wgs + 511) / 512);
    return apart < 0.95 * joint;
}

}  // namespace bpdq

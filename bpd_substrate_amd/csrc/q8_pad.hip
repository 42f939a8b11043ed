// q8_pad.hip — the padded Q8 layout [K/32][N][64] (records {f16 d, 0, 0, int8 q[32],
// 28 zero bytes}): the order-T product of one activation row, and of a gate/up pair with
// SwiGLU.
#include <algorithm>
#include <mutex>
#include <numeric>

#include "bpdq_device.h"
#include "bpdq_launch.h"
#include "bpdq_math.h"
#include "bpdq_q8_0.h"

namespace bpdq {

// ----------------------------------------------------------------------------
// k_pad_gemv.  Block b of 16 consecutive rows is 1 KB of contiguous records, one
// 12-byte load per lane: lane (row, p) of a wave loads bytes 8p..8p+11 of its record,
// i.e. the quant dwords L = 2p and 2p + 1 in its last two dwords and, for p = 0, the
// scale in the first, which the quad takes by DPP.  The lane runs the chains
//   acc_L = RN(RN(RN(Ad*Bd) * p_L) + acc_L)
// of its two L over all blocks in order, with the loads of the next U blocks in flight,
// and the quad ends with the hsum ((a0+a4)+(a2+a6))+((a1+a5)+(a3+a7)): nothing but the
// activation row goes through LDS, as one 16-byte read {2 quant dwords, scale} per block.
// The kernel needs 11 VALU operations per block for 16 rows, so it streams at the rate
// its loads in flight allow.  NW waves of 16 rows per workgroup, NH more that only help
// stage the activation row.
// ----------------------------------------------------------------------------
constexpr int kPadG = 4;  // blocks per group
constexpr int kPadX = 8;  // activation units in flight per thread

struct PadRec {
    uint32_t a, lo, hi;
};

__device__ __forceinline__ PadRec pad_load(const uint8_t* p) {
    PadRec r;
    __builtin_memcpy(&r, __builtin_assume_aligned(p, 4), 12);
    return r;
}

template <int NW, int NH, int U, bool SWG>
__global__ __launch_bounds__(64 * (NW + NH)) void k_pad_gemv(GemmW gw, const uint8_t* __restrict__ Xq, int nb) {
    static_assert(U % (2 * kPadG) == 0, "the activation slots alternate");
    static_assert(!SWG || (NW == 4 && NH == 0), "two gate and two up waves");
    constexpr int NT = 64 * (NW + NH);
    extern __shared__ __align__(16) uint4 xs[];  // [nb + kPadG][4]: quant dwords 2p, 2p + 1, scale
    __shared__ uint32_t wave_m128[NW + NH];
    __shared__ float gu[SWG ? 64 : 1];
    const int tid = threadIdx.x, lane = tid & 63, p = lane & 3, tok = blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bx = blockIdx.x;
    const int mi = SWG ? wave >> 1 : (bx >= gw.first[1]) + (bx >= gw.first[2]);
    const uint8_t* __restrict__ W = gw.w[mi];
    const int N = gw.m[mi];
    const int row0 = SWG ? bx * 32 + 16 * (wave & 1) : (bx - gw.first[mi]) * 16 * NW + 16 * min(wave, NW - 1);
    const int row = min(row0 + (lane >> 2), N - 1);  // rows past the end repeat the last one
    const int64_t stride = (int64_t)N * 64;
    const int base = min(row0, N - 1);
    const uint8_t* wb = W + (int64_t)base * 64;
    const bool work = wave < NW;

    // loads go out in groups of kPadG blocks; wnext is the next block to load (past the end
    // the last block again, unused)
    PadRec r[U];
    const uint32_t off = (uint32_t)(row - base) * 64 + 8 * p;
    const uint8_t* wnext = wb;
    int issued = 0;
    const auto load = [&](PadRec (&q)[U], int u0) {
#pragma unroll
        for (int u = u0; u < u0 + kPadG; u++) {
            q[u] = pad_load(wnext + off);
            issued++;
            wnext += issued < nb ? stride : 0;
        }
    };
    // the activation row: unit i is dwords 2p, 2p + 1 of block i / 4.  The first kPadX
    // units per thread are loaded before the weights (loads return in order), the rest
    // (rows over kPadX * NT / 4 blocks) after them.
    const uint8_t* xr = Xq + (int64_t)tok * nb * kQ80Bytes;
    uint32_t any_m128 = 0;
    uint32_t q0[kPadX], q1[kPadX], d[kPadX];
    const auto xload = [&](int i0) {
#pragma unroll
        for (int k = 0; k < kPadX; k++) {
            const int i = min(i0 + k * NT, 4 * nb - 1);
            const uint8_t* s = xr + (i >> 2) * kQ80Bytes;
            q0[k] = ld_u32(s + 2 + 8 * (i & 3));
            q1[k] = ld_u32(s + 6 + 8 * (i & 3));
            d[k] = ld_u16(s);
        }
    };
    const auto xstore = [&](int i0) {
#pragma unroll
        for (int k = 0; k < kPadX; k++)
            if (i0 + k * NT < 4 * nb) {
                xs[i0 + k * NT] = make_uint4(q0[k], q1[k], __float_as_uint(f16_ieee(d[k])), 0u);
                any_m128 |= has_m128(q0[k]) | has_m128(q1[k]);
            }
    };
    xload(tid);
    __builtin_amdgcn_sched_barrier(0);
    if (work) {
#pragma unroll
        for (int u = 0; u < U; u += kPadG) load(r, u);
    }
    __builtin_amdgcn_sched_barrier(0);
    xstore(tid);
    for (int i0 = tid + kPadX * NT; i0 < 4 * nb; i0 += kPadX * NT) {
        xload(i0);
        xstore(i0);
    }
    {
        const bool m = __ballot(any_m128 != 0) != 0;
        if (lane == 0) wave_m128[wave] = m ? 1u : 0u;
    }
    lds_barrier();
    if (!work) return;
    uint32_t xm128 = 0;
#pragma unroll
    for (int i = 0; i < NW + NH; i++) xm128 |= wave_m128[i];

    float a0 = 0.0f, a1 = 0.0f;
    const auto use = [&](const PadRec& w, const uint4& x) {
        const float delta = f16_ieee((uint32_t)dpp_i<0x00>((int)w.a)) * __uint_as_float(x.z);  // the quad's lane 0
        const float p0 = delta * (float)sdot4(w.lo, x.x, 0), p1 = delta * (float)sdot4(w.hi, x.y, 0);
        a0 = p0 + a0;
        a1 = p1 + a1;
    };
    // the next group's activation is read, and this group's slots are refilled, around the
    // group's arithmetic, in that order (so a group waits for its own loads only)
    uint4 x[2][kPadG];
    const uint4* xp = xs + p;  // nb blocks, then kPadG spare ones that are read and not used
#pragma unroll
    for (int g = 0; g < kPadG; g++) x[0][g] = xp[4 * g];
    int b = 0;
    for (; b + U <= nb; b += U) {
#pragma unroll
        for (int u = 0; u < U; u += kPadG) {
            const int h = (u / kPadG) & 1;
#pragma unroll
            for (int g = 0; g < kPadG; g++) x[h ^ 1][g] = xp[4 * (b + u + kPadG + g)];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < kPadG; g++) use(r[u + g], x[h][g]);
            __builtin_amdgcn_sched_barrier(0);
            load(r, u);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++)
        if (b + u < nb) use(r[u], xp[4 * (b + u)]);
    a0 = a0 + dpp_f<0x4E>(a0);  // L ^ 4
    a0 = a0 + dpp_f<0xB1>(a0);  // L ^ 2
    a1 = a1 + dpp_f<0x4E>(a1);
    a1 = a1 + dpp_f<0xB1>(a1);
    float y = a0 + a1;
    const bool writes = p == 0 && row0 + (lane >> 2) < N;
    if (writes && (__builtin_isnan(y) || xm128 != 0))
        y = t_order_cell(W + (int64_t)row * 64, stride, 4, xr, nb, row, tok, N, (int)gridDim.y);
    if constexpr (SWG) {
        if (p == 0) gu[16 * wave + (lane >> 2)] = y;
        __syncthreads();
        if (tid < 32) {
            const float g = gu[tid], u = gu[32 + tid];
            const float v = (g / (1.0f + expf_libm(-g))) * u;
            gw.out[0][bx * 32 + tid] = v;
            q8_0_lane_store(v, gw.yq + (int64_t)bx * kQ80Bytes, tid);
        }
    } else {
        if (writes) gw.out[mi][(int64_t)tok * N + row] = y;
    }
}

constexpr int kPadMaxLds = 160 * 1024;
constexpr int kPadMaxNb = 2540;  // blocks whose activation fits in it
constexpr size_t pad_lds(int nb) { return (size_t)(nb + kPadG) * 64; }

template <int NW, int NH, int U, bool SWG>
static bool launch_pad(const GemmW& g, int blocks, int m_tokens, const uint8_t* Xq, int nb, hipStream_t s) {
    const size_t lds = pad_lds(nb);
    if (nb > kPadMaxNb) return false;
    if (lds > 64 * 1024 - 512) {  // asked for once per process
        static std::once_flag once;
        static bool ok = false;
        std::call_once(once, [] {
            ok = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_pad_gemv<NW, NH, U, SWG>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)pad_lds(kPadMaxNb)) == hipSuccess;
            (void)hipGetLastError();
        });
        if (!ok) return false;
    }
    hipLaunchKernelGGL((k_pad_gemv<NW, NH, U, SWG>), dim3(blocks, m_tokens), dim3(64 * (NW + NH)), lds, s, g, Xq, nb);
    return true;
}

// n <= 3 matrices of N[i] >= 1 rows: 64 rows per workgroup (4 waves), or 16 rows and three waves
// that help to stage the activation, or false for k_q8_0_gemv_TP, which splits the products
// from the chains of its 8 rows.  us on MI355X, weights beyond the MALL, TP / 16 rows / 64 rows:
//   few cells (rows * tokens), the chains set the time:
//     K = 1024   1024x1 4.0 / 4.9 / 4.9, 4096x1 4.8 / 5.0 / 5.0, 5120x1 7.0 / 5.7 / 5.2
//     K = 4096   1024x1 6.0 / 8.9 / 9.6, 1024x4 7.3 / 9.0 / 9.6, 2048x2 7.8 / 9.3 / 10.0,
//                3584x1 9.4 / 9.9 / 14.5, 4096x1 10.2 / 9.9 / 14.3, 3072x2 13.8 / 10.7 / 14.0
//     K = 14336  1024x4 17.8 / 23.4 / 35.8, 3072x1 22.6 / 24.1 / 38.9, 4096x1 26.1 / 24.7 / 40.0
//     K = 512    2048x1 4.0 / 4.3 / 4.4, 4096x1 4.6 / 4.4 / 4.3; K = 128 1024x1 3.8 / 3.2 / 3.1
//   many: K = 4096 12288x1 - / 18.8 / 18.3, 28672x1 - / 41 / 40; 4096x14336 one row 24.7
//   16-row workgroups that do not run at once, long rows: K = 28672 3072x3 85 / 86 / 74,
//     K = 40960 3072x2 85 / 119 / 108, 2048x4 111 / 119 / 104
//   several tokens read a matrix once where its workgroups meet on an XCD again (a count that 8
//   divides): 7296x4 K = 1856 (456 / 114 workgroups) 13.3 / 18.0, 9689x2 K = 2880 (606 / 152)
//     23.2 / 14.0, 5568x3 K = 11552 (348 / 87) 49 / 66.
bool launch_pad_gemv(const uint8_t* const* W, float* const* y, const int* N, int n, const uint8_t* Xq, int m_tokens,
                     int K, bool ring_fits, hipStream_t s) {
    const int nb = K / 32;
    int64_t cells = 0;
    for (int i = 0; i < n; i++) cells += N[i];
    cells *= m_tokens;
    const GemmW g16 = gemm_args<16>(W, y, N, n), g64 = gemm_args<64>(W, y, N, n);
    const int b16 = g16.first[kGemmMulti], b64 = g64.first[kGemmMulti];
    // 16-row workgroups per CU: 4 waves of 52 VGPRs, the activation in LDS
    const int64_t at_once = std::min<int64_t>(8, kPadMaxLds / pad_lds(nb));
    const bool fits = (int64_t)b16 * m_tokens <= 256 * at_once;
    const int64_t few = !fits && at_once == 1 ? 6144 : K < 768 ? 3071 : m_tokens > 1 || K < 4096 ? 4096 : 3840;
    if (ring_fits && K >= 512 && cells <= few) return false;
    bool wide = cells >= 12288;
    if (m_tokens > 1) {
        const int x16 = std::gcd(b16, 8), x64 = std::gcd(b64, 8);
        if (x16 > x64) wide = cells >= 32768;
        if (x64 > x16) wide = cells >= 8192;
    }
    if (wide || !fits) return launch_pad<4, 0, 8, false>(g64, b64, m_tokens, Xq, nb, s);
    return launch_pad<1, 3, 16, false>(g16, b16, m_tokens, Xq, nb, s);
}

// Gate and up (F rows each, F % 32 == 0) of one activation row: y = silu(gate) * up and its
// Q8_0 blocks; false (nothing launched) where the activation does not fit in LDS, and for few
// rows of a long K, where two products and k_swiglu are faster: us, apart in brackets, 1024 rows
// K = 2048 7.3 (7.9), K = 4096 10.7 (10.1), K = 8192 25.4 (14.3), K = 14336 37.8 (19.5); 4096 rows
// K = 4096 17.0 (16.3), K = 14336 46.2 (42.5); 5632 rows K = 8192 31.7 (34.3).
bool launch_pad_swiglu(const uint8_t* Wg, const uint8_t* Wu, float* y, uint8_t* yq, int F, const uint8_t* Xq, int K,
                       hipStream_t s) {
    if (F <= 4096 && K >= 4096) return false;
    GemmW g{};
    for (int i = 0; i < kGemmMulti; i++) {
        g.w[i] = i == 1 ? Wu : Wg;
        g.out[i] = y;
        g.m[i] = F;
    }
    g.yq = yq;
    return launch_pad<4, 0, 8, true>(g, F / 32, 1, Xq, K / 32, s);
}

}  // namespace bpdq

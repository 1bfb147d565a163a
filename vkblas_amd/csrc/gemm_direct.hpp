// gemm_direct.hpp — GEMM on small tiles whose MFMA fragments come straight
// from global memory, for small and unaligned problems.
//
// Bound: latency.  Such a call has too few tiles to fill the chip and too
// little work per tile to hide a load behind a barrier, so the kernel keeps
// the chain from launch to store short instead of saving bytes: no LDS, no
// barrier and no branch in the K loop, and U K steps of loads in flight per
// wave.  One workgroup computes one TM x TN tile (TM = 16 MF, TN = 16 NF); its
// four waves take a quarter of the K steps each, the four sums are added in
// LDS in wave order (bitwise reproducible) and leave as row segments.
//
// A K step is 64 bytes of k (16 fp32, 32 fp16 / bf16): lane group g = lane /
// 16 takes the g-th 16 bytes.
//  * K-major operand (A with op_a = N, B with op_b = T): lane r + 16 g loads
//    16 bytes of row r of each 16-row fragment: v_mfma_f32_16x16x32 takes
//    them as they are, and four v_mfma_f32_16x16x4_f32 take one element each.
//    Rows past the matrix repeat its last row (their results are not stored).
//  * MN-major operand: lane r + 16 g loads columns MF r .. MF r + MF - 1 of
//    its k rows; column c of them is row r of fragment c, so fragment c holds
//    rows MF r + c of the tile.  fp32: element e of the four MFMAs is k row
//    4 g + e as it stands; 16-bit: v_perm gathers the column from 8 k rows.
//    The tile moves back inside the matrix at its edge (the launcher checks
//    M >= TM, N >= TN) and stores only what the tile before it does not.
//  * Loads are plain vector loads of any element alignment: an odd leading
//    dimension costs nothing.
//  * The step that crosses K loads element by element at clamped addresses
//    and zeroes what lies past K in both operands.
#pragma once
#include "gemm_mfma.hpp"

namespace vkb {

typedef uint32_t u32x2_d __attribute__((ext_vector_type(2)));

// N consecutive dwords from an address of any element alignment (2 bytes:
// gfx950's vector loads take it, the compiler splits nothing)
typedef uint32_t u32_any __attribute__((aligned(2), may_alias));
typedef u32x2_d u32x2_any __attribute__((aligned(2), may_alias));
template <int N>
__device__ __forceinline__ void ld_dwords(uint32_t* d, const void* p) {
    static_assert(N == 1 || N == 2 || N == 4, "1, 2 or 4 dwords");
    if constexpr (N == 1) {
        d[0] = *(const u32_any*)p;
    } else if constexpr (N == 2) {
        const u32x2_d v = *(const u32x2_any*)p;
        d[0] = v[0]; d[1] = v[1];
    } else {
        const u32x4 v = *(const u32x4_any*)p;
        d[0] = v[0]; d[1] = v[1]; d[2] = v[2]; d[3] = v[3];
    }
}

// One operand of the tile: F fragments of 16 rows (m of A or n of B).
template <typename T, bool KMAJ, int F>
struct DirectOperand {
    static constexpr int VEC = Elem<T>::VEC;    // elements of 16 bytes
    static constexpr int ROWS = VEC;            // k rows per lane and step (MN-major)
    static constexpr int RD = F * (int)sizeof(T) / 4;   // dwords per k row (MN-major)
    static_assert(KMAJ || RD >= 1, "an MN-major 16-bit operand needs F >= 2");
    const T* base;      // the slice's first k of the tile's first row / column (uniform)
    int64_t ld;
    uint32_t off[KMAJ ? F : 1];                 // per-lane byte offsets

    __device__ __forceinline__ void init(const T* p, int64_t ld_, int row0, int rows, int kbeg, int r, int g) {
        ld = ld_;
        if constexpr (KMAJ) {
            base = p + (int64_t)row0 * ld + kbeg;
#pragma unroll
            for (int i = 0; i < F; ++i)
                off[i] = (uint32_t)((int64_t)min(16 * i + r, rows - 1 - row0) * ld + g * VEC) * (uint32_t)sizeof(T);
        } else {
            base = p + (int64_t)kbeg * ld + row0;
            off[0] = (uint32_t)((int64_t)(ROWS * g) * ld + F * r) * (uint32_t)sizeof(T);
        }
    }
    // the loads of a whole step whose first k is kbeg + k
    __device__ __forceinline__ void load(uint32_t (&v)[4 * F], int k) const {
        if constexpr (KMAJ) {
            const char* b = (const char*)(base + k);
#pragma unroll
            for (int i = 0; i < F; ++i) ld_dwords<4>(v + 4 * i, b + off[i]);
        } else {
#pragma unroll
            for (int j = 0; j < ROWS; ++j)
                ld_dwords<RD>(v + RD * j, (const char*)(base + (int64_t)(k + j) * ld) + off[0]);
        }
    }
    // a step of which only the first nk k exist (0 < nk < 4 VEC): the others
    // are read at the last one that does and replaced by zero
    __device__ __forceinline__ void load_tail(uint32_t (&v)[4 * F], int k, int nk, int g) const {
        if constexpr (KMAJ) {
            const char* b = (const char*)(base + k);
#pragma unroll
            for (int i = 0; i < F; ++i) {
                uint32_t x[VEC];
                const T* row = (const T*)(b + off[i]) - g * VEC;
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const int kk = g * VEC + e;
                    const T* q = row + min(kk, nk - 1);
                    if constexpr (sizeof(T) == 4) x[e] = *(const uint32_t*)q;
                    else x[e] = *(const uint16_t*)q;
                    if (kk >= nk) x[e] = 0u;
                }
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    if constexpr (sizeof(T) == 4) v[4 * i + d] = x[d];
                    else v[4 * i + d] = x[2 * d] | (x[2 * d + 1] << 16);
                }
            }
        } else {
            const char* col = (const char*)(base + (int64_t)k * ld) + off[0] - (int64_t)(ROWS * g) * ld * sizeof(T);
#pragma unroll
            for (int j = 0; j < ROWS; ++j) {
                const int kk = ROWS * g + j;
                ld_dwords<RD>(v + RD * j, (const T*)col + (int64_t)min(kk, nk - 1) * ld);
#pragma unroll
                for (int d = 0; d < RD; ++d)
                    if (kk >= nk) v[RD * j + d] = 0u;
            }
        }
    }
    // fragment i: 16 bytes of k of tile row row_of(i, r)
    __device__ __forceinline__ u32x4 frag(const uint32_t (&v)[4 * F], int i) const {
        if constexpr (KMAJ) {
            return u32x4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
        } else if constexpr (sizeof(T) == 4) {
            return u32x4{v[i], v[F + i], v[2 * F + i], v[3 * F + i]};
        } else {
            u32x4 f;
            const uint32_t sel = (i & 1) ? 0x07060302u : 0x05040100u;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                f[q] = __builtin_amdgcn_perm(v[RD * (2 * q + 1) + i / 2], v[RD * (2 * q) + i / 2], sel);
            return f;
        }
    }
};

// T, TC, AK, BKM as gemm_kernel; MF x NF fragments of 16 rows / columns per
// workgroup, U K steps of loads in flight per wave.
template <typename T, typename TC, bool AK, bool BKM, int MF, int NF, int U>
__global__ __launch_bounds__(256) void gemm_direct_kernel(KParams p) {
    constexpr int TM = 16 * MF, TN = 16 * NF;
    constexpr int KS = 4 * Elem<T>::VEC;            // k per step
    constexpr int LDR = TN + 4;                     // padded row of the sums in LDS
    __shared__ float red[4][TM * LDR];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;

    // tile / batch / split decode with XCD-aware remap, as gemm_kernel
    uint32_t bid = blockIdx.x;
    const uint32_t nwg = gridDim.x;
    if ((nwg & 7u) == 0) bid = (bid & 7u) * (nwg >> 3) + (bid >> 3);
    const uint32_t per = p.tiles_m * p.tiles_n;
    const uint32_t z = bid / per;
    const uint32_t t = bid - z * per;
    const uint32_t b = z / p.split;
    const uint32_t s = z - b * p.split;
    const int m_lo = (int)(t % p.tiles_m) * TM, n_lo = (int)(t / p.tiles_m) * TN;
    const int m0 = AK ? m_lo : min(m_lo, (int)p.M - TM);
    const int n0 = BKM ? n_lo : min(n_lo, (int)p.N - TN);

    const int kbeg = (int)(s * p.kps);
    const int klen = (int)min(p.K - (uint32_t)kbeg, p.kps);
    DirectOperand<T, AK, MF> oa;
    DirectOperand<T, BKM, NF> ob;
    oa.init((const T*)p.A + (int64_t)b * p.sa, p.lda, m0, (int)p.M, kbeg, r, g);
    ob.init((const T*)p.B + (int64_t)b * p.sb, p.ldb, n0, (int)p.N, kbeg, r, g);

    floatx4 acc[MF][NF];
#pragma unroll
    for (int i = 0; i < MF; ++i)
#pragma unroll
        for (int j = 0; j < NF; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    uint32_t va[U][4 * MF], vb[U][4 * NF];
    auto compute = [&](const uint32_t (&xa)[4 * MF], const uint32_t (&xb)[4 * NF]) {
        u32x4 af[MF], bf[NF];
#pragma unroll
        for (int i = 0; i < MF; ++i) af[i] = oa.frag(xa, i);
#pragma unroll
        for (int j = 0; j < NF; ++j) bf[j] = ob.frag(xb, j);
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < MF; ++i)
#pragma unroll
                    for (int j = 0; j < NF; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(bf[j][e]),
                                                                         __uint_as_float(af[i][e]), acc[i][j], 0, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < MF; ++i)
#pragma unroll
                for (int j = 0; j < NF; ++j) acc[i][j] = mfma_16x16x32<T>(bf[j], af[i], acc[i][j]);
        }
    };

    // this wave's whole steps [s0, s0 + n); the partial last step is the last
    // wave's, which never has more whole steps than the others
    const int nfull = klen / KS;
    const int per_w = (nfull + 3) / 4;
    const int s0 = min(nfull, wave * per_w);
    const int n = min(nfull, s0 + per_w) - s0;
    auto load = [&](int u, int i) {
        oa.load(va[u], (s0 + i) * KS);
        ob.load(vb[u], (s0 + i) * KS);
    };
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (u < n) load(u, u);
    int i = 0;
    for (; i + 2 * U <= n; i += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            compute(va[u], vb[u]);
            load(u, i + u + U);
        }
    }
    // fewer than 2 U steps left, the first U of them loaded
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (i + u < n) compute(va[u], vb[u]);
        if (i + u + U < n) load(u, i + u + U);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (i + U + u < n) compute(va[u], vb[u]);
    if (wave == 3 && klen % KS) {
        oa.load_tail(va[0], nfull * KS, klen - nfull * KS, g);
        ob.load_tail(vb[0], nfull * KS, klen - nfull * KS, g);
        compute(va[0], vb[0]);
    }

    // ---- the four waves' sums, added in wave order ----
    // acc[i][j][e] is row (AK ? 16 i + r : MF r + i), column (BKM ? 16 j +
    // 4 g + e : NF (4 g + e) + j) of the tile
    float* mine = red[wave];
#pragma unroll
    for (int i = 0; i < MF; ++i) {
        float* row = mine + (AK ? 16 * i + r : MF * r + i) * LDR;
        if constexpr (BKM) {
#pragma unroll
            for (int j = 0; j < NF; ++j) *(floatx4*)(row + 16 * j + 4 * g) = acc[i][j];
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < NF; ++j) row[NF * (4 * g + e) + j] = acc[i][j][e];
        }
    }
    __syncthreads();

    float alpha, beta;
    load_scalars(p, alpha, beta);
    TC* Cb = (TC*)p.C + (int64_t)b * p.sc + (int64_t)s * p.s_split;
    const TC* Ci = (const TC*)p.epi.cin + (int64_t)b * p.epi.scin;
    typedef TC c4 __attribute__((ext_vector_type(4)));
    typedef c4 c4u __attribute__((aligned(2), may_alias));
    for (int q = tid; q < TM * TN / 4; q += 256) {
        const int ml = q / (TN / 4), nl = 4 * (q % (TN / 4));
        const int m = m0 + ml, n = n0 + nl;
        if (m < m_lo || m >= (int)p.M) continue;
        const float* src = &red[0][ml * LDR + nl];
        floatx4 x = *(const floatx4*)src;
#pragma unroll
        for (int w = 1; w < 4; ++w) {
            const floatx4 y = *(const floatx4*)(src + w * TM * LDR);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] += y[e];
        }
        TC* dst = Cb + (int64_t)m * p.ldc + n;
        const TC* cin = Ci + (int64_t)m * p.epi.ldcin + n;
        if (n >= n_lo && n + 4 <= (int)p.N) {
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = alpha * x[e];
            if (beta != 0.0f) {
                const c4 c = *(const c4u*)cin;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] += beta * (float)c[e];
            }
            add_bias4(p.epi, n, 4, o);
            c4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (TC)o[e];
            *(c4u*)dst = v;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (n + e < n_lo || n + e >= (int)p.N) continue;
                float o = alpha * x[e];
                if (beta != 0.0f) o += beta * (float)cin[e];
                if (p.epi.bias) o += bias_at(p.epi, n + e);
                dst[e] = (TC)o;
            }
        }
    }
}

}  // namespace vkb

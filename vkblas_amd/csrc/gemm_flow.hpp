// gemm_flow.hpp — 16-bit GEMM on 128 x 128 and 128 x 64 tiles with two or more
// workgroups per CU, any K in whole 16-byte chunks, any M and N and any
// alignment of C.
//
// For the aligned 16-bit calls that the pipelined kernel (gemm_pipe.hpp) does
// not take or serves badly: K not in pairs of 64 (an attention head's 64, 80 or
// 96), an N that is no multiple of 4 or a C without aligned rows (an output
// layer over an odd number of classes), N of one head (64). Their K loops are
// short or their tiles few, so they are bound by memory latency and by the
// stores of C, not by the matrix cores: instead of one workgroup per CU whose
// loads, MFMAs and stores are interleaved by hand, several per CU overlap each
// other's phases.
//
// Per workgroup: 4 waves (128 x 128: 2 x 2 of 64 x 64; 128 x 64: 4 x 1 of 32 x
// 64; or 8 waves, 4 x 2 of 32 x 64), v_mfma_f32_16x16x32, a K step of 64 (128 bytes). Operand tiles go to LDS
// by buffer -> LDS copies, NST - 1 steps ahead, one barrier per step:
//  * K-major (128-byte rows): row r at 8 r (16-byte units), chunk c at slot c ^
//    (r & 7), as the pipelined kernel's tiles; rows past the matrix repeat its
//    last row;
//  * MN-major (k rows of W = 128 or 64 columns, CPR = W / 8 chunks): k row k at
//    CPR k, chunk c at slot c ^ t(k), read with ds_read_b64_tr_b16 (W 128: t =
//    2 (k & 3) + 8 (((k >> 3) ^ (k >> 4)) & 1); W 64: t = 2 (k >> 1 & 1) + 4 (k >>
//    3 & 1); gemm_pipe.hpp and gemm_wavek.hpp say why these are free of bank
//    conflicts); chunks past the matrix repeat its last chunk (M or N a
//    multiple of 8).
//  * K past the end of the last step: the copies of those chunks or k rows go
//    out of the buffer's range, which the hardware answers with zeros.
// No tile moves and no load leaves the operands; C rows and columns past the
// matrix are not stored.
//
// Epilogue, every alignment: each wave passes 16 rows at a time through its own
// part of LDS in fp32 and stores 16 bytes of a row per lane (row segments of WN
// columns, element by element only where a group crosses N), reading beta's
// matrix the same way.
#pragma once
#include "gemm_pipe.hpp"

namespace vkb {

// BN: tile columns; NST: LDS stages; WAVES: 4, or 8 for 128 x 128 (4 x 2 waves of
// 32 x 64). Workgroups per CU (the register budget): what LDS holds, at one
// stage four (three with an MN-major operand, whose addresses need registers).
constexpr int flow_wg_per_cu(int BN, int NST, bool kmajor) {
    return NST == 1 ? (kmajor ? 4 : 3) : NST * (128 + BN) * 128 > 80 * 1024 ? 1 : 2;
}
// EARLY: beta's matrix is read before the K loop, which then hides its latency
// (bf16 -> fp32 TN 4096 x 1024 x 512, beta = 1: 14.5 -> 12.5 us); a form of its own,
// as its registers and the early scalars cost the others 3 % (attention bf16).
template <typename T, typename TC, bool AK, bool BKM, int BN, int NST, int WAVES, bool EARLY = false>
__global__ __launch_bounds__(64 * WAVES, flow_wg_per_cu(BN, NST, AK && BKM) * WAVES / 4)
void gemm_flow_kernel(KParams p) {
    static_assert(sizeof(T) == 2, "16-bit operands");
    static_assert(BN == 128 || BN == 64, "128 x 128 or 128 x 64 tiles");
    static_assert(NST >= 1 && NST <= 3, "LDS stages");
    static_assert(WAVES == 4 || (WAVES == 8 && BN == 128), "4 or 8 waves");
    constexpr int BM = 128, BK = 64;
    constexpr int WM = BN == 128 ? 256 / WAVES : 128 / WAVES, WN = 64;   // wave tile
    constexpr int NFM = WM / 16, NFN = WN / 16;
    constexpr int AU = BM * 8, BU = BN * 8;           // 16-byte units of a stage's A and B
    constexpr int STG = AU + BU;
    constexpr int NDA = BM / 8 / WAVES, NDB = BN / 8 / WAVES;   // copies per wave and step
    constexpr int ND = NDA + NDB;
    constexpr int EROW = WN + 4;                      // floats of a padded epilogue row
    constexpr int EU = WAVES * 16 * EROW / 4;             // units of the epilogue's rows
    constexpr int LU = NST * STG > EU ? NST * STG : EU;
    __shared__ u32x4 lds[LU];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = BN == 128 ? wave >> 1 : wave, wn = BN == 128 ? wave & 1 : 0;
    const int r16 = lane & 15, g = lane >> 4;

    // tile / batch / split decode, XCD-aware, groups of 8 tile rows, as gemm_kernel
    uint32_t bid = blockIdx.x;
    const uint32_t nwg = gridDim.x;
    if ((nwg & 7u) == 0) bid = (bid & 7u) * (nwg >> 3) + (bid >> 3);
    const uint32_t per = p.tiles_m * p.tiles_n;
    const uint32_t z = bid / per;
    const uint32_t t = bid - z * per;
    const uint32_t b = z / p.split;
    const uint32_t s = z - b * p.split;
    constexpr uint32_t GM = 8;
    const uint32_t width = GM * p.tiles_n;
    const uint32_t group = t / width;
    const uint32_t first_m = group * GM;
    const uint32_t gm = min(p.tiles_m - first_m, GM);
    const uint32_t tin = t - group * width;
    const int m0 = (int)(first_m + tin % gm) * BM;
    const int n0 = (int)(tin / gm) * BN;
    const int M = (int)p.M, N = (int)p.N;
    const int lda = (int)p.lda, ldb = (int)p.ldb;
    const int64_t kbeg = (int64_t)s * p.kps;
    const int klen = (int)min(p.K - (uint32_t)kbeg, p.kps);
    const int nkt = (klen + BK - 1) / BK;

    // Buffers on the tile's first element; 2 GiB of range (the launcher bounds
    // every offset below that), so an offset of OUT reads as zero.
    const T* At = (const T*)p.A + (int64_t)b * p.sa + (AK ? (int64_t)m0 * p.lda + kbeg : kbeg * p.lda);
    const T* Bt = (const T*)p.B + (int64_t)b * p.sb + (BKM ? (int64_t)n0 * p.ldb + kbeg : kbeg * p.ldb);
    auto rsrc_words = [](const void* base) {
        const uint64_t a = (uint64_t)base;
        return i32x4{__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                     __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32) & 0xffff), (int)0x80000000u, 0x00020000};
    };
    const i32x4 ra = rsrc_words(At), rb = rsrc_words(Bt);
    constexpr int OUT = (int)0x80000000u;

    // Copy i of this wave, per lane: K-major rows 8 (ND. wave + i) + lane / 8,
    // slot lane % 8, which holds chunk (lane % 8) ^ (lane / 8); MN-major k rows
    // RPB (ND. wave + i) + lane / CPR, slot lane % CPR.
    const int kc = (lane & 7) ^ (lane >> 3);          // K-major: this lane's chunk
    auto tsw = [](int w, int k) {
        return w == 128 ? 2 * (k & 3) + 8 * (((k >> 3) ^ (k >> 4)) & 1) : 2 * ((k >> 1) & 1) + 4 * ((k >> 3) & 1);
    };
    int va[NDA], vb[NDB];
#pragma unroll
    for (int i = 0; i < NDA; ++i) {
        if constexpr (AK) {
            va[i] = (min(8 * (NDA * wave + i) + (lane >> 3), M - 1 - m0) * lda + 8 * kc) * 2;
        } else {
            const int k = 4 * (NDA * wave + i) + (lane >> 4);   // W 128: 4 k rows per copy
            va[i] = (k * lda + min(m0 + 8 * ((lane & 15) ^ tsw(128, k)), M - 8)) * 2;
        }
    }
#pragma unroll
    for (int i = 0; i < NDB; ++i) {
        if constexpr (BKM) {
            vb[i] = (min(8 * (NDB * wave + i) + (lane >> 3), N - 1 - n0) * ldb + 8 * kc) * 2;
        } else {
            constexpr int CPR = BN / 8, RPB = 64 / CPR;
            const int k = RPB * (NDB * wave + i) + lane / CPR;
            vb[i] = (k * ldb + min(n0 + 8 * ((lane % CPR) ^ tsw(BN, k)), N - 8)) * 2;
        }
    }
    auto dma = [&](const i32x4& rs, int unit, int voff, int soff) {
        const int m0r = __builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)(lds_ptr_t)&lds[unit]);
        asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds"
                     :: "v"(voff), "s"(rs), "s"(__builtin_amdgcn_readfirstlane(soff)), "{m0}"(m0r)
                     : "memory");
    };
    // the copies of step kt into stage S
    auto copy_step = [&](int kt, int S) {
        const int left = klen - kt * BK;              // k of this step and after
        const int sa = (AK ? kt * BK : kt * BK * lda) * 2, sb = (BKM ? kt * BK : kt * BK * ldb) * 2;
        const int ua = S * STG + 64 * NDA * wave, ub = S * STG + AU + 64 * NDB * wave;
        if (left >= BK) {
#pragma unroll
            for (int i = 0; i < NDA; ++i) dma(ra, ua + 64 * i, va[i], sa);
#pragma unroll
            for (int i = 0; i < NDB; ++i) dma(rb, ub + 64 * i, vb[i], sb);
        } else {
            // k past the end: out of range, zero
#pragma unroll
            for (int i = 0; i < NDA; ++i) {
                const int k = AK ? 8 * kc : 4 * (NDA * wave + i) + (lane >> 4);
                dma(ra, ua + 64 * i, k < left ? va[i] : OUT, sa);
            }
#pragma unroll
            for (int i = 0; i < NDB; ++i) {
                const int k = BKM ? 8 * kc : (512 / BN) * (NDB * wave + i) + lane / (BN / 8);
                dma(rb, ub + 64 * i, k < left ? vb[i] : OUT, sb);
            }
        }
    };

    // Fragments of sub-step ss (32 k): K-major row r16 of fragment i, chunk 4 ss
    // + g; MN-major two transposing reads, 4 k rows apart.
    auto tr_read = [&](int byte_off) {
        const v4i16 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)((char*)lds + byte_off));
        return __builtin_bit_cast(u32x2, v);
    };
    int xk[2];
#pragma unroll
    for (int ss = 0; ss < 2; ++ss) xk[ss] = 8 * r16 + ((4 * ss + g) ^ (r16 & 7));
    // per-lane byte base of an MN-major fragment at column 16 f of the tile
    auto tr_base = [&](int w, int f) {
        const int k = 8 * g + (r16 >> 2);
        return (k * (w / 8) + ((2 * f + ((r16 >> 1) & 1)) ^ tsw(w, k))) * 16 + 8 * (r16 & 1);
    };
    int ta[AK ? 1 : NFM], tb[BKM ? 1 : NFN];
    if constexpr (!AK) {
#pragma unroll
        for (int i = 0; i < NFM; ++i) ta[i] = tr_base(BM, wm * NFM + i);
    }
    if constexpr (!BKM) {
#pragma unroll
        for (int j = 0; j < NFN; ++j) tb[j] = tr_base(BN, wn * NFN + j);
    }
    auto frag_a = [&](int S, int ss, int i) -> u32x4 {
        if constexpr (AK) {
            return lds[S * STG + (wm * WM + 16 * i) * 8 + xk[ss]];
        } else {
            const int o = S * STG * 16 + ta[i] + 32 * ss * (BM / 8) * 16;
            const u32x2 lo = tr_read(o), hi = tr_read(o + 4 * (BM / 8) * 16);
            return u32x4{lo[0], lo[1], hi[0], hi[1]};
        }
    };
    auto frag_b = [&](int S, int ss, int j) -> u32x4 {
        if constexpr (BKM) {
            return lds[S * STG + AU + (wn * WN + 16 * j) * 8 + xk[ss]];
        } else {
            const int o = (S * STG + AU) * 16 + tb[j] + 32 * ss * (BN / 8) * 16;
            const u32x2 lo = tr_read(o), hi = tr_read(o + 4 * (BN / 8) * 16);
            return u32x4{lo[0], lo[1], hi[0], hi[1]};
        }
    };

    // the epilogue's share of C: row segments of WN columns, CV of them per lane
    constexpr int CV = 16 / (int)sizeof(TC);
    constexpr int LPR = WN / CV;                      // lanes per row
    constexpr int IT = 16 * LPR / 64;                 // rounds per 16 rows
    typedef TC cvec __attribute__((ext_vector_type(CV)));
    typedef cvec cvec_any __attribute__((aligned(2), may_alias));
    float alpha, beta;
    cvec old[EARLY ? NFM : 1][EARLY ? IT : 1];
    if constexpr (EARLY) {
        load_scalars(p, alpha, beta);
        const int n = n0 + wn * WN + lane % LPR * CV;
        const TC* Ci = (const TC*)p.epi.cin + (int64_t)b * p.epi.scin;
#pragma unroll
        for (int i = 0; i < NFM; ++i)
#pragma unroll
            for (int it = 0; it < IT; ++it) {
                const int m = m0 + wm * WM + 16 * i + it * (64 / LPR) + lane / LPR;
                if (m < M && n + CV <= N) old[i][it] = *(const cvec_any*)(Ci + (int64_t)m * p.epi.ldcin + n);
            }
    }

    floatx4 acc[NFM][NFN];
#pragma unroll
    for (int i = 0; i < NFM; ++i)
#pragma unroll
        for (int j = 0; j < NFN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](int S) {
#pragma unroll
        for (int ss = 0; ss < 2; ++ss) {
            u32x4 af[NFM], bf[NFN];
#pragma unroll
            for (int j = 0; j < NFN; ++j) bf[j] = frag_b(S, ss, j);
#pragma unroll
            for (int i = 0; i < NFM; ++i) af[i] = frag_a(S, ss, i);
#pragma unroll
            for (int i = 0; i < NFM; ++i)
#pragma unroll
                for (int j = 0; j < NFN; ++j) acc[i][j] = mfma_16x16x32<T>(bf[j], af[i], acc[i][j]);
        }
    };
    // this wave's copies but for the last c (0 or 1) steps' have landed and its LDS
    // reads have returned; then every wave's
    auto sync = [&](int c) {
        if (c <= 0) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(ND) : "memory");
    };
    if constexpr (NST == 1) {
        for (int kt = 0; kt < nkt; ++kt) {
            if (kt) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the stage is free
            copy_step(kt, 0);
            sync(0);
            compute(0);
        }
    } else {
#pragma unroll
        for (int i = 0; i < NST - 1; ++i)
            if (i < nkt) copy_step(i, i);
        int S = 0;
        for (int kt = 0; kt < nkt; ++kt) {
            sync(min(NST - 2, nkt - 1 - kt));
            // the stage that step kt - 1 used: every wave is past its reads
            if (kt + NST - 1 < nkt) copy_step(kt + NST - 1, S == 0 ? NST - 1 : S - 1);
            compute(S);
            S = S + 1 == NST ? 0 : S + 1;
        }
    }

    // ---- epilogue ----
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the stages are free
    if constexpr (!EARLY) load_scalars(p, alpha, beta);
    float* rows = (float*)lds + wave * 16 * EROW;
    TC* Cb = (TC*)p.C + (int64_t)b * p.sc + (int64_t)s * p.s_split;
    const TC* Ci = (const TC*)p.epi.cin + (int64_t)b * p.epi.scin;
    const int c = lane % LPR * CV;                    // this lane's first column of the wave's
    const int n = n0 + wn * WN + c;
    float bias[CV];
#pragma unroll
    for (int e = 0; e < CV; ++e)     // -0.0 where there is none: adding it changes no result's sign
        bias[e] = p.epi.bias && n + e < N ? bias_at(p.epi, n + e) : -0.0f;
#pragma unroll
    for (int i = 0; i < NFM; ++i) {
#pragma unroll
        for (int j = 0; j < NFN; ++j) *(floatx4*)(rows + r16 * EROW + 16 * j + 4 * g) = acc[i][j];
        // a wave's LDS operations complete in order; the wait keeps the
        // compiler from reordering the cross-lane read-back
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int r = it * (64 / LPR) + lane / LPR;
            const int m = m0 + wm * WM + 16 * i + r;
            float x[CV];
#pragma unroll
            for (int q = 0; q < CV / 4; ++q) {
                const floatx4 v = *(const floatx4*)(rows + r * EROW + c + 4 * q);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * q + e] = alpha * v[e];
            }
            if (m < M && n < N) {
                TC* dst = Cb + (int64_t)m * p.ldc + n;
                const TC* cin = Ci + (int64_t)m * p.epi.ldcin + n;
                if (n + CV <= N) {
                    if (beta != 0.0f) {
                        cvec o;
                        if constexpr (EARLY) o = old[i][it];
                        else o = *(const cvec_any*)cin;
#pragma unroll
                        for (int e = 0; e < CV; ++e) x[e] += beta * (float)o[e];
                    }
                    cvec v;
#pragma unroll
                    for (int e = 0; e < CV; ++e) v[e] = (TC)(x[e] + bias[e]);
                    __builtin_nontemporal_store(v, (cvec_any*)dst);
                } else {
#pragma unroll
                    for (int e = 0; e < CV; ++e) {
                        if (n + e >= N) continue;
                        float y = x[e];
                        if (beta != 0.0f) y += beta * (float)cin[e];
                        dst[e] = (TC)(y + bias[e]);
                    }
                }
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
}

}  // namespace vkb

// gemm_launch.hpp — host-side launcher for gemm_kernel<> (one instantiation
// set per element-type pair; gemm_f32.hip / gemm_f16.hip include this).
#pragma once
#include "gemm_mfma.hpp"
#include "gemm_pipe.hpp"
#include "gemm_wavek.hpp"
#include "gemm_direct.hpp"
#include "gemm_flow.hpp"
#include "vkb_launch.h"

namespace vkb {

template <int TILE> struct TileDim;
template <> struct TileDim<VKB_TILE_64>  { static constexpr int BM = 64,  BN = 64;  };
template <> struct TileDim<VKB_TILE_128> { static constexpr int BM = 128, BN = 128; };
template <> struct TileDim<VKB_TILE_256> { static constexpr int BM = 256, BN = 256; };

template <typename T, typename TC, bool AK, bool BKM, int TILE, bool CHECKED>
static int launch_one(const KParams& p, uint32_t grid, hipStream_t st) {
    constexpr int BM = TileDim<TILE>::BM, BN = TileDim<TILE>::BN;
    hipLaunchKernelGGL((gemm_kernel<T, TC, AK, BKM, BM, BN, CHECKED>), dim3(grid), dim3(256), 0, st, p);
    return (int)hipGetLastError();
}

template <typename T, typename TC, bool AK, bool BKM, int TILE>
static int launch_ck(const KParams& p, bool checked, uint32_t grid, hipStream_t st) {
    return checked ? launch_one<T, TC, AK, BKM, TILE, true>(p, grid, st)
                   : launch_one<T, TC, AK, BKM, TILE, false>(p, grid, st);
}

template <typename T, typename TC, int TILE>
static int launch_layout(const KParams& p, bool ak, bool bk, bool checked, uint32_t grid, hipStream_t st) {
    if (ak) {
        return bk ? launch_ck<T, TC, true, true, TILE>(p, checked, grid, st)
                  : launch_ck<T, TC, true, false, TILE>(p, checked, grid, st);
    }
    return bk ? launch_ck<T, TC, false, true, TILE>(p, checked, grid, st)
              : launch_ck<T, TC, false, false, TILE>(p, checked, grid, st);
}

static inline bool aligned(const void* ptr, uintptr_t a) { return ((uintptr_t)ptr % a) == 0; }

// Whether a launch can hold that many workgroups: HIP counts its threads in 32
// bits, and past them runs a few workgroups and reports success.
static inline bool launches(uint64_t workgroups, uint32_t threads) { return workgroups <= 0xffffffffull / threads; }

// Compute units of the current device (cached per device; 0 if unknown).
static inline uint32_t cu_count() {
    static int cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    int n = __atomic_load_n(&cached[dev], __ATOMIC_RELAXED);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 0) n = 0;
        __atomic_store_n(&cached[dev], n, __ATOMIC_RELAXED);
    }
    return (uint32_t)n;
}

// Tiles as a share of the chip of cu compute units: their number per 256, on
// which the lines below that compare it were measured.
static inline uint64_t per_256(uint64_t tiles, uint32_t cu) {
    return cu ? (tiles * 256 + cu - 1) / cu : tiles;
}

// Bytes of K per step of the wave-K kernel for 16-bit inputs: 128 (whole
// 128-byte rows of a K-major operand per copy).  Measured against 64 (more
// stages of half rows), M = N = 256, fp16, hipBLAS NN, split 4 / 16: K =
// 65536 45.4 / 24.1 -> 36.7 / 19.8 us, K = 262144 163.5 / 83.1 -> 133.5 /
// 66.5 us (two alternating runs, one box).
#ifndef VKB_WAVEK_KB16
#define VKB_WAVEK_KB16 128
#endif
constexpr int WK_KB16 = VKB_WAVEK_KB16;

template <typename T, typename TC, int MF, int NF, int U>
static int launch_direct_one(const KParams& p, bool ak, bool bk, uint32_t grid, hipStream_t st) {
    if (ak) {
        if (bk) hipLaunchKernelGGL((gemm_direct_kernel<T, TC, true, true, MF, NF, U>), dim3(grid), dim3(256), 0, st, p);
        else hipLaunchKernelGGL((gemm_direct_kernel<T, TC, true, false, MF, NF, U>), dim3(grid), dim3(256), 0, st, p);
    } else {
        if (bk) hipLaunchKernelGGL((gemm_direct_kernel<T, TC, false, true, MF, NF, U>), dim3(grid), dim3(256), 0, st, p);
        else hipLaunchKernelGGL((gemm_direct_kernel<T, TC, false, false, MF, NF, U>), dim3(grid), dim3(256), 0, st, p);
    }
    return (int)hipGetLastError();
}

template <typename T, typename TC, int BN, int NST, int WAVES, bool EARLY = false>
static int launch_flow_one(const KParams& p, bool ak, bool bk, uint32_t grid, hipStream_t st) {
    const dim3 wg(64 * WAVES);
    if (ak) {
        if (bk) hipLaunchKernelGGL((gemm_flow_kernel<T, TC, true, true, BN, NST, WAVES, EARLY>), dim3(grid), wg, 0, st, p);
        else hipLaunchKernelGGL((gemm_flow_kernel<T, TC, true, false, BN, NST, WAVES, EARLY>), dim3(grid), wg, 0, st, p);
    } else {
        if (bk) hipLaunchKernelGGL((gemm_flow_kernel<T, TC, false, true, BN, NST, WAVES, EARLY>), dim3(grid), wg, 0, st, p);
        else hipLaunchKernelGGL((gemm_flow_kernel<T, TC, false, false, BN, NST, WAVES, EARLY>), dim3(grid), wg, 0, st, p);
    }
    return (int)hipGetLastError();
}

// Whether gemm_flow_kernel takes a call: 16-byte aligned 16-bit operands and
// leading dimensions (vec_a, vec_b), K in whole 16-byte chunks where an operand
// is K-major, the row dimension of an MN-major one a multiple of 8, every
// offset below 2 GiB.
template <typename T>
static bool flow_ok(const vkb_gemm_args* a, const KParams& p) {
    if (sizeof(T) != 2 || p.ptr_array || !p.vec_a || !p.vec_b) return false;
    const uint64_t span_a = ((uint64_t)(a->a_kmajor ? 128 : a->K + 64) * (uint64_t)a->lda + (a->a_kmajor ? a->K + 64 : a->M)) * 2;
    const uint64_t span_b = ((uint64_t)(a->b_kmajor ? 128 : a->K + 64) * (uint64_t)a->ldb + (a->b_kmajor ? a->K + 64 : a->N)) * 2;
    return (a->a_kmajor ? a->K % 8 == 0 : a->M % 8 == 0) && (a->b_kmajor ? a->K % 8 == 0 : a->N % 8 == 0) &&
           span_a < (1ull << 31) && span_b < (1ull << 31);
}

// gemm_flow_kernel's form, from the number of 128 x 128 tiles t per 256 CUs (one box,
// fp16 us):
//  * N of one 64-column tile, or t at most half the CUs: 128 x 64 tiles, three
//    stages, two workgroups per CU (1000^3, t = 64, 11.2 against 13.8 on 128 x 128;
//    1280 x 1280 x 1000, 100, 11.2 / 13.7; 1536 x 1536 x 1000, 144, 15.9 / 13.5);
//  * up to one per CU: 128 x 128, three stages, eight waves (96 KB, one workgroup
//    per CU: two waves per SIMD; 2001 x 2000 x 2000 23.6 against 30.3 with two
//    stages and two workgroups of four waves per CU, 25.9 with four waves);
//  * more: 128 x 128, two stages, two workgroups per CU (4000^3 145 against 166);
//    K of a single step: one stage and three or four workgroups per CU (64 x 1024 x
//    1024 x 64 29.7 against 34.7 with two stages).
template <typename T, typename TC>
static int launch_flow(const vkb_gemm_args* a, KParams p, bool ak, bool bk, uint32_t cu, hipStream_t st) {
    if constexpr (sizeof(T) == 2) {
        const uint64_t mats = (uint64_t)p.batch * p.split;
        p.tiles_m = (a->M + 127) / 128;
        p.tiles_n = (a->N + 127) / 128;
        const uint64_t t = per_256((uint64_t)p.tiles_m * p.tiles_n * mats, cu);
        const bool narrow = a->N <= 64 || t <= 128;
        if (narrow) p.tiles_n = (a->N + 63) / 64;
        const uint64_t grid = (uint64_t)p.tiles_m * p.tiles_n * mats;
        if (grid == 0 || !launches(grid, t <= 256 && !narrow ? 512 : 256)) return (int)hipErrorInvalidValue;
        const bool early = a->scalar_mode == VKB_SCALAR_HOST && a->beta != 0.0f;   // beta's matrix before the K loop
        if (narrow && early) return launch_flow_one<T, TC, 64, 3, 4, true>(p, ak, bk, (uint32_t)grid, st);
        if (narrow) return launch_flow_one<T, TC, 64, 3, 4>(p, ak, bk, (uint32_t)grid, st);
        if (t <= 256 && early) return launch_flow_one<T, TC, 128, 3, 8, true>(p, ak, bk, (uint32_t)grid, st);
        if (t <= 256) return launch_flow_one<T, TC, 128, 3, 8>(p, ak, bk, (uint32_t)grid, st);
        if ((p.split > 1 ? p.kps : a->K) <= 64) return launch_flow_one<T, TC, 128, 1, 4>(p, ak, bk, (uint32_t)grid, st);
        return launch_flow_one<T, TC, 128, 2, 4>(p, ak, bk, (uint32_t)grid, st);
    }
    return (int)hipErrorInvalidValue;
}

// gemm_direct_kernel's tile for a call: 64 x 64 where that gives at least 144
// workgroups, else 32 x 32, and 16 x 32 for fp32 where 32 x 32 gives fewer
// than 128.  The line is where the larger tile's extra reuse makes up for the
// CUs it leaves idle (one box, us, 64 / 32 / 16 x 32):
//   fp32 NT 512 x 1024 x 1024 (128 tiles of 64) 30.9 / 23.2 / 27.0, 768^3 (144)
//   24.5 / 25.9 / 26.0, 1024^3 31.3 / 42.0 / 49.6; fp32 NN 256^2 x 1024 (64
//   tiles of 32) 25.1 / 12.0 / 8.2, 384^2 x 2048 (144) TN 37.8 / 16.9 / 20.0;
//   fp16 NT 512^2 x 1024 11.9 / 8.4, 512 x 1024 x 1024 11.9 / 10.7, 768^3 10.4 / 12.1.
// Returns 0 if no tile fits the operands (an MN-major operand needs a whole
// tile in its dimension; a tile's rows must span less than 2^31 bytes) or the
// launch: the larger tiles of the generic kernel then may.
template <typename T>
static uint32_t direct_tile(const vkb_gemm_args* a, uint64_t mats, uint32_t cu) {
    auto tiles = [&](uint32_t tm, uint32_t tn) {
        return (uint64_t)((a->M + tm - 1) / tm) * ((a->N + tn - 1) / tn) * mats;
    };
    auto fits = [&](uint32_t tm, uint32_t tn) {
        // per-lane offsets: the rows of a K-major tile, 32 k rows (or fewer)
        // of an MN-major one
        const uint64_t ra = a->a_kmajor ? tm : 32, rb = a->b_kmajor ? tn : 32;
        return (a->a_kmajor || a->M >= tm) && (a->b_kmajor || a->N >= tn) &&
               launches(tiles(tm, tn), 256) &&
               (ra * (uint64_t)a->lda + 64) * sizeof(T) < (1ull << 31) &&
               (rb * (uint64_t)a->ldb + 64) * sizeof(T) < (1ull << 31);
    };
    if (per_256(tiles(64, 64), cu) >= 144 && fits(64, 64)) return 64;
    if ((sizeof(T) == 2 || per_256(tiles(32, 32), cu) >= 128) && fits(32, 32)) return 32;
    if (sizeof(T) == 4 && fits(16, 32)) return 16;
    return 0;
}

// The generic kernel's 128 x 128 tiles, each operand read once, against many
// small tiles whose operands come from the caches over and over: the line by
// layout, since an operand read along K costs gemm_direct_kernel more loads and
// one read across it costs the generic kernel a transpose (unaligned, us,
// generic / direct, in brackets the tiles of 64 x 64):
//   fp32 NT 999^3 (256) 81 / 32, 1500^2 x 1003 (576) 82 / 83, 2001 x 2003 x 2005
//   (1024) 156 / 214; NN 228 / 197, TN 276 / 161 there, 321 / 282 and 358 / 237 at
//   4001 x 3001 x 1003 (2961): direct throughout;
//   fp16 NT 333 x 1001 x 2003 (96) 27 / 42, 999^3 25 / 22, 777 x 3001 x 1003 (611)
//   26 / 58, 2001^3 46 / 169; NN 333 x 1001 x 2003 46 / 27, 100 x 10007 x 777 (314)
//   30 / 27, 1500^2 35 / 44, 2001^3 62 / 117; TN 2001^3 81 / 71, 4001 x 3001 x
//   1003 88 / 135.
template <typename T>
static bool direct_loses(bool ak, bool bk, uint64_t t64, uint32_t klen) {
    if (sizeof(T) == 4) return ak && bk && t64 >= 560;
    if (ak && bk) return t64 > 256 || (t64 >= 96 && klen >= 1536);
    return t64 >= (ak || bk ? 400 : 1536);
}

template <typename T, typename TC>
static int launch_direct(const vkb_gemm_args* a, KParams p, uint32_t tile, bool ak, bool bk, hipStream_t st) {
    const uint32_t tm = tile, tn = tile == 16 ? 32 : tile;
    p.tiles_m = (a->M + tm - 1) / tm;
    p.tiles_n = (a->N + tn - 1) / tn;
    const uint64_t grid = (uint64_t)p.tiles_m * p.tiles_n * p.batch * p.split;
    if (grid == 0 || !launches(grid, 256)) return (int)hipErrorInvalidValue;
    if (tile == 64) return launch_direct_one<T, TC, 4, 4, 4>(p, ak, bk, (uint32_t)grid, st);
    if (tile == 32) return launch_direct_one<T, TC, 2, 2, 8>(p, ak, bk, (uint32_t)grid, st);
    if constexpr (sizeof(T) == 4) return launch_direct_one<T, TC, 1, 2, 8>(p, ak, bk, (uint32_t)grid, st);
    return (int)hipErrorInvalidValue;
}

template <typename T, typename TC>
static int launch_gemm_typed(const vkb_gemm_args* a, int tile, hipStream_t st) {
    constexpr int VEC = Elem<T>::VEC;
    constexpr int BK = Elem<T>::BK;
    static_assert(WAVEK_NQ == VKB_WAVEK_NQ, "one part count");
    int bm = 64, bn = 64;
    if (tile == VKB_TILE_128) { bm = bn = 128; }
    else if (tile == VKB_TILE_256) { bm = bn = 256; }
    else if (tile == VKB_TILE_32) { bm = bn = 32; }
    else if (tile != VKB_TILE_64 && tile != VKB_TILE_64Q) return (int)hipErrorInvalidValue;

    KParams p{};
    p.A = a->A; p.B = a->B; p.C = a->C;
    p.lda = a->lda; p.ldb = a->ldb; p.ldc = a->ldc;
    p.sa = a->stride_a; p.sb = a->stride_b; p.sc = a->stride_c;
    p.M = a->M; p.N = a->N; p.K = a->K;
    p.batch = a->batch ? a->batch : 1;
    p.split = a->split > 1 ? a->split : 1;
    p.kps = p.split > 1 ? a->k_per_split : a->K;
    p.s_split = p.split > 1 ? a->stride_split : 0;
    p.tiles_m = (a->M + bm - 1) / bm;
    p.tiles_n = (a->N + bn - 1) / bn;
    p.alpha = a->alpha; p.beta = a->beta;
    p.scalar_mode = a->scalar_mode;
    p.alpha_dev = a->alpha_dev; p.beta_dev = a->beta_dev;
    const vkb_epilogue_args* ep = a->epi;
    const bool sep_cin = ep && ep->c_in && p.split == 1;   // pass 1 writes raw partials
    p.epi.cin = sep_cin ? ep->c_in : a->C;
    p.epi.ldcin = sep_cin ? ep->ldc_in : a->ldc;
    p.epi.scin = sep_cin ? ep->stride_c_in : a->stride_c;
    p.epi.bias = (ep && p.split == 1) ? ep->bias : nullptr;
    p.epi.bias_type = ep ? ep->bias_type : 0;
    p.ptr_array = a->ptr_array != 0;
    if (p.ptr_array && sep_cin) return (int)hipErrorInvalidValue;   // Cin pointers are not given
    // each K slice over VKB_WAVEK_NQ workgroups: the wave-K kernel only (below)
    p.nq = tile == VKB_TILE_64Q ? VKB_WAVEK_NQ : 1;
    p.qpart = a->qpart;
    p.qcnt = a->qcnt;
    if (tile == VKB_TILE_64Q &&
        (p.split < 2 || p.ptr_array || !a->qpart || !a->qcnt || ((uintptr_t)a->qpart & 15) ||
         ((uintptr_t)a->qcnt & 3) || (uint64_t)p.split * p.tiles_m * p.tiles_n > VKB_WS_COUNTERS))
        return (int)hipErrorInvalidValue;
    const bool multi = p.batch > 1;
    if (p.ptr_array) {
        // the matrices' alignment is not known here: always the checked
        // instantiation, which takes any
        if (p.split > 1) return (int)hipErrorInvalidValue;
    } else {
        p.vec_a = (a->lda % VEC == 0) && aligned(a->A, 16) && (!multi || a->stride_a % VEC == 0);
        p.vec_b = (a->ldb % VEC == 0) && aligned(a->B, 16) && (!multi || a->stride_b % VEC == 0);
        p.vec_c = (a->ldc % 4 == 0) && aligned(a->C, 4 * sizeof(TC)) && (!multi || a->stride_c % 4 == 0) &&
                  (p.split == 1 || p.s_split % 4 == 0);
        if (sep_cin)   // Cin is read with the same vector width as C
            p.vec_c = p.vec_c && p.epi.ldcin % 4 == 0 && aligned(p.epi.cin, 4 * sizeof(TC)) &&
                      (!multi || p.epi.scin % 4 == 0);
    }
    {
        constexpr int64_t CV = 16 / sizeof(TC);   // elements per 16 bytes of C
        // an edge tile (N not a multiple of the tile) stores from a shifted
        // column N - BN on: whole 16-byte chunks need N % CV == 0 as well
        p.c_rows16 = !p.ptr_array && a->ldc % CV == 0 && aligned(a->C, 16) && (!multi || a->stride_c % CV == 0) &&
                     (p.split == 1 || p.s_split % CV == 0) && (a->N % bn == 0 || a->N % CV == 0);
        // the operands and C together near the 256 MiB of the Infinity Cache or
        // below: past 320 MiB storing C past the caches is level or ahead for
        // the same C on each call too (8192 x 8192 x 2048, 320 MiB, 315 / 320 us)
        p.c_stays = p.batch * (((uint64_t)a->M + a->N) * a->K * sizeof(T) + (uint64_t)a->M * a->N * sizeof(TC)) <=
                    (320ull << 20);
        p.cin_rows16 = !p.ptr_array && p.epi.ldcin % CV == 0 && aligned(p.epi.cin, 16) &&
                       (!multi || p.epi.scin % CV == 0);
    }
    auto report = [&](int k) {
        if (a->kernel_out) *a->kernel_out = k;
    };
    if (p.split > 1 && (p.kps == 0 || p.kps % BK != 0)) return (int)hipErrorInvalidValue;

    const bool full = !p.ptr_array && (a->M % bm == 0) && (a->N % bn == 0) && (a->K % BK == 0) &&
                      p.vec_a && p.vec_b && p.vec_c;
    const uint64_t grid64 = (uint64_t)p.tiles_m * p.tiles_n * p.batch * p.split * p.nq;
    if (grid64 == 0 || !launches(grid64, 256)) return (int)hipErrorInvalidValue;
    const uint32_t grid = (uint32_t)grid64;
    const bool ak = a->a_kmajor != 0, bk = a->b_kmajor != 0;
    {
        // software-pipelined kernel for full 256x256 and 128x128 tiles (also
        // split-K pass 1 on them).  K and the split-K slice a multiple of two
        // K steps (128 bytes each): the loop runs pairs.  Buffer offsets are
        // signed 32-bit: bound the byte span of each operand tile.
        // Edge tiles (M or N not a multiple of the tile) shift back inside
        // the matrix: M >= bm, N >= bn; the shifted start of an MN-major
        // operand stays 16-byte aligned (M or N a multiple of VEC); the
        // epilogue masks groups of four columns (N % 4 == 0).
        constexpr uint64_t ES = sizeof(T);
        constexpr uint32_t KPAIR = 256 / sizeof(T);
        const uint64_t span_a = ((uint64_t)(a->a_kmajor ? bm : a->K) * (uint64_t)a->lda + a->K) * ES;
        const uint64_t span_b = ((uint64_t)(a->b_kmajor ? bn : a->K) * (uint64_t)a->ldb + a->K) * ES;
        // M < bm: 128x128 tiles with K-major A (rows past M read as row M - 1)
        const bool edges_ok = (a->M >= (uint32_t)bm || (bm == 128 && ak)) && a->N >= (uint32_t)bn && a->N % 4 == 0 &&
                              (a->a_kmajor || a->M % VEC == 0) && (a->b_kmajor || a->N % VEC == 0);
        const bool tiles_ok = !p.ptr_array && (a->K % BK == 0) && p.vec_a && p.vec_b && p.vec_c &&
                              (full || edges_ok);
        const bool pipe_ok = tiles_ok && (p.split == 1 || p.kps % KPAIR == 0) && !a->generic_only &&
                             a->K % KPAIR == 0 && span_a < (1ull << 31) && span_b < (1ull << 31);
        // Where the planner leaves the choice open (a->direct) and the wave-K
        // kernel does not take the call (split-K pass 1 on whole 64x64 tiles):
        //  * aligned 16-bit operands that the pipelined kernel does not take:
        //    gemm_flow_kernel from 144 tiles of 64x64 on (fp16 NT 2000 x 2001 x 1000
        //    26 -> 19 us, TN 2000^3 136 -> 24, 64 x 512 x 512 x 80 35 -> 12, 64 x 1024 x
        //    1024 x 64 58 -> 30 against the generic kernel; 768 x 768 x 1000, 144
        //    tiles, 11.9 -> 10.9 against the direct one, 640 x 640, 100, 10.4 / 10.9);
        //    and instead of the pipelined 128x128 kernel on one wave of tiles
        //    where beta adds to C after at most 1024 k, as it reads C before the K
        //    loop and not after it (us, pipelined / this: bf16 -> fp32 TN 4096 x 1024 x
        //    512 13.5 / 12.5, 1024 x 1024 x 512 10.0 / 7.7, x 1024 13.1 / 10.8, 4096 x
        //    1024 x 1024 level, fp16 NT 2000 x 1000 x 1024 11.9 / 10.8; at K = 2048
        //    the pipelined kernel is ahead, 24.9 / 26.2 before its own row reads);
        //  * gemm_direct_kernel (small tiles, fragments straight from memory)
        //    - instead of the pipelined 128x128 kernel for fp32 on at most 128
        //      of its tiles, half the CUs (fp32 us, NT / NN / TN: 512 x 1024^2,
        //      32 tiles, 60 -> 23 / 20 / 18; 1024^3, 64, 60 -> 31 / 27 / 24;
        //      512 x 4096 x 1024, 128, 61 -> 57 / 49 / 45; 1536^3, 144 tiles,
        //      89 against 122 / 102 / 85).  16-bit inputs stay there: level at
        //      32 tiles, ahead from 36 on (768 x 1024 x 3072 fp16 22 against 26);
        //    - instead of the generic kernel with edge handling, but not where
        //      direct_loses (many tiles) or past 256 tiles with a short K, where
        //      the four waves have too little to share (of random calls with K below
        //      512 bytes 4 of 283 lost up to 128 tiles, 6 of 57 up to 256, 25 of 49
        //      up to 512; fp16 TT 64 of 343 x 13 x 5, 384 tiles, 6.5 -> 7.7);
        //    - instead of the generic kernel on whole tiles where 64 x 64 ones
        //      would leave CUs idle (fp32 NT 512^2 x 2048 49 -> 25): with both
        //      operands along K, where the generic kernel has nothing to
        //      transpose, below 144 tiles in fp32 (128 tiles 8.4 -> 6.8, 144 73 ->
        //      83) and 96 in 16 bits (64 tiles 3.5 -> 3.0, 96 13.7 -> 16.8), else
        //      below 192 (fp16 TN 176, K = 1216, 22 -> 10), 144 for a short K
        //      (fp32 TN 160, K = 64, 5.1 -> 5.5).
        if (a->direct && !p.ptr_array && !a->generic_only &&
            (tile == VKB_TILE_64 || tile == VKB_TILE_128 || tile == VKB_TILE_256) &&
            !(tile == VKB_TILE_64 && p.split > 1 && full)) {
            const uint32_t cu = cu_count();
            const uint64_t mats = (uint64_t)p.batch * p.split;
            const uint64_t t64 = per_256((uint64_t)((a->M + 63) / 64) * ((a->N + 63) / 64) * mats, cu);
            const bool pipe = pipe_ok && tile != VKB_TILE_64;
            const bool add = pipe && tile == VKB_TILE_128 && p.split == 1 && per_256(grid, cu) <= 256 &&
                             a->scalar_mode == VKB_SCALAR_HOST && a->beta != 0.0f && a->K <= 1024;
            if (a->direct == 1 && ((!pipe && t64 >= 144) || add) && flow_ok<T>(a, p)) {
                report(VKB_KERN_FLOW);
                return launch_flow<T, TC>(a, p, ak, bk, cu, st);
            }
            const uint32_t klen = p.split > 1 ? p.kps : a->K;
            const bool want = a->direct == 2 ? true
                            : pipe ? sizeof(T) == 4 && tile == VKB_TILE_128 && p.split == 1 &&
                                   per_256(grid, cu) <= 128
                            : full ? t64 < (ak && bk ? (sizeof(T) == 4 ? 144u : 96u) : klen * sizeof(T) >= 512 ? 192u : 144u)
                                   : !direct_loses<T>(ak, bk, t64, klen) &&
                                         ((uint64_t)klen * sizeof(T) >= 512 || t64 <= 256);
            const uint32_t dt = want ? direct_tile<T>(a, mats, cu) : 0;
            if (dt) {
                report(VKB_KERN_DIRECT);
                return launch_direct<T, TC>(a, p, dt, ak, bk, st);
            }
        }
        if (tile == VKB_TILE_256 && pipe_ok) {
            report(VKB_KERN_PIPE256);
            if (ak) {
                if (bk) hipLaunchKernelGGL((gemm_pipe_kernel<T, TC, true, true>), dim3(grid), dim3(256), 0, st, p);
                else hipLaunchKernelGGL((gemm_pipe_kernel<T, TC, true, false>), dim3(grid), dim3(256), 0, st, p);
            } else {
                if (bk) hipLaunchKernelGGL((gemm_pipe_kernel<T, TC, false, true>), dim3(grid), dim3(256), 0, st, p);
                else hipLaunchKernelGGL((gemm_pipe_kernel<T, TC, false, false>), dim3(grid), dim3(256), 0, st, p);
            }
            return (int)hipGetLastError();
        }
        // 128x128 tiles: the pipelined kernel with 64x64 wave tiles.  16-bit
        // types take four LDS stages when the grid is at most one workgroup
        // per CU (the 144 KB they take allow no second one), else two; fp32
        // (a K step is 4096 MFMA cycles, longer than the load latency) always
        // two.
        if (tile == VKB_TILE_128 && pipe_ok) {
            const bool four = sizeof(T) == 2 && grid <= cu_count();
            report(four ? VKB_KERN_PIPE128_4 : VKB_KERN_PIPE128);
            if constexpr (sizeof(T) == 2) {
                if (four) {
                    if (ak) {
                        if (bk) hipLaunchKernelGGL((gemm_pipe_kernel<T, TC, true, true, 64, 4>), dim3(grid), dim3(256), 0, st, p);
                        else hipLaunchKernelGGL((gemm_pipe_kernel<T, TC, true, false, 64, 4>), dim3(grid), dim3(256), 0, st, p);
                    } else {
                        if (bk) hipLaunchKernelGGL((gemm_pipe_kernel<T, TC, false, true, 64, 4>), dim3(grid), dim3(256), 0, st, p);
                        else hipLaunchKernelGGL((gemm_pipe_kernel<T, TC, false, false, 64, 4>), dim3(grid), dim3(256), 0, st, p);
                    }
                    return (int)hipGetLastError();
                }
            }
            if (ak) {
                if (bk) hipLaunchKernelGGL((gemm_pipe_kernel<T, TC, true, true, 64>), dim3(grid), dim3(256), 0, st, p);
                else hipLaunchKernelGGL((gemm_pipe_kernel<T, TC, true, false, 64>), dim3(grid), dim3(256), 0, st, p);
            } else {
                if (bk) hipLaunchKernelGGL((gemm_pipe_kernel<T, TC, false, true, 64>), dim3(grid), dim3(256), 0, st, p);
                else hipLaunchKernelGGL((gemm_pipe_kernel<T, TC, false, false, 64>), dim3(grid), dim3(256), 0, st, p);
            }
            return (int)hipGetLastError();
        }
    }
    // Split-K pass 1 on 32x32 or 64x64 tiles (few output tiles, a caller's
    // split): the wave-K kernel, whose four waves each take a quarter of the
    // slice's K.  Whole tiles, K and the slice in whole K steps, aligned
    // operands; buffer offsets are signed 32-bit.
    if constexpr (std::is_same<TC, float>::value) {
        if ((tile == VKB_TILE_32 || tile == VKB_TILE_64 || tile == VKB_TILE_64Q) && p.split > 1 && !p.ptr_array &&
            !a->generic_only) {
            constexpr uint64_t ES = sizeof(T);
            const uint32_t tt = (uint32_t)bm;
            const uint64_t span_a = ((uint64_t)(ak ? tt : a->K) * (uint64_t)a->lda + a->K) * ES;
            const uint64_t span_b = ((uint64_t)(bk ? tt : a->K) * (uint64_t)a->ldb + a->K) * ES;
            constexpr uint32_t KS = sizeof(T) == 2 ? WK_KB16 / 2 : 32;   // k per step
            if (a->M % tt == 0 && a->N % tt == 0 && a->K % KS == 0 && p.kps % KS == 0 && p.vec_a && p.vec_b &&
                p.vec_c && span_a < (1ull << 31) && span_b < (1ull << 31)) {
                report(VKB_KERN_WAVEK);
                if (tt == 32) {
                    if (ak) {
                        if (bk) hipLaunchKernelGGL((gemm_wavek_kernel<T, true, true, 32, WK_KB16>), dim3(grid), dim3(256), 0, st, p);
                        else hipLaunchKernelGGL((gemm_wavek_kernel<T, true, false, 32, WK_KB16>), dim3(grid), dim3(256), 0, st, p);
                    } else {
                        if (bk) hipLaunchKernelGGL((gemm_wavek_kernel<T, false, true, 32, WK_KB16>), dim3(grid), dim3(256), 0, st, p);
                        else hipLaunchKernelGGL((gemm_wavek_kernel<T, false, false, 32, WK_KB16>), dim3(grid), dim3(256), 0, st, p);
                    }
                } else {
                    if (ak) {
                        if (bk) hipLaunchKernelGGL((gemm_wavek_kernel<T, true, true, 64, WK_KB16>), dim3(grid), dim3(256), 0, st, p);
                        else hipLaunchKernelGGL((gemm_wavek_kernel<T, true, false, 64, WK_KB16>), dim3(grid), dim3(256), 0, st, p);
                    } else {
                        if (bk) hipLaunchKernelGGL((gemm_wavek_kernel<T, false, true, 64, WK_KB16>), dim3(grid), dim3(256), 0, st, p);
                        else hipLaunchKernelGGL((gemm_wavek_kernel<T, false, false, 64, WK_KB16>), dim3(grid), dim3(256), 0, st, p);
                    }
                }
                return (int)hipGetLastError();
            }
        }
    }
    // only the wave-K kernel takes 32x32 tiles or divided slices
    if (tile == VKB_TILE_32 || tile == VKB_TILE_64Q) return (int)hipErrorInvalidValue;
    report(full ? VKB_KERN_GENERIC : VKB_KERN_GENERIC_CHECKED);
    switch (tile) {
        case VKB_TILE_64:  return launch_layout<T, TC, VKB_TILE_64>(p, ak, bk, !full, grid, st);
        case VKB_TILE_128: return launch_layout<T, TC, VKB_TILE_128>(p, ak, bk, !full, grid, st);
        default:           return launch_layout<T, TC, VKB_TILE_256>(p, ak, bk, !full, grid, st);
    }
}

}  // namespace vkb

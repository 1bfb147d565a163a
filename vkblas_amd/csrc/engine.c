/*
 * engine.c — host dispatcher of the MI355X-native vkblas (C11).
 *
 * Implements the public API of include/vkblas.h and include/vkblas_ext.h on
 * top of the HIP launch layer (vkb_launch.h).  It replaces the reference's
 * Vulkan engine entry points vkblas_gemm_f32 (src/vkblas.c:3104-3341) and
 * vkblas_gemm_f16 (src/vkblas.c:3517-3651) and their path selection
 * (pick_tile128 src/vkblas.c:914-928, split-K gates src/vkblas.c:2850-2867 and
 * 1636-1668, M==1 matvec gates src/vkblas.c:3122-3161 and 3535-3559).
 *
 * Differences by design:
 *   - no global lock: the only shared state is initialised once
 *     (pthread_once) and the split-K workspace is kept per stream (allocated
 *     from a stream-ordered memory pool), so concurrent calls on different
 *     streams never share it;
 *   - launches are asynchronous on the caller's stream;
 *   - every TA/TB variant runs natively (no transposed copies, no cache).
 */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <time.h>
#include <hip/hip_runtime_api.h>

#include "vkblas_ext.h"
#include "vkb_launch.h"
#include "vkb_engine.h"

#define VKBLAS_VERSION_STRING "vkblas-mi355x 0.1.0 (gfx950)"

/* ------------------------------------------------------------------ state */

#define VKB_MAX_DEVICES 64

static pthread_once_t g_once = PTHREAD_ONCE_INIT;
static int g_ndev = 0;          /* visible devices, 0 = no GPU */
static int g_trace = 0;         /* VKBLAS_TRACE */
static int g_force_tile = -1;   /* VKBLAS_TILE = 64 | 128 | 256 */
static uint32_t g_force_split = 0; /* VKBLAS_SPLITK = n (applies when split_k == 0) */
static int g_no_skinny = 0;     /* VKBLAS_NO_SKINNY = 1 */
static int g_generic_only = 0;  /* VKBLAS_KERNEL = generic */
static int g_profile = 0;       /* VKBLAS_PROFILE */
/* The reference's own path knobs, honoured under their names:
 *   VKBLAS_TILE128=0|1 (src/vkblas.c:914-919): 64x64 | 128x128 tiles (as
 *     VKBLAS_TILE=64|128, which wins when both are set);
 *   VKBLAS_NOSPLITK (any value, src/vkblas.c:2858): no split-K the planner
 *     chooses itself (a caller's split still runs);
 *   VKBLAS_HSPLITK=0 (src/vkblas.c:1637): the same for fp16 / bf16 only;
 *   VKBLAS_HT256=0|1 (src/vkblas.c:1356): fp16 / bf16 GEMMs never | always
 *     on the largest tile (256x256 here, where the pipelined kernel takes it;
 *     the reference's largest half tile was 128x256).
 * VKBLAS_M_SPLITK (the reference's skinny K split, src/vkblas.c:2309) is not
 * honoured: each decode kernel here takes the split its plan derives. */
static int g_no_split = 0;      /* VKBLAS_NOSPLITK */
static int g_no_split16 = 0;    /* VKBLAS_HSPLITK=0 */
static int g_ht256 = -1;        /* VKBLAS_HT256: -1 planner, 0 never, 1 always */

static pthread_mutex_t g_pool_lock = PTHREAD_MUTEX_INITIALIZER;
static hipMemPool_t g_pool[VKB_MAX_DEVICES];

static __thread int g_last_path = VKBLAS_PATH_NONE;
static __thread int g_last_kernel = VKBLAS_KERNEL_NONE;

static void init_once(void) {
    const char* e;
    g_trace = (e = getenv("VKBLAS_TRACE")) != NULL && e[0] && e[0] != '0';
    if ((e = getenv("VKBLAS_TILE128")) != NULL && (e[0] == '0' || e[0] == '1') && e[1] == '\0')
        g_force_tile = e[0] == '1' ? VKB_TILE_128 : VKB_TILE_64;
    if ((e = getenv("VKBLAS_TILE")) != NULL) {
        int v = atoi(e);
        g_force_tile = v == 64 ? VKB_TILE_64 : v == 128 ? VKB_TILE_128 : v == 256 ? VKB_TILE_256 : -1;
    }
    g_no_split = getenv("VKBLAS_NOSPLITK") != NULL;
    g_no_split16 = (e = getenv("VKBLAS_HSPLITK")) != NULL && e[0] == '0';
    if ((e = getenv("VKBLAS_HT256")) != NULL && (e[0] == '0' || e[0] == '1')) g_ht256 = e[0] - '0';
    if ((e = getenv("VKBLAS_SPLITK")) != NULL) {
        long v = atol(e);
        g_force_split = v > 0 ? (uint32_t)v : 0;
    }
    g_no_skinny = (e = getenv("VKBLAS_NO_SKINNY")) != NULL && e[0] == '1';
    g_generic_only = (e = getenv("VKBLAS_KERNEL")) != NULL && strcmp(e, "generic") == 0;
    g_profile = (e = getenv("VKBLAS_PROFILE")) != NULL && e[0] && e[0] != '0';
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
    g_ndev = n;
    if (g_trace) fprintf(stderr, "[vkblas] init: %s, %d device(s)\n", VKBLAS_VERSION_STRING, n);
}

static int ensure_init(void) {
    pthread_once(&g_once, init_once);
    return g_ndev > 0;
}

/* Stream-ordered workspace for split-K partials: a private pool per device
 * that keeps its memory between calls (release threshold = max). */
static hipMemPool_t pool_for_current_device(void) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= VKB_MAX_DEVICES) return NULL;
    pthread_mutex_lock(&g_pool_lock);
    if (!g_pool[dev]) {
        hipMemPoolProps props;
        memset(&props, 0, sizeof(props));
        props.allocType = hipMemAllocationTypePinned;
        props.handleTypes = hipMemHandleTypeNone;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = dev;
        hipMemPool_t pool = NULL;
        if (hipMemPoolCreate(&pool, &props) == hipSuccess) {
            uint64_t thr = UINT64_MAX;
            hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &thr);
            g_pool[dev] = pool;
        }
    }
    hipMemPool_t p = g_pool[dev];
    pthread_mutex_unlock(&g_pool_lock);
    return p;
}

/* Split-K and decode partials (the workspace).
 *
 * Eager calls: one workspace per (device, stream), kept between calls.  A
 * slot is found by the stream handle and the stream's unique id
 * (hipStreamGetId), so a stream created at a destroyed stream's address does
 * not inherit its buffer.  Work on a stream runs in order, so a call reuses
 * its stream's buffer after the kernels of the calls queued before it; a
 * stream-ordered malloc / free pair per call instead left the GPU idle for
 * about 6 us between calls.
 *  - A call holds its slot's lock from taking the buffer until its last
 *    kernel is enqueued, so two threads launching on one stream cannot
 *    interleave their pass-1 and reduce kernels on the same partials.
 *  - A call that needs more replaces the buffer (at least twice the size, up
 *    to 1 GiB) and frees the old one on the stream, ordered after the kernels
 *    that used it.
 *  - The slots hold at most VKB_WS_CACHE_BYTES together.  Calls beyond that,
 *    calls when all slots are taken, and calls on hipStreamPerThread (one
 *    handle value, a different stream in every thread) allocate their own
 *    buffer and free it on the stream after their kernels.
 * Under stream capture no buffer is handed out: a captured kernel would keep
 * the address of a buffer that later calls reuse or free, and this library
 * does not allocate inside a capture (graph-owned allocations are not used).
 * Such calls fail with VKBLAS_ERR_INIT before launching anything: the hipBLAS
 * and rocBLAS entry points then forward them to the vendor library, and
 * engine callers use vkblas_gemm_noalloc_async, whose partials live in a
 * fixed per-device array.  Calls that need no partials capture normally.
 * vkblas_workspace_release() frees every cached buffer. */
#define VKB_WS_SLOTS 64
#define VKB_WS_CACHE_BYTES ((size_t)4 << 30)
#define VKB_WS_GROW_CAP ((size_t)1 << 30)
typedef struct {
    pthread_mutex_t lock;  /* held by the call using the buffer */
    int dev;
    hipStream_t stream;
    unsigned long long sid;
    void* ptr;
    size_t bytes;
} ws_slot_t;
static ws_slot_t g_ws[VKB_WS_SLOTS] = {[0 ... VKB_WS_SLOTS - 1] = {.lock = PTHREAD_MUTEX_INITIALIZER}};
static int g_nws = 0;            /* slots claimed (never unclaimed) */
static size_t g_ws_total = 0;    /* bytes cached in the slots */

typedef struct {
    void* ptr;
    int slot;                    /* locked slot, or -1 */
    int owned;                   /* free ptr on the stream after the kernels */
    hipStream_t stream;
} ws_lease_t;

/* A workspace starts with VKB_WS_HEADER bytes of arrival counters, zero
 * when the buffer is new (the partials follow; see vkb_launch.h).  Never
 * called under stream capture: a capturing stream gets no workspace. */
static int ws_clear_header(void* p, hipStream_t stream) {
    return hipMemsetAsync(p, 0, VKB_WS_HEADER, stream) == hipSuccess ? 0 : -1;
}

static int ws_owned(hipStream_t stream, size_t bytes, hipMemPool_t pool, ws_lease_t* L) {
    if (hipMallocFromPoolAsync(&L->ptr, bytes, pool, stream) != hipSuccess) {
        L->ptr = NULL;
        return -1;
    }
    L->owned = 1;
    if (ws_clear_header(L->ptr, stream) != 0) {
        hipFreeAsync(L->ptr, stream);
        L->ptr = NULL;
        L->owned = 0;
        return -1;
    }
    return 0;
}

/* The stream's unique id, or 0.  hipStreamGetId is resolved at run time: HIP
 * runtimes before 7.1 (PyTorch's bundled one among them) lack it, and a
 * direct reference would keep the library from loading into such a
 * process.  Without it slots are keyed by the handle value alone. */
typedef hipError_t (*stream_id_fn_t)(hipStream_t, unsigned long long*);
static stream_id_fn_t g_stream_id_fn;
static pthread_once_t g_stream_id_once = PTHREAD_ONCE_INIT;
static void stream_id_init(void) { g_stream_id_fn = (stream_id_fn_t)dlsym(RTLD_DEFAULT, "hipStreamGetId"); }
static unsigned long long stream_id(hipStream_t stream) {
    pthread_once(&g_stream_id_once, stream_id_init);
    unsigned long long sid = 0;
    if (!g_stream_id_fn || g_stream_id_fn(stream, &sid) != hipSuccess) sid = 0;
    return sid;
}

/* 0 and L->ptr set, or -1.  Always pair with ws_release. */
static int ws_acquire(hipStream_t stream, size_t bytes, ws_lease_t* L) {
    L->ptr = NULL;
    L->slot = -1;
    L->owned = 0;
    L->stream = stream;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return -1;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) {
        if (g_trace) fprintf(stderr, "[vkblas] stream is capturing: no workspace for partials, declined\n");
        return -1;
    }
    hipMemPool_t pool = pool_for_current_device();
    if (!pool) return -1;
    if (stream == hipStreamPerThread) return ws_owned(stream, bytes, pool, L);
    unsigned long long sid = stream_id(stream);

    pthread_mutex_lock(&g_pool_lock);
    int i = 0;
    while (i < g_nws && !(g_ws[i].dev == dev && g_ws[i].stream == stream && g_ws[i].sid == sid)) ++i;
    if (i == g_nws && g_nws < VKB_WS_SLOTS) {
        g_ws[i].dev = dev;
        g_ws[i].stream = stream;
        g_ws[i].sid = sid;
        g_ws[i].ptr = NULL;
        g_ws[i].bytes = 0;
        ++g_nws;
    }
    pthread_mutex_unlock(&g_pool_lock);
    if (i >= VKB_WS_SLOTS) return ws_owned(stream, bytes, pool, L);

    ws_slot_t* s = &g_ws[i];
    pthread_mutex_lock(&s->lock);
    if (s->bytes >= bytes) {
        L->ptr = s->ptr;
        L->slot = i;
        return 0;
    }
    size_t want = bytes;
    if (s->bytes * 2 > want) want = s->bytes * 2 < VKB_WS_GROW_CAP ? s->bytes * 2 : (VKB_WS_GROW_CAP > want ? VKB_WS_GROW_CAP : want);
    pthread_mutex_lock(&g_pool_lock);
    const int fits = g_ws_total - s->bytes + want <= VKB_WS_CACHE_BYTES;
    if (fits) g_ws_total = g_ws_total - s->bytes + want;
    pthread_mutex_unlock(&g_pool_lock);
    if (!fits) {
        pthread_mutex_unlock(&s->lock);
        return ws_owned(stream, bytes, pool, L);
    }
    void* p = NULL;
    if (hipMallocFromPoolAsync(&p, want, pool, stream) != hipSuccess || ws_clear_header(p, stream) != 0) {
        if (p) hipFreeAsync(p, stream);
        pthread_mutex_lock(&g_pool_lock);
        g_ws_total = g_ws_total + s->bytes - want;
        pthread_mutex_unlock(&g_pool_lock);
        pthread_mutex_unlock(&s->lock);
        return -1;
    }
    if (s->ptr) hipFreeAsync(s->ptr, stream);   /* after the kernels that used it */
    s->ptr = p;
    s->bytes = want;
    L->ptr = p;
    L->slot = i;
    return 0;
}

static void ws_release(ws_lease_t* L) {
    if (L->owned && L->ptr) hipFreeAsync(L->ptr, L->stream);
    if (L->slot >= 0) pthread_mutex_unlock(&g_ws[L->slot].lock);
    L->ptr = NULL;
    L->slot = -1;
    L->owned = 0;
}

vkblas_status_t vkblas_workspace_release(void) {
    pthread_once(&g_once, init_once);
    if (g_ndev <= 0) return VKBLAS_OK;
    int cur = 0;
    if (hipGetDevice(&cur) != hipSuccess) return VKBLAS_ERR_INIT;
    vkblas_status_t st = VKBLAS_OK;
    /* A slot's lock before g_pool_lock, the order ws_acquire takes them in.
     * Slots below g_nws stay claimed, so the count read here stays valid. */
    pthread_mutex_lock(&g_pool_lock);
    const int nws = g_nws;
    pthread_mutex_unlock(&g_pool_lock);
    for (int i = 0; i < nws; ++i) {
        ws_slot_t* s = &g_ws[i];
        pthread_mutex_lock(&s->lock);
        if (s->ptr) {
            /* the stream may be gone: order the free after everything on the device */
            if (hipSetDevice(s->dev) != hipSuccess || hipDeviceSynchronize() != hipSuccess ||
                hipFreeAsync(s->ptr, NULL) != hipSuccess || hipStreamSynchronize(NULL) != hipSuccess)
                st = VKBLAS_ERR_INIT;
            pthread_mutex_lock(&g_pool_lock);
            g_ws_total -= s->bytes;
            pthread_mutex_unlock(&g_pool_lock);
            s->ptr = NULL;
            s->bytes = 0;
        }
        pthread_mutex_unlock(&s->lock);
    }
    pthread_mutex_lock(&g_pool_lock);
    for (int d = 0; d < VKB_MAX_DEVICES && d < g_ndev; ++d)
        if (g_pool[d] && (hipSetDevice(d) != hipSuccess || hipMemPoolTrimTo(g_pool[d], 0) != hipSuccess))
            st = VKBLAS_ERR_INIT;
    pthread_mutex_unlock(&g_pool_lock);
    if (hipSetDevice(cur) != hipSuccess) st = VKBLAS_ERR_INIT;
    return st;
}

/* --------------------------------------------------------------- planning */

static uint32_t cdiv(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

static int tile_path(int tile) {
    return tile == VKB_TILE_256 ? VKBLAS_PATH_TILE256
         : tile == VKB_TILE_128 ? VKBLAS_PATH_TILE128 : VKBLAS_PATH_TILE64;
}

/* vkblas_dtype_t -> kernel element type (vkb_launch.h); the values match */
static int kernel_type(vkblas_dtype_t t) {
    return t == VKBLAS_DT_F16 ? VKB_T_F16 : t == VKBLAS_DT_BF16 ? VKB_T_BF16 : VKB_T_F32;
}

static const char* type_name(int t) {
    return t == VKB_T_F16 ? "f16" : t == VKB_T_BF16 ? "bf16" : "f32";
}

/* The pipelined kernel runs the given tile (256x256 or 128x128): M and N at
 * least the tile (edge tiles shift back inside the matrix), N % 4 == 0, the
 * ragged dimension of an MN-major operand (A with op_a = T, B with op_b = N)
 * a multiple of 16 bytes, K a multiple of two K steps, 16-byte aligned
 * operands with vector-multiple leading dimensions.  The launcher checks the
 * rest (C alignment, 32-bit spans) and otherwise runs the generic kernel on
 * the same plan. */
#define PIPE_MIN_STEPS 4u
static int pipe_ok(vkblas_dtype_t ab_type, int tile, vkblas_op_t op_a, vkblas_op_t op_b, uint32_t M, uint32_t N,
                   uint32_t K, uint32_t lda, uint32_t ldb, int aligned) {
    const uint32_t vec = ab_type == VKBLAS_DT_F32 ? 4 : 8;
    const uint32_t kpair = 2 * vkb_tile_bk(kernel_type(ab_type));
    const uint32_t edge = vkb_tile_bm(tile);
    if (tile != VKB_TILE_256 && tile != VKB_TILE_128) return 0;
    /* M below the tile: 128x128 tiles with K-major A (op_a = N), fp32 from
     * 65 rows (fewer waste three quarters of the tile's MFMAs or more: fp32
     * M = 64 / 32 against N = K = 8192 took 124 / 122 us there, 84 / 130 on
     * the generic kernel; M = 65 / 96 fp32 207 / 206 -> 131 / 132 us, fp16
     * 42.2 / 49.7 -> 36.9 / 38.5), 16-bit from 25 (the planner prefers them
     * to the decode kernels there, see below) */
    return aligned && !g_generic_only &&
           (M >= edge || (tile == VKB_TILE_128 && op_a == VKBLAS_OP_N && M > (ab_type == VKBLAS_DT_F32 ? 64u : 24u))) &&
           N >= edge && N % 4 == 0 &&
           (op_a == VKBLAS_OP_N || M % vec == 0) && (op_b == VKBLAS_OP_T || N % vec == 0) && K % kpair == 0 &&
           lda % vec == 0 && ldb % vec == 0;
}

/* Split-K pass 1 on tt x tt tiles (32 or 64) by the wave-K kernel (its
 * launcher's conditions): whole tiles, K in whole steps (32 k for fp32, 64
 * for 16-bit types; the planner's slices are multiples of that), aligned
 * operands and leading dimensions, operand spans below 2^31 bytes. */
static int wavek_ok(vkblas_dtype_t ab_type, uint32_t tt, vkblas_op_t op_a, vkblas_op_t op_b, uint32_t M, uint32_t N,
                    uint32_t K, uint32_t lda, uint32_t ldb, int aligned) {
    const uint32_t vec = ab_type == VKBLAS_DT_F32 ? 4 : 8;
    const uint64_t es = ab_type == VKBLAS_DT_F32 ? 4 : 2;
    const uint64_t span_a = ((uint64_t)(op_a == VKBLAS_OP_N ? tt : K) * lda + K) * es;
    const uint64_t span_b = ((uint64_t)(op_b == VKBLAS_OP_T ? tt : K) * ldb + K) * es;
    return aligned && !g_generic_only && M % tt == 0 && N % tt == 0 && K % (vec == 4 ? 32 : 64) == 0 &&
           lda % vec == 0 &&
           ldb % vec == 0 && span_a < (1ull << 31) && span_b < (1ull << 31);
}

/* Tile choice for 256 CUs: the largest tile that still gives about one
 * workgroup per CU; smaller tiles only when the large one would starve. */
static int choose_tile(uint32_t M, uint32_t N, uint32_t batch) {
    if (g_force_tile >= 0) return g_force_tile;
    uint64_t t256 = (uint64_t)cdiv(M, 256) * cdiv(N, 256) * batch;
    uint64_t t128 = (uint64_t)cdiv(M, 128) * cdiv(N, 128) * batch;
    if (M >= 256 && N >= 256 && t256 >= 224) return VKB_TILE_256;
    if (M >= 96 && N >= 96 && t128 >= 96) return VKB_TILE_128;
    if (M > 64 && N > 64 && t128 >= 32) return VKB_TILE_128;
    return VKB_TILE_64;
}

vkblas_status_t vkblas_plan_gemm(vkblas_dtype_t ab_type, vkblas_dtype_t c_type,
                                 vkblas_op_t op_a, vkblas_op_t op_b,
                                 uint32_t M, uint32_t N, uint32_t K,
                                 uint32_t lda, uint32_t ldb, uint32_t ldc,
                                 uint32_t batch, uint32_t split_k, int aligned,
                                 vkblas_plan_t* plan) {
    pthread_once(&g_once, init_once);
    if (!plan) return VKBLAS_ERR_PARAM;
    memset(plan, 0, sizeof(*plan));
    if (M == 0 || N == 0 || K == 0 || batch == 0) return VKBLAS_ERR_PARAM;
    /* the kernels index rows, columns and k with 32-bit signed integers (their
     * pointer arithmetic is 64-bit); larger dimensions are declined, and the
     * hipBLAS / rocBLAS / hipBLASLt entry points forward such calls */
    if (M > 0x7fffffffu || N > 0x7fffffffu || K > 0x7fffffffu) return VKBLAS_ERR_PARAM;
    if (!((ab_type == VKBLAS_DT_F32 && (c_type == VKBLAS_DT_F32 || c_type == VKBLAS_DT_F16 || c_type == VKBLAS_DT_BF16)) ||
          (ab_type == VKBLAS_DT_F16 && (c_type == VKBLAS_DT_F16 || c_type == VKBLAS_DT_F32)) ||
          (ab_type == VKBLAS_DT_BF16 && (c_type == VKBLAS_DT_BF16 || c_type == VKBLAS_DT_F32))))
        return VKBLAS_ERR_PARAM;
    /* Leading dimensions are taken as given, as the reference engine does
     * (its tests pass lda < M with op_a = T: test/test_h.c:105); only 0 is
     * rejected.  BLAS-style ld >= rows checks live in the hipBLAS shim. */
    if (lda == 0 || ldb == 0 || ldc == 0) return VKBLAS_ERR_PARAM;
    if (split_k == 0 && g_force_split) split_k = g_force_split;
    if (split_k == 0 && (g_no_split || (g_no_split16 && ab_type != VKBLAS_DT_F32))) split_k = 1;

    /* decode-shaped: X[M, K] (K-contiguous rows) against a weight W.
     * fp16 / bf16: M <= 64, W stored N x K (op_b = T) or K x N (op_b = N);
     * fp32, fp32 output: M <= 64 with W stored N x K (17-64 rows: the decode
     * kernel; 17-32 rows against 14336 x 4096 52 us where the tile paths
     * took 160, 4096 x 4096 20 against 48), M <= 64 with W K x N (17-32 rows
     * 14336 x 4096 56-58 against 242-244 us).  At exactly 64
     * rows the tile paths are within -8 .. +11 % of it; at 48 rows they are
     * 1.6-2.2x slower (edge rows).  vkb_skinny_plan holds the
     * kernels' own limits (leading dimensions, 32-bit buffer spans) and
     * returns their K split, or 0: then a tile path. */
    /* 16-bit, 33-64 rows against a weight of at most 12288 x 4096 elements,
     * K >= 4096 and at most 128 column tiles of 128: the short-M pipelined
     * tiles with a K split (below) beat the decode kernels.  fp16, one box,
     * three weight copies rotated per call (no reuse of the 256 MB MALL
     * between calls), M = 40 / 48 / 64, decode -> tiles: 4096^2 15.3 / 15.7 /
     * 18.6 -> 13.5 / 13.4 / 14.4 us, 11008 x 4096 27.6 / 29.4 / 32.8 -> 22.7 /
     * 23.2 / 24.8, 12288 x 4096 28.6 / 30.5 / 33.7 -> 27.0 / 27.6 / 28.5.
     * Larger weights keep the decode kernels: 8192^2 29.9 / 30.5 / 32.8
     * against 39.4 / 39.6 / 40.4 on tiles (weight K x N 32.1 / 32.0 / 35.2
     * against 33.6 / 35.9 / 37.9), 14336 x 4096 29.9 / 31.5 / 34.3 against
     * 34.1 / 34.4 / 35.0, 4096 x 14336 27.2 / 28.0 / 31.8 against 29.7 /
     * 29.0 / 29.3.  (With one weight resident in MALL the tiles measure
     * 25-28 us at 8192^2: a single-weight loop overstates them.) */
    const int tiles_first = ab_type != VKBLAS_DT_F32 && M > 32u && (uint64_t)N * K <= 12288ull * 4096ull &&
                            K >= 4096 && split_k == 0 && batch == 1 &&
                            g_force_tile < 0 && cdiv(N, 128) <= 128 &&
                            pipe_ok(ab_type, VKB_TILE_128, op_a, op_b, M, N, K, lda, ldb, aligned);
    if (op_a == VKBLAS_OP_N && batch == 1 && split_k <= 1 && aligned && !g_no_skinny && !tiles_first &&
        (ab_type != VKBLAS_DT_F32 || c_type == VKBLAS_DT_F32)) {
        const uint32_t sp = vkb_skinny_plan(kernel_type(ab_type), op_b == VKBLAS_OP_T, M, N, K, lda, ldb);
        if (sp) {
            plan->path = VKBLAS_PATH_SKINNY;
            plan->tile = VKB_TILE_64;
            plan->split = sp;
            plan->k_per_split = K;   /* the skinny kernels split K themselves */
            return VKBLAS_OK;
        }
    }

    const uint32_t bk = vkb_tile_bk(kernel_type(ab_type));
    int tile = choose_tile(M, N, batch);
    if (g_force_tile < 0) {
        /* Where both pipelined tile sizes apply, the measured crossovers
         * (square shapes, NN and NT, one box):
         * - fp32: 128x128 tiles are never slower, and faster wherever
         *   256x256 tiles leave a partial wave of one workgroup per CU
         *   (5120^3 131.5 against 116.3 TFLOP/s, 6144^3 147.7 / 110.9;
         *   4096^3 and the 64 x 512^3 batch equal): 256x256 only for about
         *   whole waves.
         * - 16-bit: 256x256 tiles from more than 128 of them on (3072^3
         *   fp16, 144 tiles, 963 against 793 TFLOP/s, 3584^3 1154-1245 /
         *   1017-1048; 2560^3, 100 tiles: 656 against 989; exactly 128,
         *   half the CUs: 2048 x 4096 x 4096 81.1 against 58.8 us, 1024 x
         *   8192 x 8192 144.0 against 112.3). */
        const uint64_t t256 = (uint64_t)cdiv(M, 256) * cdiv(N, 256) * batch;
        if (ab_type == VKBLAS_DT_F32 && tile == VKB_TILE_256 &&
            pipe_ok(ab_type, VKB_TILE_128, op_a, op_b, M, N, K, lda, ldb, aligned) &&
            8 * t256 < 7 * 256 * ((t256 + 255) / 256))
            tile = VKB_TILE_128;
        if (ab_type != VKBLAS_DT_F32 && tile == VKB_TILE_128 && t256 > 128 &&
            pipe_ok(ab_type, VKB_TILE_256, op_a, op_b, M, N, K, lda, ldb, aligned))
            tile = VKB_TILE_256;
        if (ab_type != VKBLAS_DT_F32 && g_ht256 == 1 &&
            pipe_ok(ab_type, VKB_TILE_256, op_a, op_b, M, N, K, lda, ldb, aligned))
            tile = VKB_TILE_256;
        if (ab_type != VKBLAS_DT_F32 && g_ht256 == 0 && tile == VKB_TILE_256) tile = VKB_TILE_128;
    }
    uint32_t split = 1;
    if (batch == 1) {
        if (split_k > 1) {
            split = split_k;
            /* a caller's split with whole 128x128 tiles that give at least
             * 224 workgroups: pass 1 on the pipelined 128x128 kernel (at
             * M = N = 256 with 64 slices, as the planner's own choice below) */
            if (g_force_tile < 0 && pipe_ok(ab_type, VKB_TILE_128, op_a, op_b, M, N, K, lda, ldb, aligned) &&
                (uint64_t)cdiv(M, 128) * cdiv(N, 128) * split_k >= 224 && K / split_k >= PIPE_MIN_STEPS * bk)
                tile = VKB_TILE_128;
            /* fewer: the wave-K kernel on 64x64 tiles if they give at least
             * 224 workgroups; else on 64x64 tiles with each K slice over
             * VKB_WAVEK_NQ workgroups if that gives 224 (slices of at least
             * 4 K steps per workgroup); else on 32x32 tiles.  M = N = 256:
             * split 16 -> 256 workgroups of 64x64, split 4 -> 256 of 64x64
             * in quarter slices.  Split 4, whole call, 32x32 tiles against
             * quarter slices (bench.py --only splitk, two boxes): K = 65536
             * fp32 87.5-88.2 -> 74.2-74.5 us, fp16 36.3-37.2 -> 20.3-20.6 us;
             * K = 262144 fp32 344.4-344.8 -> 270.6-271.0 us, fp16 133.2-
             * 133.6 -> 68.5-69.2 us. */
            else if (g_force_tile < 0 && wavek_ok(ab_type, 64, op_a, op_b, M, N, K, lda, ldb, aligned) &&
                     (uint64_t)(M / 64) * (N / 64) * split_k >= 224)
                tile = VKB_TILE_64;
            else if (g_force_tile < 0 && wavek_ok(ab_type, 64, op_a, op_b, M, N, K, lda, ldb, aligned) &&
                     (uint64_t)(M / 64) * (N / 64) * split_k * VKB_WAVEK_NQ >= 224 &&
                     (uint64_t)(M / 64) * (N / 64) * split_k <= VKB_WS_COUNTERS &&
                     K / split_k >= VKB_WAVEK_NQ * 4u * (ab_type == VKBLAS_DT_F32 ? 32u : 64u))
                tile = VKB_TILE_64Q;
            else if (g_force_tile < 0 && wavek_ok(ab_type, 32, op_a, op_b, M, N, K, lda, ldb, aligned))
                tile = VKB_TILE_32;
        } else if (split_k == 0 && g_force_tile < 0 && pipe_ok(ab_type, VKB_TILE_128, op_a, op_b, M, N, K, lda, ldb, aligned) &&
                   (uint64_t)cdiv(M, 128) * cdiv(N, 128) <= 128 && K >= 4096) {
            /* 128x128 tiles, at most 128 of them (at most half the CUs), and
             * a long K: the pipelined kernel runs pass 1 on 128x128 tiles
             * with 256 / tiles slices, a workgroup per CU.  Each workgroup
             * reads its A and B slices once; the tiles of one slice sit on
             * one XCD and share those reads in L2.
             * Mid-size M against a large weight (fp16, N = K = 8192, one
             * box): M = 128 (64 tiles) 73.0 -> 43.0 us with 4 slices, M = 192
             * / 256 (128 tiles) 71.7 / 70.9 -> 54.8 / 56.8 us with 2; 192
             * tiles (M = 384) are fastest unsplit.
             * 16-bit inputs (HBM-bound here): the launcher runs four LDS
             * stages (three K steps of loads in flight).  Measured at
             * M = N = 256, fp16, K = 262144: 54.5 us (4.9 TB/s) against
             * 79.7 us with 256x256 tiles and 128 slices; 32 / 48 / 96 / 128
             * slices of 128x128: 79.6 / 65.1 / 72.9 / 63.4 us.
             * fp32 (MFMA-bound): at M = N = 256, K = 65536 / 262144, 64
             * slices take 70.7 / 260.9 us; 32 / 128 / 256 slices 126.9 /
             * 74.0 / 85.9 and 482.4 / 260.9 / 271.6 us; 256x256 tiles with
             * 256 slices (a quarter of the K steps per workgroup, four times
             * the partials) 88.7 / 263.2 us. */
            const uint32_t kpair = 2 * bk;
            const uint64_t t128 = (uint64_t)cdiv(M, 128) * cdiv(N, 128);
            uint64_t want = 256 / t128;
            uint64_t kmax = K / (PIPE_MIN_STEPS * bk);
            if (want > kmax) want = kmax;
            if (want >= 2) {
                uint32_t kps = cdiv(cdiv(K, want), kpair) * kpair;
                split = cdiv(K, kps);
                tile = VKB_TILE_128;
            }
        } else if (split_k == 0 && g_force_tile < 0 && ab_type != VKBLAS_DT_F32 && K >= 16384 &&
                   pipe_ok(ab_type, VKB_TILE_256, op_a, op_b, M, N, K, lda, ldb, aligned) &&
                   (uint64_t)cdiv(M, 256) * cdiv(N, 256) > 64 && (uint64_t)cdiv(M, 256) * cdiv(N, 256) <= 128) {
            /* 16-bit, 65-128 tiles of 256x256 (a quarter to a half of the
             * CUs) and a very long K: 256 / tiles slices of 256x256 tiles
             * rather than unsplit 128x128 ones.  1024 x 8192 x 28672 fp16
             * (128 tiles, one box): 393.4 against 524.4 us; at K = 14336
             * the two are level (195.3 / 198.9), at 8192 128x128 wins. */
            split = 256 / (uint32_t)((uint64_t)cdiv(M, 256) * cdiv(N, 256));
            tile = VKB_TILE_256;
        } else if (split_k == 0) {
            /* Few output tiles and a long K: split K.  128x128 tiles (reuse
             * of each A / B slice over 128 columns / rows) when the output
             * allows; slices of at least 1024 k; up to ~512 workgroups (two
             * per CU) and 128 slices.  Measured at M = N = 256: K = 65536 ->
             * 64 slices, K = 262144 -> 128 slices are the fastest choices;
             * M = 65 / 96 against N = K = 8192 (64 generic 128x128 tiles):
             * 147.1 / 143.7 -> 43.5 / 49.5 us with 8 slices. */
            const int stile = (M >= 128 && N >= 128 && g_force_tile < 0) ? VKB_TILE_128 : tile;
            uint64_t tiles = (uint64_t)cdiv(M, vkb_tile_bm(stile)) * cdiv(N, vkb_tile_bn(stile));
            if (tiles <= 128 && K >= 4096) {
                uint64_t want = K / 1024;
                if (want > 512 / tiles) want = 512 / tiles;
                if (want > 128) want = 128;
                uint64_t kmax = K / (8 * bk);   /* keep >= 8 K steps per slice */
                if (want > kmax) want = kmax;
                if (want >= 2) {
                    split = (uint32_t)want;
                    tile = stile;
                }
            }
        }
    }
    if (split > 1) {
        /* slices of whole K steps; of whole step pairs for the pipelined kernel */
        const int pipe = pipe_ok(ab_type, tile, op_a, op_b, M, N, K, lda, ldb, aligned);
        const uint32_t gran = pipe ? 2 * bk : bk;
        uint32_t kps = cdiv(cdiv(K, split), gran) * gran;
        split = cdiv(K, kps);                     /* every slice non-empty */
        /* cap the fp32 partials at 1 GiB */
        while (split > 1 && (uint64_t)split * M * N * 4 > (1ull << 30)) {
            split = (split + 1) / 2;
            kps = cdiv(cdiv(K, split), gran) * gran;
            split = cdiv(K, kps);
        }
        if (split > 1) {
            plan->path = VKBLAS_PATH_SPLITK;
            plan->tile = tile;
            plan->split = split;
            plan->k_per_split = kps;
            return VKBLAS_OK;
        }
        /* no split left (K within one slice): 32x32 tiles and divided
         * slices exist only for split-K pass 1 */
        if (tile == VKB_TILE_32 || tile == VKB_TILE_64Q) tile = choose_tile(M, N, batch);
    }
    /* A partial last wave: with T tiles on `slots` concurrent workgroups
     * (one 256x256 or two 128x128 per CU on 256 CUs), T = W slots + R and
     * R at most half a wave leaves most CUs idle for a whole tile time.
     * The rows of the first tiles_m - r tile rows then run as tiles (W
     * waves, a few slots idle) and the last r rows (the R tiles rounded up
     * to whole rows) as split-K with as many slices as fit in one wave,
     * pass 1 on the same pipelined tile.  Measured (one box): fp32 3072^3
     * on 128x128 tiles 509.0 -> 411.3 us (7 slices of 3 tile rows; 4 / 8
     * slices 439.9 / 428.1), fp32 5120^3 1991.7 -> 1819.2 us (6 slices of
     * 2 rows). */
    if (split_k == 0 && batch == 1 && (tile == VKB_TILE_128 || tile == VKB_TILE_256) &&
        pipe_ok(ab_type, tile, op_a, op_b, M, N, K, lda, ldb, aligned)) {
        const uint32_t edge = vkb_tile_bm(tile);
        const uint64_t slots = tile == VKB_TILE_256 ? 256 : 512;
        const uint64_t tm = cdiv(M, edge), tn = cdiv(N, edge), T = tm * tn;
        const uint64_t W = T / slots, R = T % slots;
        if (W >= 1 && R > 0 && 2 * R <= slots) {
            const uint64_t rows_t = (R + tn - 1) / tn;            /* tail tile rows */
            const uint32_t head = (uint32_t)((tm - rows_t) * edge);
            const uint32_t tail = M - head;
            uint64_t s = slots / (rows_t * tn);
            const uint64_t kmax = K / (PIPE_MIN_STEPS * bk);
            if (s > kmax) s = kmax;
            const uint32_t kpair = 2 * bk;
            if (s >= 2 && tail >= edge && s * tail * (uint64_t)N * 4 <= (1ull << 30)) {
                const uint32_t kps = cdiv(cdiv(K, s), kpair) * kpair;
                plan->path = VKBLAS_PATH_TAIL;
                plan->tile = tile;
                plan->split = cdiv(K, kps);
                plan->k_per_split = kps;
                plan->tail_rows = tail;
                return VKBLAS_OK;
            }
        }
    }
    plan->path = tile_path(tile);
    plan->tile = tile;
    plan->split = 1;
    plan->k_per_split = K;
    return VKBLAS_OK;
}

/* -------------------------------------------------------------- execution */

static const char* path_name(int p) {
    switch (p) {
        case VKBLAS_PATH_TILE64: return "tile64";
        case VKBLAS_PATH_TILE128: return "tile128";
        case VKBLAS_PATH_TILE256: return "tile256";
        case VKBLAS_PATH_SPLITK: return "splitk";
        case VKBLAS_PATH_SKINNY: return "skinny";
        case VKBLAS_PATH_TAIL: return "tail";
        default: return "none";
    }
}

/* VKBLAS_PROFILE: per call, the host time to plan and enqueue and the GPU
 * time of the call's kernels (events on the stream; the call then waits for
 * its kernels, as every call of the reference's engine did,
 * src/vkblas.c:954-968).  Not under stream capture. */
typedef struct {
    int on;
    double t0, t1;
    hipEvent_t e0, e1;
} prof_t;

static double now_us(void) {
    struct timespec ts;
    clock_gettime(CLOCK_MONOTONIC, &ts);
    return ts.tv_sec * 1e6 + ts.tv_nsec * 1e-3;
}

static void prof_begin(prof_t* pf, hipStream_t stream) {
    memset(pf, 0, sizeof(*pf));
    if (!g_profile) return;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) return;
    if (hipEventCreate(&pf->e0) != hipSuccess) return;
    if (hipEventCreate(&pf->e1) != hipSuccess) {
        hipEventDestroy(pf->e0);
        return;
    }
    pf->on = 1;
    pf->t0 = now_us();
    hipEventRecord(pf->e0, stream);
}

static void prof_end(prof_t* pf, hipStream_t stream, const char* what, int ok) {
    if (!pf->on) return;
    pf->t1 = now_us();
    hipEventRecord(pf->e1, stream);
    float ms = -1.0f;
    if (ok && hipEventSynchronize(pf->e1) == hipSuccess) hipEventElapsedTime(&ms, pf->e0, pf->e1);
    fprintf(stderr, "[vkblas] prof: %s enqueue=%.1fus gpu=%.1fus\n", what, pf->t1 - pf->t0, ms * 1e3);
    hipEventDestroy(pf->e0);
    hipEventDestroy(pf->e1);
}

/* A decode-planned call small enough for gemm_direct_kernel, one launch of
 * small tiles: the decode kernels then run a handful of workgroups, or split
 * K and pay a second launch for the reduce.  Measured (us, decode kernels
 * against direct, one box; calls under 8.2 us are bound by the launch):
 *   fp32 NT, 64 rows: 128 x 256 9.5 / 8.1, 1024^2 13.6 / 10.1; 512 x 4096
 *   14.4 / 22.1, 2048^2 15.3 / 24.1; NN, 1-64 rows: 1024^2 11.2-13.9 / 8.2-8.8,
 *   2048^2 11.2-17.9 / 11.6-20.7;
 *   fp16 NT, 17-64 rows: 1024^2 10.9-11.8 / 8.4-8.6, 2048^2 11.5 / 9.6-10.9,
 *   512 x 4096 10.9-12.3 / 11.4-12.5; NN, 1-64 rows: 2048^2 11.0-13.9 / 8.8-10.6,
 *   512 x 4096 11.3 / 11.3.
 * Up to 16 rows against N x K the decode kernels are level or ahead.  So they
 * are (us of GPU time, 1500 calls of random sizes)
 *   where N alone is large and the tiles many: from N = 8192 on, fp16 K x N
 *   from 16384 (fp32 NT 17 x 12264 x 64 3.5 / 4.7, NN 1 x 9392 x 16 2.8 / 3.9, 1 x
 *   52168 x 16 3.2 / 7.1; fp16 NT 20 x 17784 x 16 4.8 / 8.0, NN 2 x 19440 x 24 3.7 /
 *   6.1, 2 x 59080 x 24 3.8 / 10.8; 4 x 12032 x 56 4.5 / 3.7);
 *   fp32 past K = 1280, where four waves share too long a K on few tiles (NT 48
 *   x 96 x 1920 10.8 / 13.5, 20 x 440 x 1776 9.0 / 10.8; NN 32 x 40 x 1896 8.7 / 9.7);
 *   fp32 K x N, one or two rows and at most 32 k (1 x 6888 x 8 3.0 / 3.4);
 *   fp16 NT past K = 512 where the tiles of 32 x 32 are more than the CUs (33 x
 *   5576 x 640, 350 tiles, 5.6 / 7.2; 64 x 4088 x 856, 256, 9.3 / 5.8; 64 x 6272 x
 *   352, 392, 7.3 / 4.1).
 * They keep leading dimensions of which 64 rows span 2 GiB (the last token of
 * each of a few long sequences): gemm_direct_kernel's offsets are 32-bit. */
static int small_decode(vkblas_dtype_t ab_type, vkblas_op_t op_b, uint32_t M, uint32_t N, uint32_t K, uint32_t lda,
                        uint32_t ldb) {
    const int f32 = ab_type == VKBLAS_DT_F32, kn = op_b == VKBLAS_OP_N;
    const uint64_t span = 65ull * (lda > ldb ? lda : ldb) * (f32 ? 4 : 2);
    return span < 1ull << 31 && g_force_tile < 0 && !g_generic_only && (M >= 17 || kn) && N >= 32 &&
           N <= (kn && !f32 ? 16384u : 8192u) && K <= (f32 ? 1280u : 2048u) && !(f32 && kn && M <= 2 && K <= 32) &&
           (f32 || kn || K <= 512 || ((M + 31) / 32) * ((N + 31) / 32) <= 256) &&
           (uint64_t)N * K <= (f32 ? 1ull << 20 : 1ull << 22);
}

/* The body of vkblas_gemm_async.  ws_ext != NULL: the split-K / decode
 * partials go to that buffer of ws_ext_bytes (a call that needs more is
 * rejected with VKBLAS_ERR_PARAM) and nothing is allocated; else the
 * stream's workspace. */
static vkblas_status_t gemm_impl(vkblas_dtype_t ab_type, vkblas_dtype_t c_type, vkblas_op_t op_a, vkblas_op_t op_b,
                                 uint32_t M, uint32_t N, uint32_t K, float alpha, const void* A, uint32_t lda,
                                 const void* B, uint32_t ldb, float beta, void* C, uint32_t ldc, uint32_t batch,
                                 int64_t stride_a, int64_t stride_b, int64_t stride_c,
                                 vkblas_scalar_mode_t scalar_mode, const void* alpha_dev, const void* beta_dev,
                                 uint32_t split_k, const vkblas_epilogue_t* epi, void* stream, void* ws_ext,
                                 size_t ws_ext_bytes) {
    if (!A || !B || !C) return VKBLAS_ERR_PARAM;
    vkb_epilogue_args ep;
    memset(&ep, 0, sizeof(ep));
    if (epi) {
        if (epi->bias && epi->bias_type != VKBLAS_DT_F32 && epi->bias_type != VKBLAS_DT_F16 &&
            epi->bias_type != VKBLAS_DT_BF16)
            return VKBLAS_ERR_PARAM;
        if (epi->c_in && epi->ldc_in == 0) return VKBLAS_ERR_PARAM;
        ep.c_in = epi->c_in;
        ep.ldc_in = epi->ldc_in;
        ep.stride_c_in = epi->stride_c_in;
        ep.bias = epi->bias;
        ep.bias_type = kernel_type(epi->bias_type);
    }
    const vkb_epilogue_args* epp = epi ? &ep : NULL;
    if (scalar_mode != VKBLAS_SCALAR_HOST && (!alpha_dev || !beta_dev)) return VKBLAS_ERR_PARAM;
    if (scalar_mode != VKBLAS_SCALAR_HOST && scalar_mode != VKBLAS_SCALAR_DEV_F32 &&
        scalar_mode != VKBLAS_SCALAR_DEV_F16)
        return VKBLAS_ERR_PARAM;
    const int aligned = ((uintptr_t)A % 16 == 0) && ((uintptr_t)B % 16 == 0);
    vkblas_plan_t plan;
    vkblas_status_t st = vkblas_plan_gemm(ab_type, c_type, op_a, op_b, M, N, K, lda, ldb, ldc,
                                          batch, split_k, aligned, &plan);
    if (st != VKBLAS_OK) return st;
    if (!ensure_init()) return VKBLAS_ERR_INIT;

    const int ab = kernel_type(ab_type);
    const int ct = kernel_type(c_type);
    const hipStream_t hs = (hipStream_t)stream;
    int rc = 0;
    int c_written = 0; /* a kernel writing part of C was enqueued before a later launch of this call failed */
    int kernel = VKBLAS_KERNEL_SKINNY;
    if (g_trace)
        fprintf(stderr, "[vkblas] gemm %s%s %s->%s M=%u N=%u K=%u lda=%u ldb=%u ldc=%u batch=%u path=%s split=%u%s\n",
                op_a ? "T" : "N", op_b ? "T" : "N", type_name(ab), type_name(ct), M, N, K, lda, ldb, ldc, batch,
                path_name(plan.path), plan.split, ws_ext ? " (scratch)" : "");

    /* workspace: the arrival counters (VKB_WS_HEADER bytes), then the
     * partials: [split][M][N] fp32 for split-K and the split decode kernel,
     * [split][tail_rows][N] for the split tail; with divided K slices
     * (VKB_TILE_64Q) then the parts' sums, VKB_WAVEK_NQ x the partials */
    const int direct = plan.path == VKBLAS_PATH_SKINNY && small_decode(ab_type, op_b, M, N, K, lda, ldb);
    if (direct && plan.split > 1 && !ws_ext) {
        /* Under stream capture a decode plan with a K split has always been
         * refused (for its partials), and a caller has to know from the plan
         * whether a call can be captured: so also where the kernel chosen
         * needs no partials.  With the no-alloc entry point such a plan always
         * runs: its partials are at most 4.1 MiB of the scratch's 64. */
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(hs, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) return VKBLAS_ERR_INIT;
    }
    int partials = !direct && plan.split > 1 && (plan.path == VKBLAS_PATH_SKINNY || plan.path == VKBLAS_PATH_SPLITK ||
                                      plan.path == VKBLAS_PATH_TAIL);
    const size_t part_bytes =
        partials ? (((size_t)plan.split * (plan.path == VKBLAS_PATH_TAIL ? plan.tail_rows : M) * N * sizeof(float) +
                     255) & ~(size_t)255)
                 : 0;
    const int divided = partials && plan.path == VKBLAS_PATH_SPLITK && plan.tile == VKB_TILE_64Q;
    size_t ws_bytes = partials ? VKB_WS_HEADER + part_bytes * (divided ? 1 + VKB_WAVEK_NQ : 1) : 0;
    /* The planner's own K splits (split-K for few output tiles, the split
     * tail) only speed a call up: where their partials have no room (the
     * caller's scratch is smaller; a capturing stream declines the
     * workspace) the call runs the plan without a split instead of failing.
     * A caller's split (split_k > 1) and the decode kernels' splits keep
     * their plan and fail. */
    const int optional = split_k == 0 && (plan.path == VKBLAS_PATH_SPLITK || plan.path == VKBLAS_PATH_TAIL);
    prof_t pf;
    if (!ws_ext) prof_begin(&pf, hs);
    else memset(&pf, 0, sizeof(pf));
    ws_lease_t lease = {NULL, -1, 0, hs};
    void* ws = ws_ext;
    int room = 1;
    if (partials && ws_ext) room = ws_bytes <= ws_ext_bytes;
    if (partials && !ws_ext) {
        room = ws_acquire(hs, ws_bytes, &lease) == 0;
        if (!room) ws_release(&lease);
        ws = lease.ptr;
    }
    if (!room && optional && !divided &&
        vkblas_plan_gemm(ab_type, c_type, op_a, op_b, M, N, K, lda, ldb, ldc, batch, 1, aligned, &plan) ==
            VKBLAS_OK &&
        plan.split == 1) {
        if (g_trace) fprintf(stderr, "[vkblas] no room for the partials: plan without a split (%s)\n",
                             path_name(plan.path));
        partials = 0;
        ws_bytes = 0;
        room = 1;
        ws = NULL;
    }
    if (!room) {
        if (g_trace && ws_ext)
            fprintf(stderr, "[vkblas] partials of %zu bytes exceed the %zu-byte scratch buffer\n", ws_bytes,
                    ws_ext_bytes);
        prof_end(&pf, hs, "gemm", 0);
        return ws_ext ? VKBLAS_ERR_PARAM : VKBLAS_ERR_INIT;
    }

    float* part = partials ? (float*)((char*)ws + VKB_WS_HEADER) : NULL;
    if (plan.path == VKBLAS_PATH_SKINNY && !direct) {
        /* decode; with a K split over workgroups: fp32 partials, fixed-order reduce */
        rc = vkb_launch_skinny(ab, op_b == VKBLAS_OP_T, A, lda, B, ldb, C, ldc, ct, M, N, K, alpha, beta,
                               (int)scalar_mode, alpha_dev, beta_dev, epp, part, partials ? plan.split : 1, stream);
        if (rc == 0 && partials)
            rc = vkb_launch_splitk_reduce(part, (int64_t)M * N, plan.split, M, N, C, ldc, ct, alpha, beta,
                                          (int)scalar_mode, alpha_dev, beta_dev, epp, stream);
    } else {
        vkb_gemm_args a;
        memset(&a, 0, sizeof(a));
        a.A = A; a.B = B; a.C = C;
        a.lda = lda; a.ldb = ldb; a.ldc = ldc;
        a.stride_a = stride_a; a.stride_b = stride_b; a.stride_c = stride_c;
        a.M = M; a.N = N; a.K = K;
        a.batch = batch;
        a.split = 1;
        a.k_per_split = K;
        a.a_kmajor = op_a == VKBLAS_OP_N;
        a.b_kmajor = op_b == VKBLAS_OP_T;
        a.ab_type = ab;
        a.c_type = ct;
        a.alpha = alpha; a.beta = beta;
        a.scalar_mode = (int)scalar_mode;
        a.alpha_dev = alpha_dev; a.beta_dev = beta_dev;
        a.generic_only = g_generic_only;
        a.direct = direct ? 2 : g_force_tile < 0;   /* a forced tile keeps its own kernels */
        a.kernel_out = &kernel;
        a.epi = epp;
        if (plan.path == VKBLAS_PATH_TAIL) {
            /* rows [0, head) as tiles, rows [head, M) split-K into the
             * workspace and reduced into C with the epilogue; batch == 1.
             * The tail's pass 1 goes first: it writes only the workspace, so
             * a failure there or at the head's launch leaves C untouched and
             * the caller may forward the call; a failure after the head's
             * tiles were enqueued returns VKBLAS_ERR_PARTIAL. */
            const uint32_t head = M - plan.tail_rows;
            const size_t es_ab = ab == VKB_T_F32 ? 4 : 2, es_c = ct == VKB_T_F32 ? 4 : 2;
            a.M = head;
            vkb_gemm_args t = a;
            t.M = plan.tail_rows;
            t.A = (const char*)A + (size_t)head * (op_a == VKBLAS_OP_N ? (size_t)lda : 1) * es_ab;
            t.C = part;
            t.ldc = N;
            t.c_type = VKB_T_F32;
            t.split = plan.split;
            t.k_per_split = plan.k_per_split;
            t.stride_split = (int64_t)plan.tail_rows * N;
            t.alpha = 1.0f; t.beta = 0.0f;
            t.scalar_mode = VKB_SCALAR_HOST;
            t.alpha_dev = t.beta_dev = NULL;
            t.epi = NULL;
            int tail_kernel = 0;
            t.kernel_out = &tail_kernel;
            rc = vkb_launch_gemm(&t, plan.tile, stream);
            if (rc == 0) rc = vkb_launch_gemm(&a, plan.tile, stream);
            if (rc == 0) c_written = 1;
            vkb_epilogue_args tep;
            memset(&tep, 0, sizeof(tep));
            if (epp) {
                tep = *epp;
                if (tep.c_in) tep.c_in = (const char*)tep.c_in + (size_t)head * tep.ldc_in * es_c;
            }
            if (rc == 0)
                rc = vkb_launch_splitk_reduce(part, (int64_t)plan.tail_rows * N, plan.split,
                                              plan.tail_rows, N, (char*)C + (size_t)head * ldc * es_c, ldc, ct,
                                              alpha, beta, (int)scalar_mode, alpha_dev, beta_dev,
                                              epp ? &tep : NULL, stream);
        } else if (plan.path == VKBLAS_PATH_SPLITK) {
            a.C = part;
            if (divided) {
                a.qcnt = (uint32_t*)ws;
                a.qpart = (float*)((char*)part + part_bytes);
            }
            a.ldc = N;
            a.stride_c = 0;
            a.c_type = VKB_T_F32;
            a.split = plan.split;
            a.k_per_split = plan.k_per_split;
            a.stride_split = (int64_t)M * N;
            a.alpha = 1.0f; a.beta = 0.0f;
            a.scalar_mode = VKB_SCALAR_HOST;
            a.alpha_dev = a.beta_dev = NULL;
            a.epi = NULL;
            rc = vkb_launch_gemm(&a, plan.tile, stream);
            if (rc == 0)
                rc = vkb_launch_splitk_reduce(part, (int64_t)M * N, plan.split, M, N, C, ldc, ct,
                                              alpha, beta, (int)scalar_mode, alpha_dev, beta_dev, epp, stream);
        } else {
            rc = vkb_launch_gemm(&a, plan.tile, stream);
        }
    }
    ws_release(&lease);
    prof_end(&pf, hs, path_name(plan.path), rc == 0);
    if (rc != 0) {
        if (g_trace) fprintf(stderr, "[vkblas] launch failed: %s%s\n", hipGetErrorString((hipError_t)rc),
                             c_written ? " (after part of C was written)" : "");
        return c_written ? VKBLAS_ERR_PARTIAL : VKBLAS_ERR_INIT;
    }
    g_last_path = plan.path;
    g_last_kernel = kernel;
    return VKBLAS_OK;
}

vkblas_status_t vkblas_gemm_async(vkblas_dtype_t ab_type, vkblas_dtype_t c_type,
                                  vkblas_op_t op_a, vkblas_op_t op_b,
                                  uint32_t M, uint32_t N, uint32_t K,
                                  float alpha,
                                  const void* A, uint32_t lda,
                                  const void* B, uint32_t ldb,
                                  float beta,
                                  void* C, uint32_t ldc,
                                  uint32_t batch,
                                  int64_t stride_a, int64_t stride_b, int64_t stride_c,
                                  vkblas_scalar_mode_t scalar_mode, const void* alpha_dev,
                                  const void* beta_dev, uint32_t split_k, void* stream) {
    return gemm_impl(ab_type, c_type, op_a, op_b, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, batch, stride_a,
                     stride_b, stride_c, scalar_mode, alpha_dev, beta_dev, split_k, NULL, stream, NULL, 0);
}

vkblas_status_t vkblas_gemm_ex_async(vkblas_dtype_t ab_type, vkblas_dtype_t c_type,
                                     vkblas_op_t op_a, vkblas_op_t op_b,
                                     uint32_t M, uint32_t N, uint32_t K,
                                     float alpha,
                                     const void* A, uint32_t lda,
                                     const void* B, uint32_t ldb,
                                     float beta,
                                     void* C, uint32_t ldc,
                                     uint32_t batch,
                                     int64_t stride_a, int64_t stride_b, int64_t stride_c,
                                     vkblas_scalar_mode_t scalar_mode, const void* alpha_dev,
                                     const void* beta_dev, uint32_t split_k,
                                     const vkblas_epilogue_t* epilogue, void* stream) {
    return gemm_impl(ab_type, c_type, op_a, op_b, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, batch, stride_a,
                     stride_b, stride_c, scalar_mode, alpha_dev, beta_dev, split_k, epilogue, stream, NULL, 0);
}

vkblas_status_t vkb_gemm_with_scratch(vkblas_dtype_t ab_type, vkblas_dtype_t c_type, vkblas_op_t op_a,
                                      vkblas_op_t op_b, uint32_t M, uint32_t N, uint32_t K, float alpha,
                                      const void* A, uint32_t lda, const void* B, uint32_t ldb, float beta,
                                      void* C, uint32_t ldc, uint32_t batch, int64_t stride_a, int64_t stride_b,
                                      int64_t stride_c, vkblas_scalar_mode_t scalar_mode, const void* alpha_dev,
                                      const void* beta_dev, uint32_t split_k, void* stream, void* scratch,
                                      size_t scratch_bytes) {
    if (!scratch || scratch_bytes == 0) return VKBLAS_ERR_PARAM;
    return gemm_impl(ab_type, c_type, op_a, op_b, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, batch, stride_a,
                     stride_b, stride_c, scalar_mode, alpha_dev, beta_dev, split_k, NULL, stream, scratch,
                     scratch_bytes);
}

vkblas_status_t vkblas_gemm_batched_async(vkblas_dtype_t ab_type, vkblas_dtype_t c_type,
                                          vkblas_op_t op_a, vkblas_op_t op_b,
                                          uint32_t M, uint32_t N, uint32_t K,
                                          float alpha,
                                          const void* const* A, uint32_t lda,
                                          const void* const* B, uint32_t ldb,
                                          float beta,
                                          void* const* C, uint32_t ldc,
                                          uint32_t batch,
                                          vkblas_scalar_mode_t scalar_mode, const void* alpha_dev,
                                          const void* beta_dev, void* stream) {
    if (!A || !B || !C) return VKBLAS_ERR_PARAM;
    if (scalar_mode != VKBLAS_SCALAR_HOST && (!alpha_dev || !beta_dev)) return VKBLAS_ERR_PARAM;
    if (scalar_mode != VKBLAS_SCALAR_HOST && scalar_mode != VKBLAS_SCALAR_DEV_F32 &&
        scalar_mode != VKBLAS_SCALAR_DEV_F16)
        return VKBLAS_ERR_PARAM;
    /* split_k = 1 and aligned = 0: a tile path (no split, no skinny) */
    vkblas_plan_t plan;
    vkblas_status_t st = vkblas_plan_gemm(ab_type, c_type, op_a, op_b, M, N, K, lda, ldb, ldc, batch, 1, 0, &plan);
    if (st != VKBLAS_OK) return st;
    if (plan.path == VKBLAS_PATH_SPLITK || plan.path == VKBLAS_PATH_SKINNY) return VKBLAS_ERR_PARAM;
    if (!ensure_init()) return VKBLAS_ERR_INIT;
    const int ab = kernel_type(ab_type);
    const int ct = kernel_type(c_type);
    if (g_trace)
        fprintf(stderr, "[vkblas] gemm batched %s%s %s->%s M=%u N=%u K=%u lda=%u ldb=%u ldc=%u batch=%u path=%s\n",
                op_a ? "T" : "N", op_b ? "T" : "N", type_name(ab), type_name(ct), M, N, K, lda, ldb, ldc, batch,
                path_name(plan.path));
    vkb_gemm_args a;
    memset(&a, 0, sizeof(a));
    a.A = (const void*)A; a.B = (const void*)B; a.C = (void*)C;
    a.lda = lda; a.ldb = ldb; a.ldc = ldc;
    a.M = M; a.N = N; a.K = K;
    a.batch = batch;
    a.split = 1;
    a.k_per_split = K;
    a.a_kmajor = op_a == VKBLAS_OP_N;
    a.b_kmajor = op_b == VKBLAS_OP_T;
    a.ab_type = ab;
    a.c_type = ct;
    a.alpha = alpha; a.beta = beta;
    a.scalar_mode = (int)scalar_mode;
    a.alpha_dev = alpha_dev; a.beta_dev = beta_dev;
    a.ptr_array = 1;
    int kernel = VKBLAS_KERNEL_NONE;
    a.kernel_out = &kernel;
    prof_t pf;
    prof_begin(&pf, (hipStream_t)stream);
    const int rc = vkb_launch_gemm(&a, plan.tile, stream);
    prof_end(&pf, (hipStream_t)stream, "batched", rc == 0);
    if (rc != 0) {
        if (g_trace) fprintf(stderr, "[vkblas] launch failed: %s\n", hipGetErrorString((hipError_t)rc));
        return VKBLAS_ERR_INIT;
    }
    g_last_path = plan.path;
    g_last_kernel = kernel;
    return VKBLAS_OK;
}

int vkblas_last_path(void) { return g_last_path; }

int vkblas_last_kernel(void) { return g_last_kernel; }

vkblas_status_t vkblas_set_override(int tile, int generic) {
    pthread_once(&g_once, init_once);
    if (tile < -1 || tile >= VKB_TILE_COUNT) return VKBLAS_ERR_PARAM;
    __atomic_store_n(&g_force_tile, tile, __ATOMIC_RELAXED);
    __atomic_store_n(&g_generic_only, generic ? 1 : 0, __ATOMIC_RELAXED);
    return VKBLAS_OK;
}

const char* vkblas_version(void) { return VKBLAS_VERSION_STRING; }

/* ------------------------------------------------------ reference C API */

/* The reference's engine calls return once C is written (src/vkblas.c:963
 * waits for its queue); these do the same on the null stream they launch on. */
static vkblas_status_t finish_sync(vkblas_status_t st) {
    if (st == VKBLAS_OK && hipStreamSynchronize(NULL) != hipSuccess) return VKBLAS_ERR_INIT;
    return st;
}

vkblas_status_t vkblas_gemm_f32(vkblas_op_t op_a, vkblas_op_t op_b, uint32_t M, uint32_t N, uint32_t K,
                                float alpha, const void* A, uint32_t lda, const void* B, uint32_t ldb,
                                float beta, void* C, uint32_t ldc, uint32_t batch,
                                int64_t stride_a, int64_t stride_b, int64_t stride_c) {
    return finish_sync(vkblas_gemm_async(VKBLAS_DT_F32, VKBLAS_DT_F32, op_a, op_b, M, N, K, alpha, A, lda, B, ldb,
                                         beta, C, ldc, batch, stride_a, stride_b, stride_c, VKBLAS_SCALAR_HOST, NULL,
                                         NULL, 0, NULL));
}

vkblas_status_t vkblas_gemm_f16(vkblas_op_t op_a, vkblas_op_t op_b, uint32_t M, uint32_t N, uint32_t K,
                                float alpha, const void* A, uint32_t lda, const void* B, uint32_t ldb,
                                float beta, void* C, uint32_t ldc, uint32_t batch,
                                int64_t stride_a, int64_t stride_b, int64_t stride_c) {
    return finish_sync(vkblas_gemm_async(VKBLAS_DT_F16, VKBLAS_DT_F16, op_a, op_b, M, N, K, alpha, A, lda, B, ldb,
                                         beta, C, ldc, batch, stride_a, stride_b, stride_c, VKBLAS_SCALAR_HOST, NULL,
                                         NULL, 0, NULL));
}

vkblas_status_t vkblas_gemm_bf16(vkblas_op_t op_a, vkblas_op_t op_b, uint32_t M, uint32_t N, uint32_t K,
                                 float alpha, const void* A, uint32_t lda, const void* B, uint32_t ldb,
                                 float beta, void* C, uint32_t ldc, uint32_t batch,
                                 int64_t stride_a, int64_t stride_b, int64_t stride_c) {
    return finish_sync(vkblas_gemm_async(VKBLAS_DT_BF16, VKBLAS_DT_BF16, op_a, op_b, M, N, K, alpha, A, lda, B,
                                         ldb, beta, C, ldc, batch, stride_a, stride_b, stride_c, VKBLAS_SCALAR_HOST,
                                         NULL, NULL, 0, NULL));
}

/* The reference's second bf16 entry (src/vkblas.c:3448-3512) differs from the
 * first only in how it avoids a transpose pass of its own; every layout is
 * read natively here, so both entries are the same call. */
vkblas_status_t vkblas_gemm_bf16_hipblas(vkblas_op_t op_a, vkblas_op_t op_b, uint32_t M, uint32_t N,
                                         uint32_t K, float alpha, const void* A, uint32_t lda, const void* B,
                                         uint32_t ldb, float beta, void* C, uint32_t ldc, uint32_t batch,
                                         int64_t stride_a, int64_t stride_b, int64_t stride_c) {
    return vkblas_gemm_bf16(op_a, op_b, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, batch, stride_a,
                            stride_b, stride_c);
}

int vkblas_gemm_c64(vkblas_op_t op_a, vkblas_op_t op_b, uint32_t M, uint32_t N, uint32_t K, float alpha_r,
                    float alpha_i, const void* A, uint32_t lda, const void* B, uint32_t ldb, float beta_r,
                    float beta_i, void* C, uint32_t ldc, uint32_t batch, int64_t stride_a, int64_t stride_b,
                    int64_t stride_c) {
    (void)op_a; (void)op_b; (void)M; (void)N; (void)K; (void)alpha_r; (void)alpha_i; (void)A; (void)lda;
    (void)B; (void)ldb; (void)beta_r; (void)beta_i; (void)C; (void)ldc; (void)batch; (void)stride_a;
    (void)stride_b; (void)stride_c;
    return VKBLAS_ERR_INIT;
}

int vkblas_gemm_f64(vkblas_op_t op_a, vkblas_op_t op_b, uint32_t M, uint32_t N, uint32_t K, double alpha,
                    const void* A, uint32_t lda, const void* B, uint32_t ldb, double beta, void* C,
                    uint32_t ldc, uint32_t batch, int64_t stride_a, int64_t stride_b, int64_t stride_c) {
    (void)op_a; (void)op_b; (void)M; (void)N; (void)K; (void)alpha; (void)A; (void)lda; (void)B; (void)ldb;
    (void)beta; (void)C; (void)ldc; (void)batch; (void)stride_a; (void)stride_b; (void)stride_c;
    return VKBLAS_ERR_INIT;
}

int vkblas_gemm_z64(vkblas_op_t op_a, vkblas_op_t op_b, uint32_t M, uint32_t N, uint32_t K, double alpha_r,
                    double alpha_i, const void* A, uint32_t lda, const void* B, uint32_t ldb, double beta_r,
                    double beta_i, void* C, uint32_t ldc, uint32_t batch, int64_t stride_a, int64_t stride_b,
                    int64_t stride_c) {
    (void)op_a; (void)op_b; (void)M; (void)N; (void)K; (void)alpha_r; (void)alpha_i; (void)A; (void)lda;
    (void)B; (void)ldb; (void)beta_r; (void)beta_i; (void)C; (void)ldc; (void)batch; (void)stride_a;
    (void)stride_b; (void)stride_c;
    return VKBLAS_ERR_INIT;
}

void vkblas_cache_invalidate_base(const void* ptr) { (void)ptr; }

// tlg_gemm.hip -- host side of the GEMMs behind mm / mm_bt / mm_atb: shapes,
// plans and launches of the tile kernels (tlg_tile.h, tlg_tiles.hip), grouped
// and expert-batched launches, the fills and the measurement probes.
#include "tlg_tile.h"
#include <mutex>
#include <set>
#include <string>
#include <stdio.h>
#include <string.h>

__global__ void k_split_reduce(const float *__restrict__ ws, float *__restrict__ C, int Mo, int No,
                               int ldc, int splits, int beta)
{
    const size_t n = (size_t)Mo * No;
    const size_t per = 512;
    for (size_t e0 = (size_t)blockIdx.x * per; e0 < n; e0 += (size_t)gridDim.x * per)
        reduce_range(ws, C, No, ldc, splits, beta, e0, e0 + per < n ? e0 + per : n, n);
}

__global__ void k_zero(float *__restrict__ p, size_t n)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = 0.f;
}

int tlg_zero_launch(float *dst, size_t n, hipStream_t st)
{
    if (n == 0) return TLG_OK;
    if (!dst) return tlg_fail(TLG_EINVAL, "tlg_dev_zero: NULL destination");
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_zero, dim3((unsigned)blocks), dim3(256), 0, st, dst, n);
    TLG_HIP(hipGetLastError());
    return TLG_OK;
}

// ---------------------------------------------------------------- launch --
struct TileCfg { int bm, bn, bk, wgm, wk, nr, nw, sch; };
#define TLG_ROW(i, bm, bn, bk, wgm, wk, nr, nw, sch) {bm, bn, bk, wgm, wk, nr, nw, sch},
static const TileCfg kCfgs[] = {TLG_TILES(TLG_ROW)};
#undef TLG_ROW
static const int kNumCfgs = (int)(sizeof(kCfgs) / sizeof(kCfgs[0]));

// A tile's type as rocprofv3 prints it.
static int tile_name(const TileCfg &c, char *buf, int len)
{
    if (c.sch)
        return snprintf(buf, (size_t)len, "Sched<Tile<%d, %d, %d, %d, %d, %d, %d>, %d>", c.bm, c.bn, c.bk, c.wgm,
                        c.wk, c.nr, c.nw, c.sch);
    return snprintf(buf, (size_t)len, "Tile<%d, %d, %d, %d, %d, %d, %d>", c.bm, c.bn, c.bk, c.wgm, c.wk, c.nr,
                    c.nw);
}

static inline bool al16(const void *p) { return ((uintptr_t)p & 15u) == 0; }
static inline int cdiv(int a, int b) { return (a + b - 1) / b; }

#define TLG_WHOLE_TILES 240           // 64x64 tiles of an output whose reduction is never split
struct GemmPlan { int ci; int tiles_n, tiles, splits, rps; };

// Forced choice for tuning sweeps (tlg_tune_force); -1 = automatic.
static int g_force_cfg = -1, g_force_splits = 0;

static GemmPlan make_plan(int ci, int Mo, int No, int R, int splits, size_t ws_floats)
{
    const TileCfg &c = kCfgs[ci];
    GemmPlan p;
    p.ci = ci;
    p.tiles_n = cdiv(No, c.bn);
    p.tiles = cdiv(Mo, c.bm) * p.tiles_n;
    if (splits < 1) splits = 1;
    int rps = cdiv(cdiv(R, splits), c.bk) * c.bk;
    splits = cdiv(R, rps);
    if (splits > 1 && (size_t)splits * Mo * No > ws_floats) {
        splits = 1;
        rps = cdiv(R, c.bk) * c.bk;
    }
    p.splits = splits;
    p.rps = rps;
    return p;
}

// Automatic choice: the largest of 128x128, 64x64 and 32x32 tiles that gives
// the 256 CUs about 160 work items, splitting the reduction as far as every
// split keeps >= 512 steps (small outputs with long reductions, i.e. mm_atb's
// dW), 256 on 32x32 tiles (mm_atb (1001, 77, 333) 11.3 us in 3 splits, 12.9
// whole).  Measured on one box, other shapes against the rule's: mm
// (8192, 384, 2048) 128x128 85 us, 64x64 97, 128x64 121; mm (4096, 768, 256)
// 64x64 17, 32x32 23; mm (2048, 512, 128) 32x32 7.4, 64x64 11.4; mm_atb
// (8192, 1024, 384) 7 splits of 128x128 52 (8 splits 47), 64x64 52.  64x64 tiles
// take 64-step stages (8 waves, a quarter of each stage per wave) from 512 steps
// on and 16-step stages below: 16.9 against 19.4 us at 768 steps, 19 against 11
// at 128.
//
// Outputs of 240 64x64 tiles and more run whole: a split's partials lie in the
// one workspace, which calls that overlap on two streams would both write, and
// outputs of that size are promised not to (@MEASURED@).
static GemmPlan plan_gemm(int Mo, int No, int R, size_t ws_floats)
{
    if (g_force_cfg >= 0 && g_force_cfg < kNumCfgs)
        return make_plan(g_force_cfg, Mo, No, R, g_force_splits, ws_floats);
    const int enough = 160;
    const int order[] = {9, R >= 512 ? 8 : 3, 15};
    const bool whole = (long long)cdiv(Mo, 64) * cdiv(No, 64) >= TLG_WHOLE_TILES;
    int ci = 15, splits = 1;
    for (int k = 0; k < 3; k++) {
        const TileCfg &c = kCfgs[order[k]];
        const long long tiles = (long long)cdiv(Mo, c.bm) * cdiv(No, c.bn);
        ci = order[k];
        splits = tiles >= enough ? 1 : cdiv(enough, (int)tiles);
        const int maxs = R / (k == 2 ? 256 : 512);
        if (splits > maxs) splits = maxs > 1 ? maxs : 1;
        if (whole) splits = 1;
        if (tiles * splits >= enough) break;
    }
    return make_plan(ci, Mo, No, R, splits, ws_floats);
}

// Name of the kernel instance a device-pointer call with aligned operands
// launches, as rocprofv3 prints it, and its split count.
int tlg_describe(TlgKind kind, int Mo, int No, int R, char *buf, int len, int *splits)
{
    if (tlg_ensure_init()) return TLG_ESTATE;
    if (Mo <= 0 || No <= 0 || R <= 0) {
        snprintf(buf, (size_t)len, "%s", R == 0 ? "k_zero" : "none");
        if (splits) *splits = 0;
        return TLG_OK;
    }
    if (tlg_gemv_fits(kind, Mo)) {
        tlg_gemv_describe(kind, Mo, No, R, buf, len);
        if (splits) *splits = 1;
        return TLG_OK;
    }
    const GemmPlan p = plan_gemm(Mo, No, R, g_tlg.ws_floats);
    const TileCfg &c = kCfgs[p.ci];
    const int la = (kind == TLG_TN) ? OC : RC;
    const int lb = (kind == TLG_NT) ? RC : OC;
    const bool vec = (la == RC ? (R % 4 == 0) : (Mo % 4 == 0)) && (lb == RC ? (R % 4 == 0) : (No % 4 == 0));
    char tile[96];
    TileCfg t = c;
    t.sch = 5;                                   // single calls
    tile_name(t, tile, (int)sizeof tile);
    snprintf(buf, (size_t)len, "k_gemm<%s, %d, %d, %s>", tile, la, lb, vec ? "true" : "false");
    if (splits) *splits = p.splits;
    return TLG_OK;
}

extern "C" int tlg_tune_force(int cfg, int splits)
{
    // single-call launches instantiate configs 0-15 (16+ are grouped-only shapes)
    if (cfg >= 16) return tlg_fail(TLG_EINVAL, "tlg_tune_force: config %d of 16", cfg);
    g_force_cfg = cfg;
    g_force_splits = splits;
    return TLG_OK;
}

static int launch_reduce(const float *ws, float *C, int Mo, int No, int ldc, int splits, int beta,
                         hipStream_t st)
{
    const size_t n = (size_t)Mo * No;
    size_t blocks = (n + 511) / 512;
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(k_split_reduce, dim3((unsigned)blocks), dim3(128), 0, st, ws, C, Mo, No, ldc,
                       splits, beta);
    TLG_HIP(hipGetLastError());
    return TLG_OK;
}

// One GEMM on `st` whose split partials (if any) go to ws[0, ws_floats).
// Allocates nothing: the caller owns ws (the library's workspace, or the
// no-allocation scratch below).
static int gemm_launch_ws(TlgKind kind, const float *A, const float *B, float *C, int Mo, int No, int R,
                          int lda, int ldb, int ldc, int beta, float *ws, size_t ws_floats, hipStream_t st)
{
    if (tlg_gemv_fits(kind, Mo)) return tlg_gemv_launch(kind, A, B, C, Mo, No, R, lda, ldb, ldc, beta, st);

    const int la = (kind == TLG_TN) ? OC : RC;
    const int lb = (kind == TLG_NT) ? RC : OC;
    // float4 staging needs 16-byte aligned operands whose contiguous extent
    // and leading dimension are multiples of 4.
    const bool vec = al16(A) && al16(B) && (lda % 4 == 0) && (ldb % 4 == 0) &&
                     (la == RC ? (R % 4 == 0) : (Mo % 4 == 0)) &&
                     (lb == RC ? (R % 4 == 0) : (No % 4 == 0));
    // the split count the library workspace would give, reduced to what ws holds
    GemmPlan pl = plan_gemm(Mo, No, R, TLG_WS_FLOATS);
    if (pl.splits > 1 && (size_t)pl.splits * Mo * No > ws_floats)
        pl = make_plan(pl.ci, Mo, No, R, (int)(ws_floats / ((size_t)Mo * No)), ws_floats);

    GemmArgs a;
    a.A = A; a.B = B; a.C = C;
    a.Mo = Mo; a.No = No; a.R = R;
    a.lda = lda; a.ldb = ldb; a.ldc = ldc;
    a.beta = beta;
    a.tiles_n = pl.tiles_n; a.tiles = pl.tiles;
    a.splits = pl.splits; a.rps = pl.rps;
    a.ws = ws;
    const int grid = pl.tiles * pl.splits;
    const int ci = tile_canon(pl.ci);
    if (!tlg_single_part0(ci, kind, vec, a, grid, st) && !tlg_single_part1(ci, kind, vec, a, grid, st))
        return tlg_fail(TLG_EINVAL, "GEMM: no kernel for tile configuration %d", pl.ci);
    TLG_HIP(hipGetLastError());
    if (pl.splits > 1) return launch_reduce(ws, C, Mo, No, ldc, pl.splits, beta, st);
    return TLG_OK;
}

int tlg_gemm_launch(TlgKind kind, const float *A, const float *B, float *C,
                    int Mo, int No, int R, int lda, int ldb, int ldc, int beta,
                    hipStream_t st)
{
    if (Mo < 0 || No < 0 || R < 0) return tlg_fail(TLG_EINVAL, "negative GEMM dimension");
    if (Mo == 0 || No == 0) return TLG_OK;
    if (!C) return tlg_fail(TLG_EINVAL, "NULL output pointer");
    if (R == 0) {
        // Empty reduction: mm clears its rows (tinylm.c:461), the accumulating
        // forms add nothing.
        if (beta) return TLG_OK;
        if (ldc != No) return tlg_fail(TLG_EINVAL, "strided empty-reduction clear");
        return tlg_zero_launch(C, (size_t)Mo * No, st);
    }
    if (!A || !B) return tlg_fail(TLG_EINVAL, "NULL input pointer");
    int rc = tlg_ensure_init();
    if (rc) return rc;
    // a single-problem launch must not overtake partials a grouped launch
    // left for its successor
    rc = tlg_group_flush_launch(st);
    if (rc) return rc;
    return gemm_launch_ws(kind, A, B, C, Mo, No, R, lda, ldb, ldc, beta, g_tlg.ws, g_tlg.ws_floats, st);
}

// --------------------------------------------- mm_atb without allocation --
// Callers that must not allocate device memory (code under HIP graph
// capture, serving loops, harnesses that forbid hipMalloc) get mm_atb with
// its split partials in this fixed array instead of the library workspace.
// Each GPU the library runs on holds its own copy until the process ends.
// Host code never passes `scratch` itself to a kernel (on the host the name
// is only a stand-in); it uses the device address hipGetSymbolAddress gives
// for the current device, looked up once per device.
#define TLG_SCRATCH_FLOATS ((size_t)4 << 20)          // 16 MiB
static __device__ __align__(256) float scratch[TLG_SCRATCH_FLOATS];

#define TLG_MAX_DEVICES 64
static float *g_scratch_dev[TLG_MAX_DEVICES];
static std::mutex g_scratch_mu;

static int scratch_for_current_device(float **out)
{
    int dev = -1;
    TLG_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= TLG_MAX_DEVICES) return tlg_fail(TLG_EINVAL, "no-alloc scratch: device %d", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void *p = nullptr;
        TLG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return tlg_fail(TLG_EHIP, "no-alloc scratch: no device address on device %d", dev);
        g_scratch_dev[dev] = (float *)p;
    }
    *out = g_scratch_dev[dev];
    return TLG_OK;
}

extern "C" int tlg_dev_sgemm_tn_acc_noalloc(float *dW, const float *X, const float *dY, int M, int K, int N,
                                            void *stream)
{
    if (M < 0 || K < 0 || N < 0) return tlg_fail(TLG_EINVAL, "negative dimension");
    if ((size_t)K * N > TLG_SCRATCH_FLOATS / 2)
        return tlg_fail(TLG_EINVAL,
                        "tlg_dev_sgemm_tn_acc_noalloc: dW of %d x %d floats exceeds the no-allocation limit of "
                        "%zu floats (half the %zu-float scratch)",
                        K, N, TLG_SCRATCH_FLOATS / 2, TLG_SCRATCH_FLOATS);
    if (K == 0 || N == 0 || M == 0) return TLG_OK;         // mm_atb adds nothing
    if (!dW || !X || !dY) return tlg_fail(TLG_EINVAL, "NULL pointer");
    hipStream_t st = (hipStream_t)stream;
    float *ws = nullptr;
    int rc = scratch_for_current_device(&ws);
    if (rc) return rc;
    // partials a grouped launch left for its successor must land first
    if (g_tlg.initialised) {
        rc = tlg_group_flush_launch(st);
        if (rc) return rc;
    }
    return gemm_launch_ws(TLG_TN, X, dY, dW, K, N, M, K, N, N, 1, ws, TLG_SCRATCH_FLOATS, st);
}

// ------------------------------------------------------- grouped launch --
// Host side of k_group.  Split partials of a grouped launch live in one half
// of the workspace and are reduced by the next grouped launch (or a flush);
// the halves alternate so a launch never overwrites partials still pending.
static Prob g_pending[TLG_MAXPROB];
static int g_npending = 0;
static hipStream_t g_pending_st = nullptr;     // the stream their partials were written on
#include <stdlib.h>
static int g_ws_half = 0;
static int flush_foreign(hipStream_t st);

// Tile shape of a grouped launch (all problems of a group share it): the
// first row of kAuto whose shape gives the launch enough work items.  Measured
// over the nano, m3 and m8 models' launches (replayed, us; the row's shape
// against the next one's; before operands were scaled, which took 1 to 2 %):
//   128x128  m8 FFN backward 186 / 203 (128x64), m3 60 / 73; m8 W2 48 / 50.
//            Launches without an mm_atb need whole rounds of 256 items (m8
//            Q | K | V: 320 items, 35 against 32 on 64x64 tiles); short
//            reductions run it in the compiler's order with streaming stores
//            (m3 logits 27 / 30).
//   128x64   m3 head backward 62 / 67 (64x64)
//   64x64    m3 Q | K | V 10.5 / 11.3, its backward 21.7 / 22.3
//   64x64 of 8 waves, each 64x32 of a quarter of a 64-step stage: one item per
//            CU, so the waves come from the reduction (m3 W2 16.1 / 18.8)
//   64x32, 32x32 likewise (nano head backward 23 / 28 / 29, W2 7.0 on 32x32)
// mm_atb splits aim for about 512 reduction steps.  TLG_GROUP_CANDS (or
// tlg_tune_group_policy) puts a list of its own in the rows' place,
// TLG_GROUP_MINWAVES scales the rows' items (3 = as they stand), tlg_tune_group
// pins one shape.
static const struct { int cfg, items; } kAuto[] = {{33, 160}, {34, 240}, {35, 320}, {41, 160}, {21, 128}, {15, 0}};
static int g_group_cfg = -1;
static int g_group_rt = 0;               // split target pinned for the next launches (tlg_tune_group_split)
static double g_min_waves = 3.0;
static int g_cand[4] = {-1, -1, -1, -1};  // candidates put in place of kAuto
static int g_rtarget = 512;
static int g_erps = 1024;                // expert TN slice (TLG_EXPERT_RPS)
static int g_expert_cfg = -1;            // expert tile shape pinned (TLG_EXPERT_CFG: a key of TLG_EXPERTS)
static int g_expert_sched = -1;          // expert tiles: 0, 1 plain stores, 2 streaming ones, -1 automatic: 2 for launches of
                                         // dense rows (the training step's fused SwiGLU: 2.003 -> 1.995 ms), 1 for
                                         // MoE launches (streaming measured 0.232 -> 0.237 ms per kept pair: the
                                         // next launch reads their g, u, a, y right away) (TLG_EXPERT_SCHED)
static int g_group_last = 3;          // shape of the most recent grouped launch
static const char *g_group_last_name = nullptr;   // set when that launch was a GEMV group

static bool is_group_shape(int cfg) { return cfg >= 0 && cfg < kNumCfgs && tile_grouped(cfg); }

static bool is_expert_shape(int key)
{
#define TLG_ROW(k, bm, bn, bk, wgm, wk, nw) if (key == k) return true;
    TLG_EXPERTS(TLG_ROW)
#undef TLG_ROW
    return false;
}

static void group_env(void)
{
    static int done = 0;
    if (done) return;
    done = 1;
    const char *e = getenv("TLG_GROUP_MINWAVES");
    if (e && atof(e) > 0) g_min_waves = atof(e);
    e = getenv("TLG_GROUP_CFG");
    if (e && *e && is_group_shape(atoi(e))) g_group_cfg = atoi(e);
    e = getenv("TLG_GROUP_CANDS");            // e.g. "3,13,15"
    if (e && *e) {
        int k = 0;
        for (const char *q = e; *q && k < 3; ) {
            if (is_group_shape(atoi(q))) g_cand[k++] = atoi(q);
            while (*q && *q != ',') q++;
            if (*q == ',') q++;
        }
        g_cand[k] = -1;
    }
    e = getenv("TLG_EXPERT_RPS");
    if (e && atoi(e) >= 64) g_erps = atoi(e);
    e = getenv("TLG_EXPERT_CFG");
    if (e && is_expert_shape(atoi(e)))
        g_expert_cfg = atoi(e);
    if ((e = getenv("TLG_EXPERT_SCHED")) && atoi(e) >= -1 && atoi(e) <= 2) g_expert_sched = atoi(e);
    e = getenv("TLG_GROUP_RTARGET");
    if (e && atoi(e) >= 64) g_rtarget = atoi(e);
}

// The item-count header of a launch's arguments (GroupArgs.items, devcount).
static const GroupArgs &group_seal(const GroupArgs &a)
{
    static GroupArgs b;
    b = a;
    b.devcount = 0;
    for (int p = 0; p < TLG_MAXPROB; p++) {
        b.items[p] = p < a.nprob ? a.p[p].items : 0;
        if (p < a.nprob && a.p[p].nexp && a.p[p].kind != PK_RED) b.devcount |= 1u << p;
    }
    return b;
}

static void launch_group(int ci, const GroupArgs &a, int grid, hipStream_t st)
{
    const GroupArgs &b = group_seal(a);
    const int kernel = tile_canon(ci);
#define TLG_TRY(k) if (!tlg_group_part##k(kernel, b, grid, st))
    TLG_TILE_PARTS(TLG_TRY) {}
#undef TLG_TRY
    g_group_last = ci;
    g_group_last_name = nullptr;
}

extern "C" int tlg_tune_group_policy(const int *cands, int ncands, double min_waves, int rtarget)
{
    group_env();
    if (ncands < 0 || ncands > 3 || (ncands > 0 && !cands) || min_waves < 0 || (rtarget && rtarget < 64))
        return tlg_fail(TLG_EINVAL, "tlg_tune_group_policy: bad arguments");
    const bool automatic = ncands == 1 && cands[0] == -1;
    for (int k = 0; k < ncands && !automatic; k++)
        if (!is_group_shape(cands[k]))
            return tlg_fail(TLG_EINVAL, "tlg_tune_group_policy: config %d", cands[k]);
    if (ncands > 0) {
        for (int k = 0; k < ncands; k++) g_cand[k] = cands[k];
        g_cand[ncands] = -1;
    }
    if (min_waves > 0) g_min_waves = min_waves;
    if (rtarget) g_rtarget = rtarget;
    return TLG_OK;
}

extern "C" int tlg_tune_expert(int cfg, int sched)
{
    group_env();
    if ((cfg != -1 && !is_expert_shape(cfg)) || sched < -1 || sched > 2)
        return tlg_fail(TLG_EINVAL, "tlg_tune_expert: config %d, order %d", cfg, sched);
    g_expert_cfg = cfg;
    g_expert_sched = sched;
    return TLG_OK;
}

extern "C" int tlg_tune_group(int cfg)
{
    if (cfg != -1 && !is_group_shape(cfg))
        return tlg_fail(TLG_EINVAL, "tlg_tune_group: config %d", cfg);
    g_group_cfg = cfg;
    return TLG_OK;
}

extern "C" int tlg_tune_group_split(int rtarget)
{
    if (rtarget != 0 && rtarget < 64)
        return tlg_fail(TLG_EINVAL, "tlg_tune_group_split: target %d (0 or >= 64)", rtarget);
    g_group_rt = rtarget;
    return TLG_OK;
}

// Callers keep the pointer past later launches, so each name is stored once
// (at most one string per kernel instance) and never rewritten.
const char *tlg_group_kernel_name(void)
{
    static std::set<std::string> names;
    static std::mutex mu;
    char name[128], tile[96];
    if (g_group_last_name) {
        snprintf(name, sizeof name, "%s", g_group_last_name);
    } else {
        tile_name(kCfgs[g_group_last], tile, (int)sizeof tile);
        snprintf(name, sizeof name, "k_group<%s >", tile);
    }
    std::lock_guard<std::mutex> lk(mu);
    return names.insert(name).first->c_str();
}

// Grid for the XCD-sliced mapping of group_item: 8 x the largest per-XCD
// share.
static int group_grid(const GroupArgs &a)
{
    int most = 0;
    for (int x = 0; x < 8; x++) {
        int t = 0;
        for (int p = 0; p < a.nprob; p++) {
            const int n = a.p[p].items;
            t += ((x + 1) * n >> 3) - (x * n >> 3);
        }
        if (t > most) most = t;
    }
    return 8 * most;
}

static int add_reductions(GroupArgs &a)
{
    for (int k = 0; k < g_npending; k++) {
        Prob r = g_pending[k];
        if (r.kind == PK_COLSUM) {
            r.items = cdiv(r.No / 4, TLG_COLSUM_CH);
        } else {
            r.kind = PK_RED;
            r.items = (int)(((size_t)r.Mo * r.No + TLG_RED_CHUNK - 1) / TLG_RED_CHUNK);
        }
        a.p[a.nprob++] = r;
    }
    g_npending = 0;
    return TLG_OK;
}

int tlg_group_pending(void);     // (below: the queued reductions and the held expert ones)

// Queue C[0, No) (beta ? += : =) sum over z of part[z][0, No) (z < splits,
// No % 4 == 0, 16-byte aligned rows) to ride along in the next grouped or
// expert launch (or tlg_dev_gemm_flush) on the stream.  A reduction still
// queued on the same partials, or a full queue, is flushed first, so `part`
// may be rewritten by the caller's next kernel only after this call.
int tlg_defer_colsum(const float *part, float *C, int splits, int No, int beta, hipStream_t st)
{
    int rc = TLG_OK;
    bool busy = g_npending >= TLG_MAXPROB / 2 - 1;
    for (int k = 0; k < g_npending && !busy; k++) busy = g_pending[k].ws == part;
    if (busy) {
        rc = tlg_group_flush_launch(st);
        if (rc) return rc;
    }
    rc = flush_foreign(st);
    if (rc) return rc;
    g_pending_st = st;
    Prob &r = g_pending[g_npending++];
    memset(&r, 0, sizeof r);
    r.kind = PK_COLSUM;
    r.C = C;
    r.ws = part;
    r.Mo = 1;
    r.No = No;
    r.ldc = No;
    r.beta = beta ? 1 : 0;
    r.splits = splits;
    return TLG_OK;
}

static int group_flush_dense(hipStream_t st)
{
    if (g_npending == 0) return TLG_OK;
    GroupArgs a;
    a.nprob = 0;
    a.rows1 = 0;
    add_reductions(a);
    launch_group(3, a, group_grid(a), st);
    TLG_HIP(hipGetLastError());
    return TLG_OK;
}

static int ecarry_flush(hipStream_t st);

static int ecarry_flush_with_pending(hipStream_t st, bool *done);

int tlg_group_flush_launch(hipStream_t st)
{
    int rc = flush_foreign(st);
    if (rc) return rc;
    bool done = false;
    if ((rc = ecarry_flush_with_pending(st, &done)) || done) return rc;
    rc = ecarry_flush(st);
    return rc ? rc : group_flush_dense(st);
}


// [lo, hi) byte range touched by a row-major operand of `rows` x `cols`
// with leading dimension ld.
static void span(const void *p, int rows, int cols, int ld, const char **lo, const char **hi)
{
    *lo = (const char *)p;
    *hi = *lo + ((size_t)(rows - 1) * ld + cols) * sizeof(float);
}
static bool overlap(const char *a0, const char *a1, const char *b0, const char *b1)
{
    return a0 < b1 && b0 < a1;
}

// Split problem P's reduction so one item runs about `rtarget` steps; partials
// go to ws (bounded by ws_cap floats).
static void plan_split(Prob &P, int R, int rtarget, float *ws, size_t &ws_used, size_t ws_cap)
{
    P.splits = 1;
    P.rps = R;
    if (P.kind != PK_TN || R <= rtarget + rtarget / 2) return;
    int sp = cdiv(R, rtarget);
    if (sp > 32) sp = 32;
    const int rps = cdiv(cdiv(R, sp), 64) * 64;      // a multiple of every group BK
    sp = cdiv(R, rps);
    if (sp > 1 && ws_used + (size_t)sp * P.Mo * P.No <= ws_cap) {
        P.splits = sp;
        P.rps = rps;
        P.ws = ws + ws_used;
        ws_used += (size_t)sp * P.Mo * P.No;
    }
}

int tlg_group_launch(const TlgGemmCall *calls, int n, hipStream_t st)
{
    if (n <= 0) return TLG_OK;
    int rc = tlg_ensure_init();
    if (rc) return rc;
    group_env();
    if (n > TLG_MAXPROB / 2) return tlg_fail(TLG_EINVAL, "tlg_dev_gemm_group: at most %d calls", TLG_MAXPROB / 2);

    // Decode runs (every call mm / mm_bt at M <= 8, no residual) go to the
    // GEMV kernels.
    bool gemv = true;
    int mmax = 1;
    for (int i = 0; i < n && gemv; i++) {
        gemv = (calls[i].op == 0 || calls[i].op == 1) && !calls[i].R && !calls[i].dotOut && calls[i].M >= 1 &&
               calls[i].M <= 8 &&
               calls[i].K > 0 &&
               calls[i].N > 0 && calls[i].nseg >= 1 && calls[i].nseg <= TLG_MAXSEG &&
               (calls[i].nseg == 1 || calls[i].op == 1);
        if (calls[i].M > mmax) mmax = calls[i].M;
    }
    if (gemv) {
        rc = tlg_group_flush_launch(st);
        if (rc) return rc;
        rc = tlg_gemv_group_launch(calls, n, st);
        g_group_last_name = tlg_gemv_kernel_name(mmax);
        return rc;
    }

    if ((rc = flush_foreign(st))) return rc;
    if ((rc = ecarry_flush(st))) return rc;
    // Pending reductions write their C; a call that touches such a range must
    // see them first, so they go in a launch of their own.
    for (int k = 0; k < g_npending && g_npending; k++) {
        const Prob &r = g_pending[k];
        const char *c0, *c1;
        span(r.C, r.Mo, r.No, r.ldc, &c0, &c1);
        for (int i = 0; i < n; i++) {
            const TlgGemmCall &c = calls[i];
            const int op = c.op;
            const int Mo = op == 2 ? c.K : c.M, No = op == 1 ? c.K : c.N;
            const char *o0, *o1;
            span(c.C, Mo, No, No, &o0, &o1);
            bool hit = overlap(c0, c1, o0, o1);
            for (int s = 0; s < c.nseg && !hit && op != 3; s++) {
                const int Ns = s ? c.Nseg[s] : c.N;
                const char *x0, *x1, *y0, *y1;
                if (op == 0)      { span(c.A[s], c.M, c.K, c.K, &x0, &x1); span(c.B[s], c.K, Ns, Ns, &y0, &y1); }
                else if (op == 1) { span(c.A[s], c.M, Ns, Ns, &x0, &x1); span(c.B[s], c.K, Ns, Ns, &y0, &y1); }
                else              { span(c.A[s], c.M, c.K, c.K, &x0, &x1); span(c.B[s], c.M, Ns, Ns, &y0, &y1); }
                hit = overlap(c0, c1, x0, x1) || overlap(c0, c1, y0, y1);
            }
            if (!hit && op == 0 && c.R) {
                const char *r0, *r1;
                span(c.R, c.M, c.N, c.N, &r0, &r1);
                hit = overlap(c0, c1, r0, r1);
            }
            if (!hit && op == 1 && c.dotOut) {
                const char *r0, *r1, *d0, *d1;
                span(c.dotB, c.M, c.K, c.K, &r0, &r1);
                span(c.dotOut, c.M, c.K / 32, c.K / 32, &d0, &d1);
                hit = overlap(c0, c1, r0, r1) || overlap(c0, c1, d0, d1);
            }
            if (hit) { rc = tlg_group_flush_launch(st); if (rc) return rc; break; }
        }
    }

    // Problems as the kernel sees them (tiles and splits filled in below).
    Prob probs[TLG_MAXPROB / 2];
    int Rtot[TLG_MAXPROB / 2];
    int rmax = 0;
    bool rowdot = false;
    for (int i = 0; i < n; i++) {
        const TlgGemmCall &c = calls[i];
        if (c.op == 3) {
            // a clear of C[0, M*N) riding along with the GEMMs
            if (c.M <= 0 || c.N <= 0 || !c.C)
                return tlg_fail(TLG_EINVAL, "tlg_dev_gemm_group: call %d: empty clear", i);
            Prob &P = probs[i];
            memset(&P, 0, sizeof P);
            P.kind = PK_ZERO;
            P.C = c.C;
            P.Mo = c.M;
            P.No = c.N;
            P.ldc = c.N;
            P.items = (int)(((size_t)c.M * c.N + TLG_ZERO_CHUNK - 1) / TLG_ZERO_CHUNK);
            Rtot[i] = 0;
            continue;
        }
        if (c.op < 0 || c.op > 2 || c.nseg < 1 || c.nseg > TLG_MAXSEG || (c.nseg > 1 && c.op != 1))
            return tlg_fail(TLG_EINVAL, "tlg_dev_gemm_group: call %d: bad op/nseg", i);
        if (c.M < 0 || c.K < 0 || c.N < 0) return tlg_fail(TLG_EINVAL, "negative dimension");
        Prob &P = probs[i];
        memset(&P, 0, sizeof P);
        P.kind = c.op == 0 ? PK_NN : (c.op == 1 ? PK_NT : PK_TN);
        P.C = c.C;
        P.beta = c.op == 0 ? 0 : (c.beta ? 1 : 0);
        P.nseg = c.nseg;
        int R = 0;
        bool vec = true;
        for (int s = 0; s < c.nseg; s++) {
            const int Ns = s ? c.Nseg[s] : c.N;
            Seg &g = P.seg[s];
            g.A = c.A[s]; g.B = c.B[s];
            switch (c.op) {
            case 0: P.Mo = c.M; P.No = c.N; g.R = c.K; g.lda = c.K; g.ldb = c.N; break;
            case 1: P.Mo = c.M; P.No = c.K; g.R = Ns; g.lda = Ns; g.ldb = Ns; break;
            default: P.Mo = c.K; P.No = c.N; g.R = c.M; g.lda = c.K; g.ldb = c.N; break;
            }
            R += g.R;
            const int la = (P.kind == PK_TN) ? OC : RC, lb = (P.kind == PK_NT) ? RC : OC;
            vec = vec && al16(g.A) && al16(g.B) && g.lda % 4 == 0 && g.ldb % 4 == 0 &&
                  (la == RC ? g.R % 4 == 0 : P.Mo % 4 == 0) && (lb == RC ? g.R % 4 == 0 : P.No % 4 == 0);
        }
        P.ldc = P.No;
        if (!vec || !c.C || R == 0 || P.Mo == 0 || P.No == 0)
            return tlg_fail(TLG_EINVAL, "tlg_dev_gemm_group: call %d needs aligned, non-empty operands", i);
        if (c.dotOut || c.dotB) {
            if (c.op != 1 || c.beta || !c.dotOut || !c.dotB || !al16(c.dotB) || c.K % 32 || c.dotB == c.C)
                return tlg_fail(TLG_EINVAL, "tlg_dev_gemm_group: call %d: block dot only on mm_bt with beta 0, "
                                "K %% 32 == 0, an aligned dotB that is not C", i);
            P.epi = TLG_EPI_ROWDOT;
            P.fin = c.dotB;
            P.X1 = c.dotOut;
            rowdot = true;
        }
        if (c.R) {
            if (c.op != 0 || !al16(c.R) || c.R == c.C)
                return tlg_fail(TLG_EINVAL, "tlg_dev_gemm_group: call %d: residual only on mm, aligned, not C", i);
            P.fin = c.R;
        }
        Rtot[i] = R;
        if (c.op != 2 && R > rmax) rmax = R;
    }
    // split problems aim for about the per-item work of the unsplit ones
    // (or the pinned target)
    const int rtarget = g_group_rt > 0 ? g_group_rt : rmax > g_rtarget ? rmax : g_rtarget;

    // tile shape: pinned, or by the work items it gives the launch
    auto items_of = [&](int cfg) {
        const TileCfg &tc = kCfgs[cfg];
        double items = 0;
        for (int i = 0; i < n; i++) {
            if (probs[i].kind == PK_ZERO) continue;
            const double tiles = (double)cdiv(probs[i].Mo, tc.bm) * cdiv(probs[i].No, tc.bn);
            const double sp = (probs[i].kind == PK_TN && Rtot[i] > rtarget + rtarget / 2)
                            ? (double)cdiv(Rtot[i], rtarget) : 1.0;
            items += tiles * sp;
        }
        return items;
    };
    int ci = g_group_cfg;
    if (ci < 0 && g_cand[0] >= 0) {
        for (int k = 0; k < 4 && g_cand[k] >= 0; k++) {
            ci = g_cand[k];                    // the last one if none is enough
            if (items_of(ci) >= g_min_waves * 256) break;
        }
    } else if (ci < 0) {
        bool tn = false;
        for (int i = 0; i < n; i++) tn = tn || probs[i].kind == PK_TN;
        for (const auto &row : kAuto) {
            ci = row.cfg;
            const double items = items_of(ci);
            if (items < row.items * (g_min_waves / 3.0)) continue;
            if (ci == 33 && !tn) {
                const double rounds = items / 256.0;
                if (rounds < (rounds > 1.0 ? 1.7 : 0.7)) continue;
                if (rounds < 1.0 && rmax <= 512) continue;
                if (rmax <= 512) ci = 47;
            }
            if (ci == 34 && !tn) continue;
            break;
        }
    }
    // the block-dot epilogue stages a whole tile in the stage buffers: not on
    // the 128 x 128 shapes, whose tile is larger than their stages
    if (rowdot && kCfgs[ci].bm * kCfgs[ci].bn > 64 * 128) ci = 38;
    const TileCfg &tc = kCfgs[ci];

    GroupArgs a;
    a.nprob = 0;
    a.rows1 = 0;
    add_reductions(a);
    float *ws = g_tlg.ws + (size_t)g_ws_half * (g_tlg.ws_floats / 2);
    size_t ws_used = 0;
    const size_t ws_cap = g_tlg.ws_floats / 2;
    int order[TLG_MAXPROB / 2];
    double cost[TLG_MAXPROB / 2];
    for (int i = 0; i < n; i++) {
        Prob &P = probs[i];
        order[i] = i;
        if (P.kind == PK_ZERO) { cost[i] = 0.0; continue; }
        P.tiles_n = cdiv(P.No, tc.bn);
        P.tiles = cdiv(P.Mo, tc.bm) * P.tiles_n;
        plan_split(P, Rtot[i], rtarget, ws, ws_used, ws_cap);
        P.items = P.tiles * P.splits;
        cost[i] = (double)P.rps;              // reduction steps per item
    }
    // longest item first (stable: ties keep call order)
    for (int i = 1; i < n; i++)
        for (int j = i; j > 0 && cost[order[j]] > cost[order[j - 1]]; j--) {
            const int t = order[j]; order[j] = order[j - 1]; order[j - 1] = t;
        }
    // the reduction items of the previous launch are short: they go last
    Prob red[TLG_MAXPROB];
    const int nred = a.nprob;
    for (int k = 0; k < nred; k++) red[k] = a.p[k];
    a.nprob = 0;
    for (int k = 0; k < n; k++) {
        const Prob &P = probs[order[k]];
        a.p[a.nprob++] = P;
        if (P.splits > 1) { g_pending[g_npending++] = P; g_pending_st = st; }
    }
    for (int k = 0; k < nred; k++) a.p[a.nprob++] = red[k];
    launch_group(ci, a, group_grid(a), st);
    TLG_HIP(hipGetLastError());
    if (g_npending) g_ws_half ^= 1;
    return TLG_OK;
}

// ----------------------------------------------- expert-batched launch --
// One launch runs `n` expert-batched GEMMs (every expert of each), then, if
// any is a TN problem, one more launch adds their partial slots into the
// outputs.  Rows per expert live on the device (eoff), so the host sizes the
// grid for the worst case: ceil(rows_e / u) summed over experts is at most
// rows / u + E units of u rows.
// Slice reductions an expert launch held back (carry TLG_ECARRY_OUT) for the
// next expert launch over the same row offsets (carry TLG_ECARRY_IN), which
// runs them as its last items and places its own partial slots after
// theirs: the kernel boundary between the two makes the partials visible,
// as for the grouped launches' deferred reductions.  Any other launch that
// uses the workspace launches them first.
static GroupArgs g_ecarry;              // nprob 0: nothing held
static size_t g_ecarry_used = 0;        // workspace floats their partials occupy
static const int *g_ecarry_eoff = nullptr;
static hipStream_t g_ecarry_st = nullptr;

// Queued work whose producer ran on another stream than `st` runs first on
// the producer's stream (ordered after the kernels that wrote its partials),
// so a launch on `st` never sums partials it is not ordered after.  Work
// queued on `st` itself keeps riding along.
static int flush_foreign(hipStream_t st)
{
    if (g_ecarry.nprob && g_ecarry_st != st) {
        const int rc = ecarry_flush(g_ecarry_st);
        if (rc) return rc;
    }
    if (g_npending && g_pending_st != st) {
        const int rc = group_flush_dense(g_pending_st);
        if (rc) return rc;
    }
    return TLG_OK;
}

// Launches of expert reductions alone
static void launch_reductions(const GroupArgs &a, hipStream_t st)
{
    (void)tlg_expert_part(3, group_seal(a), group_grid(a), st);
}

static int ecarry_flush(hipStream_t st)
{
    if (!g_ecarry.nprob) return TLG_OK;
    launch_reductions(g_ecarry, st);
    g_ecarry.nprob = 0;
    g_ecarry_used = 0;
    TLG_HIP(hipGetLastError());
    return TLG_OK;
}

// Held expert reductions and queued dense ones (column sums, split
// reductions) on one stream: one launch for both, the held expert
// reductions first (the expert kernel stages p[0]'s row offsets), then the
// queued ones, which it runs as the dense kernel does.  *done = false when
// there are not both kinds (or too many problems for one launch).
static int ecarry_flush_with_pending(hipStream_t st, bool *done)
{
    *done = false;
    if (!g_ecarry.nprob || !g_npending || g_ecarry.nprob + g_npending > TLG_MAXPROB) return TLG_OK;
    GroupArgs a = g_ecarry;
    add_reductions(a);
    launch_reductions(a, st);
    g_ecarry.nprob = 0;
    g_ecarry_used = 0;
    TLG_HIP(hipGetLastError());
    *done = true;
    return TLG_OK;
}

int tlg_group_pending(void) { return g_npending + g_ecarry.nprob; }

// Every queued reduction (and an expert launch's held carry) launched now,
// each on the stream its partials were written on: what tlg_dev_free runs
// before it releases memory that queued work may read or write.
int tlg_group_flush_all(void)
{
    if (g_ecarry.nprob) {
        const int rc = tlg_group_flush_launch(g_ecarry_st);
        if (rc) return rc;
    }
    return g_npending ? tlg_group_flush_launch(g_pending_st) : TLG_OK;
}

// Queued work whose partials were written on `st` launched now, on `st`:
// what tlg_stream_destroy runs before the handle goes away.
int tlg_group_flush_stream(hipStream_t st)
{
    if ((g_ecarry.nprob && g_ecarry_st == st) || (g_npending && g_pending_st == st))
        return tlg_group_flush_launch(st);
    return TLG_OK;
}

// Shutdown: the queued reductions (and an expert launch's held carry) run
// on `st` while the workspace they read still exists; then the queue is
// empty and the workspace halves start over, so nothing queued before a
// tlg_shutdown can run against freed memory after a later tlg_init.
int tlg_group_drain(hipStream_t st)
{
    const int rc = tlg_group_flush_launch(st);
    g_npending = 0;
    g_ecarry.nprob = 0;
    g_ecarry_used = 0;
    g_ecarry_eoff = nullptr;
    g_ws_half = 0;
    return rc;
}

// Extents of an expert shape.
static TileCfg expert_shape(int key)
{
#define TLG_ROW(k, bm, bn, bk, wgm, wk, nw) if (key == k) return TileCfg{bm, bn, bk, wgm, wk, 2, nw, 0};
    TLG_EXPERTS(TLG_ROW)
#undef TLG_ROW
    return expert_shape(15);
}

int tlg_expert_launch(const TlgExpertCall *calls, int n, const int *eoff, int E, int rows, hipStream_t st,
                      int carry)
{
    if (n <= 0) return TLG_OK;
    int rc = tlg_ensure_init();
    if (rc) return rc;
    if (n > TLG_MAXPROB / 2) return tlg_fail(TLG_EINVAL, "expert launch: at most %d calls", TLG_MAXPROB / 2);
    // eoff NULL: one expert owning every row (dense rows, known on the host)
    const bool dense = eoff == nullptr;
    if ((dense && E != 1) || E < 1 || E > TLG_MAX_EXPERTS || rows < 0)
        return tlg_fail(TLG_EINVAL, "expert launch: bad row offsets or %d experts", E);
    if (rows == 0) return TLG_OK;
    if ((rc = flush_foreign(st))) return rc;
    // held slice reductions join this launch only if it asks for them and
    // shares their row offsets
    const bool cin = (carry & TLG_ECARRY_IN) && g_ecarry.nprob && g_ecarry_eoff == eoff && !dense;
    if (!cin && (rc = ecarry_flush(st))) return rc;
    // Pending split reductions of grouped launches ride along when this
    // launch writes no partial slots (they reuse the whole workspace) and
    // touches none of their outputs; otherwise they are flushed first.
    bool ride = dense;
    for (int i = 0; i < n && ride; i++) {
        const TlgExpertCall &c = calls[i];
        if (c.op == 2 || c.amap || c.omap) { ride = false; break; }
        const int Nr = c.op == 0 ? c.N : c.K;          // output / epilogue row width
        const int Na = c.op == 0 ? c.K : c.N;          // A row width
        const char *r0[7], *r1[7];
        int m = 0;
        if (c.C) span(c.C, rows, Nr, Nr, &r0[m], &r1[m]), m++;
        if (c.X1) span(c.X1, rows, Nr, Nr, &r0[m], &r1[m]), m++;
        if (c.X2) span(c.X2, rows, Nr, Nr, &r0[m], &r1[m]), m++;
        if (c.fin) span(c.fin, rows, Nr, Nr, &r0[m], &r1[m]), m++;
        span(c.A[0], rows, Na, Na, &r0[m], &r1[m]), m++;
        span(c.B[0], c.K, c.N, c.N, &r0[m], &r1[m]), m++;
        if (c.B2) span(c.B2, c.K, c.N, c.N, &r0[m], &r1[m]), m++;
        for (int k = 0; k < g_npending && ride; k++) {
            const char *c0, *c1;
            span(g_pending[k].C, g_pending[k].Mo, g_pending[k].No, g_pending[k].ldc, &c0, &c1);
            for (int j = 0; j < m && ride; j++) ride = !overlap(c0, c1, r0[j], r1[j]);
        }
    }
    if (!ride) {
        rc = group_flush_dense(st);
        if (rc) return rc;
    }

    group_env();
    Prob probs[TLG_MAXPROB / 2];
    for (int i = 0; i < n; i++) {
        const TlgExpertCall &c = calls[i];
        if (c.op < 0 || c.op > 2 || c.nseg < 1 || c.nseg > 2 || (c.nseg > 1 && c.op != 1))
            return tlg_fail(TLG_EINVAL, "expert launch: call %d: bad op/nseg", i);
        Prob &P = probs[i];
        memset(&P, 0, sizeof P);
        P.kind = c.op == 0 ? PK_NN : (c.op == 1 ? PK_NT : PK_TN);
        P.C = c.C;
        P.beta = c.beta ? 1 : 0;
        P.nseg = c.nseg;
        P.eoff = eoff;
        P.nexp = E;
        P.es = c.es;
        P.amap = c.amap;
        P.omap = c.omap;
        P.B2 = c.B2;
        P.epi = c.epi;
        P.X1 = c.X1;
        P.X2 = c.X2;
        P.fin = c.fin;
        P.gate = c.gate;
        // fused forms: the pair only with the SwiGLU epilogue of an NN call;
        // SwiGLU backward on NT (da = dy W2^T); the combine on NN
        const bool epi_ok =
            (c.epi == TLG_EPI_STORE && !c.B2) ||
            (c.epi == TLG_EPI_SWIGLU && c.op == 0 && c.B2 && al16(c.B2) && c.nseg == 1 && !c.beta) ||
            (c.epi == TLG_EPI_SWIGLU_BWD && c.op == 1 && !c.B2 && c.X1 && c.X2) ||
            (c.epi == TLG_EPI_COMBINE && c.op == 0 && !c.B2 && c.omap && c.fin && c.gate && c.nseg == 1 &&
             !c.beta && !c.amap);
        if (!epi_ok || (c.amap && c.nseg != 1))
            return tlg_fail(TLG_EINVAL, "expert launch: call %d: bad epilogue %d / gather / pair", i, c.epi);
        bool vec = (c.C || c.epi == TLG_EPI_SWIGLU_BWD) && (c.es % 4 == 0);
        for (int s = 0; s < c.nseg; s++) {
            const int Ns = s ? c.Nseg[s] : c.N;
            Seg &g = P.seg[s];
            g.A = c.A[s]; g.B = c.B[s];
            switch (c.op) {
            case 0: P.No = c.N; g.R = c.K; g.lda = c.K; g.ldb = c.N; break;
            case 1: P.No = c.K; g.R = Ns; g.lda = Ns; g.ldb = Ns; break;
            default: P.Mo = c.K; P.No = c.N; g.R = rows; g.lda = c.K; g.ldb = c.N; break;
            }
            vec = vec && g.A && g.B && al16(g.A) && al16(g.B) && g.lda % 4 == 0 && g.ldb % 4 == 0 && g.R > 0;
        }
        P.ldc = P.No;
        if (!vec || P.No <= 0 || (c.op == 2 && P.Mo <= 0) || P.No % 4 || P.Mo % 4)
            return tlg_fail(TLG_EINVAL, "expert launch: call %d needs aligned operands, widths %% 4 == 0", i);
    }
    // reduction slices of the TN problems (g_erps rows, doubled until the
    // partials fit): short slices balance experts of very different sizes
    int rps = cdiv(g_erps, 64) * 64;
    const size_t used0 = cin ? g_ecarry_used : 0;     // the held partials come first
    auto need = [&](int u) {
        size_t t = used0;
        for (int i = 0; i < n; i++)
            if (probs[i].kind == PK_TN) t += (size_t)(rows / u + E) * probs[i].Mo * probs[i].No;
        return t;
    };
    while (need(rps) > g_tlg.ws_floats && rps < rows) rps *= 2;
    if (need(rps) > g_tlg.ws_floats)
        return tlg_fail(TLG_ENOMEM, "expert launch: %d experts' partials exceed the workspace", E);

    // tile shape: 128x128 (8 waves of 32x64, so a SwiGLU pair shares a lane)
    // from 160 items on, else the largest of 64x64, 64x32 and 32x32 that gives
    // about 320 (m8 training step 7.29 ms on 128x128 tiles, 7.64 on 64x64; the
    // m3 MoE layer 241 us, 243 on 64x64, 267 on 64x32)
    auto items_for = [&](const TileCfg &c) {
        double t = 0;
        for (int i = 0; i < n; i++) {
            const Prob &P = probs[i];
            const double tn = cdiv(P.No, P.B2 ? c.bn / 2 : c.bn);
            t += P.kind == PK_TN ? cdiv(P.Mo, c.bm) * tn * (rows / rps + E) : (cdiv(rows, c.bm) + E) * tn;
        }
        return t;
    };
    const double by = g_min_waves / 3.0;
    const int ci = g_expert_cfg >= 0 ? g_expert_cfg
                 : items_for(expert_shape(9)) >= 160 * by ? 9
                 : items_for(expert_shape(3)) >= 320 * by ? 3
                 : items_for(expert_shape(14)) >= 320 * by ? 14 : 15;
    const TileCfg tc = expert_shape(ci);
    GroupArgs a, red, pend;
    a.nprob = red.nprob = pend.nprob = 0;
    a.rows1 = red.rows1 = pend.rows1 = dense ? rows : 0;
    if (ride) add_reductions(pend);
    size_t used = used0;
    int order[TLG_MAXPROB / 2];
    for (int i = 0; i < n; i++) {
        Prob &P = probs[i];
        P.tiles_n = cdiv(P.No, P.B2 ? tc.bn / 2 : tc.bn);
        if (P.kind == PK_TN) {
            P.tiles = cdiv(P.Mo, tc.bm) * P.tiles_n;
            P.unit = rps;
            P.rps = rps;
            P.items = P.tiles * (rows / rps + E);
            P.ws = g_tlg.ws + used;
            used += (size_t)(rows / rps + E) * P.Mo * P.No;
        } else {
            P.unit = tc.bm;
            P.items = (cdiv(rows, tc.bm) + E) * P.tiles_n;
        }
        order[i] = i;
    }
    // longest item first: TN items run rps rows, the others their full R
    auto cost = [&](const Prob &P) {
        int r = 0;
        for (int s = 0; s < P.nseg; s++) r += P.seg[s].R;
        return P.kind == PK_TN ? P.unit : r;
    };
    for (int i = 1; i < n; i++)
        for (int j = i; j > 0 && cost(probs[order[j]]) > cost(probs[order[j - 1]]); j--) {
            const int t = order[j]; order[j] = order[j - 1]; order[j - 1] = t;
        }
    for (int k = 0; k < n; k++) {
        const Prob &P = probs[order[k]];
        a.p[a.nprob++] = P;
        if (P.kind == PK_TN) {
            Prob r = P;
            r.kind = PK_RED;
            r.items = E * (int)(((size_t)P.Mo * P.No + TLG_ERED_CHUNK - 1) / TLG_ERED_CHUNK);
            red.p[red.nprob++] = r;
        }
    }
    // the grouped launches' reductions that ride along go last (short items),
    // with the held slice reductions of the previous expert launch
    for (int k = 0; k < pend.nprob; k++) a.p[a.nprob++] = pend.p[k];
    if (cin) {
        if (a.nprob + g_ecarry.nprob > TLG_MAXPROB) return tlg_fail(TLG_EINVAL, "expert launch: too many problems");
        for (int k = 0; k < g_ecarry.nprob; k++) a.p[a.nprob++] = g_ecarry.p[k];
        g_ecarry.nprob = 0;
        g_ecarry_used = 0;
    }
    // an XCD's share of the real items can exceed its share of the upper
    // bound by one per expert problem
    static_assert(sizeof(GroupArgs) <= 4096, "kernel arguments");
    const int eg = group_grid(a) + 8 * n;
    // + 200: streaming stores
    const int key = ci + ((g_expert_sched >= 0 ? g_expert_sched : dense ? 2 : 1) == 2 ? 200 : 0);
    if (!tlg_expert_part(key, group_seal(a), eg, st))
        return tlg_fail(TLG_EINVAL, "expert launch: no kernel for tile form %d", key);
    TLG_HIP(hipGetLastError());
    if (red.nprob && (carry & TLG_ECARRY_OUT) && !dense && g_npending == 0) {
        g_ecarry = red;                  // the next expert launch runs them
        g_ecarry_used = used;
        g_ecarry_eoff = eoff;
        g_ecarry_st = st;
    } else if (red.nprob) {
        launch_reductions(red, st);
        TLG_HIP(hipGetLastError());
    }
    return TLG_OK;
}

// ------------------------------------------------------ seeded fill ------
// splitmix64 of (seed, pair index) -> two 53-bit uniforms -> Box-Muller pair.
__device__ __forceinline__ unsigned long long splitmix64(unsigned long long x)
{
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__global__ void k_fill_normal(float *__restrict__ p, size_t n, unsigned long long seed, float scale)
{
    const size_t pairs = (n + 1) / 2;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < pairs; i += stride) {
        const unsigned long long h1 = splitmix64(seed ^ (2 * i));
        const unsigned long long h2 = splitmix64(h1 ^ (2 * i + 1));
        double u1 = (double)(h1 >> 11) * (1.0 / 9007199254740992.0);
        const double u2 = (double)(h2 >> 11) * (1.0 / 9007199254740992.0);
        if (u1 < 1e-300) u1 = 1e-300;
        const double r = sqrt(-2.0 * log(u1));
        const double t = 6.283185307179586 * u2;
        p[2 * i] = scale * (float)(r * cos(t));
        if (2 * i + 1 < n) p[2 * i + 1] = scale * (float)(r * sin(t));
    }
}

int tlg_fill_normal_launch(float *dst, size_t n, unsigned long long seed, float scale, hipStream_t st)
{
    if (n == 0) return TLG_OK;
    if (!dst) return tlg_fail(TLG_EINVAL, "tlg_dev_fill_normal: NULL destination");
    size_t blocks = ((n + 1) / 2 + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_fill_normal, dim3((unsigned)blocks), dim3(256), 0, st, dst, n, seed, scale);
    TLG_HIP(hipGetLastError());
    return TLG_OK;
}

// ------------------------------------------------------ measurement probes --
// Plain streaming copy (the calibration kernel for HBM byte counters and the
// achievable-bandwidth probe): dst[i] = src[i], float4 per thread.
// Streaming probes: each thread moves 8 float4 per round (all 8 loads in
// flight before any is used), rounds stride over the grid's chunks of 8 x 256
// float4; loads and stores are nontemporal (the data is not reused).
#define TLG_CP_U 8
__global__ __launch_bounds__(256) void k_copy(const f32x4 *__restrict__ src, f32x4 *__restrict__ dst, size_t n4)
{
    const size_t chunk = (size_t)TLG_CP_U * 256;
    for (size_t c = (size_t)blockIdx.x * chunk; c < n4; c += (size_t)gridDim.x * chunk) {
        f32x4 v[TLG_CP_U];
#pragma unroll
        for (int k = 0; k < TLG_CP_U; k++) {
            const size_t i = c + threadIdx.x + (size_t)k * 256;
            v[k] = __builtin_nontemporal_load(src + (i < n4 ? i : n4 - 1));
        }
#pragma unroll
        for (int k = 0; k < TLG_CP_U; k++) {
            const size_t i = c + threadIdx.x + (size_t)k * 256;
            if (i < n4) __builtin_nontemporal_store(v[k], dst + i);
        }
    }
}

// Read-only stream: the sum of src (kept so the loads are not removed) goes
// to sink[0] only if it equals a value no probe input produces.
__global__ __launch_bounds__(256) void k_read(const f32x4 *__restrict__ src, size_t n4, float *__restrict__ sink)
{
    const size_t chunk = (size_t)TLG_CP_U * 256;
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
    for (size_t c = (size_t)blockIdx.x * chunk; c < n4; c += (size_t)gridDim.x * chunk) {
        f32x4 v[TLG_CP_U];
#pragma unroll
        for (int k = 0; k < TLG_CP_U; k++) {
            const size_t i = c + threadIdx.x + (size_t)k * 256;
            v[k] = __builtin_nontemporal_load(src + (i < n4 ? i : n4 - 1));
        }
#pragma unroll
        for (int k = 0; k < TLG_CP_U; k++) a += v[k];
    }
    if (a.x + a.y + a.z + a.w == -1.2345e30f) sink[0] = 1.f;
}

static size_t stream_blocks(size_t n4)
{
    size_t blocks = (n4 + TLG_CP_U * 256 - 1) / (TLG_CP_U * 256);
    return blocks > 256 * 8 ? 256 * 8 : blocks;
}

int tlg_copy_launch(float *dst, const float *src, size_t n, hipStream_t st)
{
    if (n % 4 || ((uintptr_t)dst & 15) || ((uintptr_t)src & 15))
        return tlg_fail(TLG_EINVAL, "tlg_dev_copy: needs 16-byte aligned buffers and n %% 4 == 0");
    const size_t n4 = n / 4, blocks = stream_blocks(n4);
    if (blocks == 0) return TLG_OK;
    hipLaunchKernelGGL(k_copy, dim3((unsigned)blocks), dim3(256), 0, st,
                       (const f32x4 *)src, (f32x4 *)dst, n4);
    TLG_HIP(hipGetLastError());
    return TLG_OK;
}

int tlg_read_launch(const float *src, size_t n, float *sink, hipStream_t st)
{
    if (n % 4 || ((uintptr_t)src & 15) || !sink)
        return tlg_fail(TLG_EINVAL, "tlg_dev_read: needs a 16-byte aligned buffer, n %% 4 == 0 and a sink");
    const size_t n4 = n / 4, blocks = stream_blocks(n4);
    if (blocks == 0) return TLG_OK;
    hipLaunchKernelGGL(k_read, dim3((unsigned)blocks), dim3(256), 0, st, (const f32x4 *)src, n4, sink);
    TLG_HIP(hipGetLastError());
    return TLG_OK;
}

// Achievable fp32 MFMA rate: every wave runs `iters` x 4 independent
// v_mfma_f32_32x32x2_f32 chains on register operands, then stores one value
// per lane so the work is not eliminated.
__global__ __launch_bounds__(256) void k_mfma_peak(float *__restrict__ out, int iters, float seed)
{
    f32x16 c0 = {}, c1 = {}, c2 = {}, c3 = {};
    const float a = seed + threadIdx.x * 1e-7f, b = seed - threadIdx.x * 1e-7f;
    for (int i = 0; i < iters; i++) {
        c0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f32_32x32x2f32(b, a, c1, 0, 0, 0);
        c2 = __builtin_amdgcn_mfma_f32_32x32x2f32(a, a, c2, 0, 0, 0);
        c3 = __builtin_amdgcn_mfma_f32_32x32x2f32(b, b, c3, 0, 0, 0);
    }
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < 16; v++) s += c0[v] + c1[v] + c2[v] + c3[v];
    out[(size_t)blockIdx.x * blockDim.x + threadIdx.x] = s;
}

// The same of the bf16 matrix cores, which the tiles use: v_mfma_f32_32x32x16_bf16.
__global__ __launch_bounds__(256) void k_mfma_bf16_peak(float *__restrict__ out, int iters, float seed)
{
    f32x16 c0 = {}, c1 = {}, c2 = {}, c3 = {};
    bf16x8 a, b;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        a[k] = (__bf16)(seed + k * 0.01f + threadIdx.x * 1e-3f);
        b[k] = (__bf16)(seed - k * 0.01f - threadIdx.x * 1e-3f);
    }
    for (int i = 0; i < iters; i++) {
        c0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a, c1, 0, 0, 0);
        c2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, a, c2, 0, 0, 0);
        c3 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, b, c3, 0, 0, 0);
    }
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < 16; v++) s += c0[v] + c1[v] + c2[v] + c3[v];
    out[(size_t)blockIdx.x * blockDim.x + threadIdx.x] = s;
}

int tlg_mfma_bf16_peak_launch(float *out, int blocks, int iters, hipStream_t st)
{
    if (blocks <= 0 || iters <= 0) return tlg_fail(TLG_EINVAL, "tlg_dev_mfma_bf16_peak: bad size");
    hipLaunchKernelGGL(k_mfma_bf16_peak, dim3(blocks), dim3(256), 0, st, out, iters, 0.5f);
    TLG_HIP(hipGetLastError());
    return TLG_OK;
}

int tlg_mfma_peak_launch(float *out, int blocks, int iters, hipStream_t st)
{
    if (blocks <= 0 || iters <= 0) return tlg_fail(TLG_EINVAL, "tlg_dev_mfma_peak: bad size");
    hipLaunchKernelGGL(k_mfma_peak, dim3(blocks), dim3(256), 0, st, out, iters, 0.5f);
    TLG_HIP(hipGetLastError());
    return TLG_OK;
}

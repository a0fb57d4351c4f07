// tlg_tile.h -- the GEMM tile and its kernels for gfx950 (device code of
// tlg_gemm.hip), behind mm / mm_bt / mm_atb.
//
// One tile routine serves the three reference primitives (tinylm.c:438-537):
//
//   mm      Y  = X  W      C(i,j) = sum_r X[i][r]  W[r][j]     NN
//   mm_bt   dX += dY W^T   C(i,j) = sum_r dY[i][r] W[j][r]     NT
//   mm_atb  dW += X^T dY   C(i,j) = sum_r X[r][i]  dY[r][j]    TN
//
// Each operand is either contiguous along the reduction index r ("RC") or
// along its output index ("OC").  A workgroup owns a BM x BN tile of C; its
// waves form a WGM x WGN grid over the tile and WK groups along each stage of
// BK reduction steps, each wave 32x32 blocks of it.
//
// The arithmetic: gfx950's matrix cores run bf16 at 14 times the fp32 rate
// (k_mfma_bf16_peak 2.0 PFLOP/s, k_mfma_peak 146 TFLOP/s), so every fp32 operand
// is split, exactly, into three bf16 pieces while it is staged, and a product into the
// six piece products that reach 2^-25 of it: 336 TFLOP/s of fp32 work at that
// rate.  Products of bf16 are exact in fp32 and a 32x32x16 MFMA rounds its
// running sum once per 16 steps, so the result is closer to fp64's than the
// fp32 MFMA chain's, which rounds at every step: 2.5 to 3 times, at 32 to 8192
// steps (2.9e-7 -> 0.9e-7 at 256, 1.7e-6 -> 5.7e-7 at 8192, N(0, 1) values).
//
// What bounds it: a stage's waits.  By counters (8192 x 384 x 2048, dX / fwd /
// dW) the matrix cores are busy 40 / 41 / 38 % and the LDS 25 / 33 / 38 % of the
// time, 0 / 16 / 37 % of the latter bank conflicts (operands along their output
// index).  Beside them run the splits (13 vector instructions per pair of
// values) and the loads, and one 8-wave workgroup a CU has nothing else to run
// at a stage's barrier.  With reads, splits and loads left out the 128x128
// tile's MFMAs alone ran at 319 TFLOP/s at R = 1536; with them 190.  Loads run
// NR stages ahead into registers, the split runs between the MFMAs, LDS is
// double buffered, one barrier per stage.
// 8192 x 384 x 2048 (fwd / dX / dW) 117 / 152 / 157 -> 80 / 77 / 84 us against
// the fp32 MFMA tiles this replaces; 4096 x 256 x 768 24 / 22 / 35 -> 14 / 16 / 21.
//
// Reduction order inside a 16-step MFMA: lanes 0-31 supply steps 0-7, lanes
// 32-63 steps 8-15.  The result differs from the reference's sequential chain
// only by rounding (parity bar: max|err| / mean|ref| <= 1e-4).
//
// Split reduction: when output tiles are too few to fill 256 CUs (mm_atb's
// dW is small, its reduction long), the r range is split over `splits`
// workgroups.  Each writes its partial sum as a plain Mo x No matrix into a
// workspace; a later kernel adds the partials to C in split order
// (deterministic) and applies beta.  Nothing crosses workgroups inside a
// kernel, so no device-scope fence is needed: on gfx950 such a fence writes
// back and invalidates the XCD's L2, which costs every co-resident workgroup
// its cached operands.
//
// Grouped launches (tlg_dev_gemm_group): one kernel runs a list of problems
// of any of the three kinds -- the GEMMs a caller issues back to back with
// no other work in between -- plus the deferred split reductions of the
// previous grouped launch.  The kernel boundary between the two launches is
// what makes the partials visible, so a split costs no extra launch.
#ifndef TLG_TILE_H
#define TLG_TILE_H
#include "tlg_internal.h"

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

enum { RC = 0, OC = 1 };

// 2^16 x = h + m + l in bf16 pieces, each the round to nearest of what the ones
// before it leave: 3 x 8 significant bits hold an fp32's 24, and bf16's smallest
// step, 2^-133, is 2^16 times fp32's, so the sum is exact down to fp32's last
// subnormal (unscaled, l ended at |x| = 2^-110: normwise errors of 2.7e-5 at
// 1e-36, 2.6e-3 at 1e-38).  tile_sum takes the 2^32 of a product back out.
// Operands from 2^112 and sums from 2^96 on overflow: tile_fix forms them.  The
// two multiplications cost 0 to 2 % (8192 x 384 x 2048, forward and backward,
// 244 -> 248 us; m8 training step 6.90 -> 7.06 ms); m and l alone times 2^16,
// with a third accumulator for their products, cost the m8 step 7 %.
// Only plain vector instructions: up to six of them run under each MFMA for
// nothing (measured: 33 cycles with 0 to 6, + 4 for each further one), where
// v_dot2c_f32_bf16, which would give a remainder in one instruction, stalls
// the matrix core (53 cycles with two of them).  The mask sits in a vector
// register: v_and_b32 takes 2.5 cycles so, 4.2 with a scalar or a literal.
__device__ __forceinline__ void split2(float x0, float x1, unsigned &h, unsigned &m, unsigned &l)
{
    unsigned mask = 0xffff0000u;
    asm("" : "+v"(mask));
    auto lo = [](unsigned p) { return __builtin_bit_cast(float, p << 16); };
    auto hi = [&](unsigned p) { return __builtin_bit_cast(float, p & mask); };
    x0 *= 0x1p16f, x1 *= 0x1p16f;
    h = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{x0, x1}), bf16x2));
    const float r0 = x0 - lo(h), r1 = x1 - hi(h);
    m = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{r0, r1}), bf16x2));
    const float q0 = r0 - lo(m), q1 = r1 - hi(m);
    l = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{q0, q1}), bf16x2));
}
__device__ __forceinline__ void split4(f32x4 x, u32x2 &h, u32x2 &m, u32x2 &l)
{
    unsigned a, b, c;
    split2(x[0], x[1], a, b, c);
    h[0] = a; m[0] = b; l[0] = c;
    split2(x[2], x[3], a, b, c);
    h[1] = a; m[1] = b; l[1] = c;
}

__device__ __forceinline__ s16x4 lds_read_tr(const char *p)
{
    typedef __attribute__((address_space(3))) s16x4 lds4;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)p);
}

// One staged operand in LDS: three planes (the h, m and l pieces) of bf16.
//   RC: [outer][BK]; the 16-byte chunks of a row are permuted by its index so
//       that the 16 rows of a ds_read_b128 phase cover the 64 banks (4.5
//       cycles per wave; 8.0 unpermuted)
//   OC: [BK][outer]; the 32-byte chunks of a row are permuted by its index so
//       that the 4 rows of a transposing read do not meet in a bank
// Rows stay unpadded, so a wave's stores fill whole 256-byte lines of banks
// (a padded pitch cost a ds_write_b64 8.3 cycles instead of 6.7).
template <int LAY, int OUTER, int BK>
struct LdsOp {
    static constexpr int PITCH = 2 * (LAY == RC ? BK : OUTER);
    static constexpr int PLANE = (LAY == RC ? OUTER : BK) * PITCH;
    static constexpr int BYTES = 3 * PLANE;
    // byte offset of (outer o, step r); o (OC) or r (RC) in units of 4
    __device__ static __forceinline__ int at(int o, int r)
    {
        static_assert(BK == 16 || BK == 32 || BK == 64, "swizzle");
        static_assert(OUTER == 32 || OUTER % 64 == 0, "swizzle");
        if constexpr (LAY == RC) {
            constexpr int CH = BK / 8, SH = BK == 16 ? 3 : BK == 32 ? 2 : 1;
            return o * PITCH + (((r >> 3) ^ ((o >> SH) & (CH - 1))) << 4) + ((r & 7) << 1);
        } else {
            const int x = OUTER == 32 ? (r >> 1) & 1 : r & 3;
            return r * PITCH + (((o >> 4) ^ x) << 5) + ((o & 15) << 1);
        }
    }
};

// Stage one operand tile into registers, four values per load (a 16-byte load
// needs 4-byte alignment only; VEC = the rows themselves are whole float4s).
// OUTER = tile extent along the operand's output index.  Tile rows (RC) or columns (OC) past `oext` re-read
// the last valid ones: they feed only outputs that are not stored.  Steps
// past `rend` (the last stage of a reduction that is no multiple of BK) are
// read from sixteen zero bytes, or left out value by value without VEC.
//
// Two forms serve the expert GEMMs of the MoE layer (float4 path only):
//   G   gathered rows: the operand's memory row of tile row x is map[x] (RC:
//       the rows are output rows, looked up once per tile) or map[r] (OC: the
//       rows are reduction steps, looked up per stage by prep(), a full
//       prefetch round ahead of the load that uses it, so waiting for the
//       map never waits for the operand loads issued after it).
//   PB  paired columns (OC only): the tile's columns alternate, pair_unit at
//       a time, between P's and P2's columns o0 + [0, OUTER/2).
static __device__ __attribute__((aligned(16))) float g_zero_chunk[4] = {0.f, 0.f, 0.f, 0.f};

// Columns of one operand before the other's in a paired tile of BN columns.
__host__ __device__ constexpr int pair_unit(int bn) { return bn >= 64 ? 32 : bn / 2; }

// Where a thread's chunks of an operand tile lie.  Stage st is at a uniform
// distance from the first one, so a load costs one 64-bit add.
template <int LAY, int OUTER, int BK, bool VEC, int NT, bool G = false, bool PB = false>
struct TilePtr {
    static constexpr int PER = OUTER * BK / 4 / NT;   // float4 chunks per thread
    static constexpr int W = PER % 2 == 0 ? 2 : 1;    // neighbouring float4s per chunk of a thread
    static constexpr int U = pair_unit(OUTER);
    // Without VEC an OC row may end inside a chunk: the chunk is then read
    // ending with the row, and its values move down by this many places.
    __device__ __forceinline__ int shift(int tid, int q) const { return o0 + col(tid, q) - (oext - 4); }
    // chunk q of thread tid: its row (outer index RC, step OC) and first column
    __device__ static __forceinline__ int row(int tid, int q)
    {
        return (tid + NT * (q / W)) / ((LAY == RC ? BK : OUTER) / (4 * W));
    }
    __device__ static __forceinline__ int col(int tid, int q)
    {
        return (tid + NT * (q / W)) % ((LAY == RC ? BK : OUTER) / (4 * W)) * (4 * W) + 4 * (q % W);
    }
    static_assert(OUTER * BK / 4 % NT == 0, "tile must split evenly over the workgroup's threads");
    static_assert(!PB || (LAY == OC && U % (4 * W) == 0), "paired columns: OC tiles");
    static_assert(!(G || PB) || VEC, "gathered / paired tiles load float4");
    const float *p[PER];
    const float *P;
    const int *map;
    int ld, o0, oext, rend;

    __device__ __forceinline__ void init(const float *__restrict__ P_, int ld_, int o0_, int oext_, int r0, int rend_,
                                         int tid, const int *__restrict__ map_, const float *__restrict__ P2)
    {
        P = P_; ld = ld_; o0 = o0_; oext = oext_; rend = rend_; map = map_;
#pragma unroll
        for (int q = 0; q < PER; q++) {
            if (LAY == RC) {
                const int o = min(o0 + row(tid, q), oext - 1);
                p[q] = P + (size_t)(G ? map[o] : o) * ld + r0 + col(tid, q);
            } else {
                int o = col(tid, q);
                const bool second = PB && (o & U);
                if (PB) o = o / (2 * U) * U + o % U;
                p[q] = (second ? P2 : P) + min(o0 + o, oext - 4);
                if (!G) p[q] += (size_t)(r0 + row(tid, q)) * ld;
            }
        }
    }
};

template <int LAY, int OUTER, int BK, bool VEC, int NT, bool G = false, bool PB = false>
struct TileLoader {
    using Ptr = TilePtr<LAY, OUTER, BK, VEC, NT, G, PB>;
    static constexpr int PER = Ptr::PER;
    f32x4 v[PER];
    int rs[G && LAY == OC ? PER : 1];                 // gathered memory rows

    __device__ __forceinline__ void prep(const Ptr &t, int r0, int tid)
    {
        if constexpr (G && LAY == OC) {
#pragma unroll
            for (int q = 0; q < PER; q++) rs[q] = t.map[min(r0 + Ptr::row(tid, q), t.rend - 1)];
        }
    }

    // Steps r0 + [0, BK) (dr = r0 - the first stage's); TAIL: steps past rend
    // read as 0.  Every load is unconditional, so the compiler counts the ones
    // outstanding exactly and waiting for one stage does not wait for the
    // stages prefetched after it.
    template <bool TAIL>
    __device__ __forceinline__ void load(const Ptr &t, int r0, int dr, int tid)
    {
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int pr = Ptr::row(tid, q), pc = Ptr::col(tid, q);
            const float *p = t.p[q];
            if constexpr (G && LAY == OC) p += (size_t)rs[q] * t.ld;
            else p += LAY == RC ? (size_t)dr : (size_t)dr * t.ld;
            if constexpr (VEC) {
                if constexpr (TAIL) {
                    if (r0 + (LAY == RC ? pc : pr) >= t.rend) p = g_zero_chunk;
                }
                v[q] = *reinterpret_cast<const f32x4 *>(p);
            } else if constexpr (!TAIL) {
                v[q] = *reinterpret_cast<const f32x4u *>(p);
            } else {
                f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const int o = min(t.o0 + (LAY == RC ? pr : pc + c), t.oext - 1);
                    const int r = r0 + (LAY == RC ? pc + c : pr);
                    if (r < t.rend) x[c] = LAY == RC ? t.P[(size_t)o * t.ld + r] : t.P[(size_t)r * t.ld + o];
                }
                v[q] = x;
            }
        }
    }
    // (see TilePtr::shift)
    __device__ __forceinline__ void align(const Ptr &t, int tid)
    {
        if constexpr (!VEC && LAY == OC) {
#pragma unroll
            for (int q = 0; q < PER; q++) {
                const int s = t.shift(tid, q);
                f32x4 x = v[q];
                if (s > 0 && (s & 1)) x = f32x4{x[1], x[2], x[3], x[3]};
                if (s > 0 && (s & 2)) x = f32x4{x[2], x[3], x[3], x[3]};
                v[q] = x;
            }
        }
    }

    // Split each staged value into its three bf16 pieces and store the pieces'
    // planes (LdsOp): a chunk's 4 or 8 neighbours are reduction steps (RC) or
    // output indices (OC), 8 or 16 bytes in each plane either way.
    __device__ __forceinline__ void store(char *__restrict__ L, int tid) const
    {
        using O = LdsOp<LAY, OUTER, BK>;
        constexpr int W = Ptr::W;
#pragma unroll
        for (int q = 0; q < PER; q += W) {
            const int pr = Ptr::row(tid, q), pc = Ptr::col(tid, q);
            const int off = LAY == RC ? O::at(pr, pc) : O::at(pc, pr);
            u32x2 h[W], m[W], l[W];
#pragma unroll
            for (int w = 0; w < W; w++) split4(v[q + w], h[w], m[w], l[w]);
            auto st = [&](int plane, const u32x2 (&x)[W]) {
                char *d = L + plane * O::PLANE + off;
                if constexpr (W == 2)
                    *reinterpret_cast<u32x4 *>(d) = __builtin_shufflevector(x[0], x[1], 0, 1, 2, 3);
                else
                    *reinterpret_cast<u32x2 *>(d) = x[0];
            };
            st(0, h);
            st(1, m);
            st(2, l);
        }
    }
};

// The three pieces of one 32-wide block for a 16-step MFMA: lane (o, h) feeds
// steps r0 + 8 h + [0, 8) of output index o.
template <int LAY, int OUTER, int BK>
__device__ __forceinline__ void read_frag(const char *__restrict__ L, int o_base, int r0, int lane, bf16x8 (&f)[3])
{
    using O = LdsOp<LAY, OUTER, BK>;
    if constexpr (LAY == RC) {
        const char *p = L + O::at(o_base + (lane & 31), r0 + 8 * (lane >> 5));
#pragma unroll
        for (int x = 0; x < 3; x++) f[x] = *reinterpret_cast<const bf16x8 *>(p + x * O::PLANE);
    } else {
        // ds_read_b64_tr_b16: the 16 lanes of a group read 4 rows of 16
        // columns (lane i: row i / 4, columns 4 (i % 4) + [0, 4)) and lane i
        // receives column i's 4 rows
        const char *p = L + O::at(o_base + 16 * ((lane >> 4) & 1) + 4 * (lane & 3),
                                  r0 + 8 * (lane >> 5) + ((lane & 15) >> 2));
#pragma unroll
        for (int x = 0; x < 3; x++) {
            const s16x4 lo = lds_read_tr(p + x * O::PLANE), hi = lds_read_tr(p + x * O::PLANE + 4 * O::PITCH);
            const s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            f[x] = __builtin_bit_cast(bf16x8, v);
        }
    }
}

// Tile geometry.  The NW waves of a workgroup form a WGM x WGN grid over the
// BM x BN tile and WK groups along the reduction: with WK > 1 every wave
// computes its (BM/WGM) x (BN/WGN) sub-tile over RW = BK/WK of each stage's
// reduction steps, and the WK partial sub-tiles are summed through LDS in
// fixed order at the end.  WK > 1 puts several waves on a tile too small to
// share (one workgroup per CU).
template <int BM_, int BN_, int BK_, int WGM_, int WK_, int NR_ = 2, int NW_ = 4>
struct Tile {
    static constexpr int BM = BM_, BN = BN_, BK = BK_, WGM = WGM_, WK = WK_, NR = NR_;
    // instruction order of a stage (sched_step): 0 = the compiler's; Sched<>
    // below selects the others
    static constexpr int SCH = 0;
    static constexpr int NW = NW_, THREADS = 64 * NW_;      // waves / threads per workgroup
    static constexpr int WGN = NW / (WGM * WK);
    static constexpr int WM = BM / WGM, WN = BN / WGN, FM = WM / 32, FN = WN / 32;
    static constexpr int RW = BK / WK;
    // accumulators per 32x32 block: the large products' and the small ones',
    // added at the store
    static constexpr int NCH = 2;
    static_assert(WGM * WGN * WK == NW && FM >= 1 && FN >= 1, "NW waves, 32x32 blocks");
    static_assert(RW == 16, "a wave takes one 16-step MFMA of each stage");
    static constexpr int TILE = BM * BN;
    template <int LA, int LB>
    static constexpr int stage_lds() { return 2 * (LdsOp<LA, BM, BK>::BYTES + LdsOp<LB, BN, BK>::BYTES) / 4; }
    static constexpr int red_lds() { return WK > 1 ? WK * TILE : 0; }
    static constexpr int mx(int a, int b) { return a > b ? a : b; }
    template <int LA, int LB>
    static constexpr int lds() { return mx(stage_lds<LA, LB>(), red_lds()); }
    static constexpr int lds_max() { return mx(mx(lds<RC, OC>(), lds<RC, RC>()), lds<OC, OC>()); }
    __device__ static int wave() { return threadIdx.x >> 6; }
    __device__ static int wk() { return wave() / (WGM * WGN); }
    __device__ static int wm() { return (wave() % (WGM * WGN)) / WGN; }
    __device__ static int wn() { return (wave() % (WGM * WGN)) % WGN; }
};

// Instruction order inside one stage's scheduling region (between two
// barriers): after the prefetch loads, behind each MFMA an even share of the
// next stage's fragment reads, of the splits and of the LDS stores.  An MFMA
// occupies the matrix core for 32 cycles and its wave's issue for 4, so the 26
// vector instructions that split a float4 run under the MFMAs instead of after
// them.
template <int NM, int VALU, int DSW, int DSR, int I = 0>
__device__ __forceinline__ void sched_mfmas()
{
    if constexpr (I < NM) {
        constexpr int DS_RD = 0x100, DS_WR = 0x200, MFMA = 0x008, VA = 0x002;
        __builtin_amdgcn_sched_group_barrier(MFMA, 1, 0);
        __builtin_amdgcn_sched_group_barrier(DS_RD, DSR * (I + 1) / NM - DSR * I / NM, 0);
        __builtin_amdgcn_sched_group_barrier(VA, VALU * (I + 1) / NM - VALU * I / NM, 0);
        __builtin_amdgcn_sched_group_barrier(DS_WR, DSW * (I + 1) / NM - DSW * I / NM, 0);
        sched_mfmas<NM, VALU, DSW, DSR, I + 1>();
    }
}
template <class T, int VALU, int DSW, int DSR>
__device__ __forceinline__ void sched_step()
{
    if constexpr ((T::SCH & 3) != 0) {
        sched_mfmas<T::FM * T::FN * 6, VALU, DSW, DSR>();
    }
}

// A tile shape with options: 1 = a stage's instructions in the order of
// sched_step (else the compiler's), + 4 = the tile's outputs leave with
// nontemporal (streaming) stores.
template <class T, int S>
struct Sched : T {
    static constexpr int SCH = S;
};

// acc += A(i0.., r) B(r, j0..) over r in [rbeg, rend).  A tile's loads run
// NR stages ahead through NR register sets; LDS is double buffered.
// GA: A's rows go through the row map `amap` (RC A: amap[i0 + x] for tile
// row x; OC A: amap[r]).  PB: B is the column pair (B, B2) of TileLoader.
template <class T, int LA, int LB, bool VEC, bool GA = false, bool PB = false>
__device__ __forceinline__ void tile_accumulate(float *__restrict__ smem, const float *__restrict__ A,
                                                const float *__restrict__ B, int lda, int ldb,
                                                int i0, int j0, int Mo, int No, int rbeg, int rend,
                                                f32x16 (&acc)[T::FM][T::FN][T::NCH],
                                                const int *__restrict__ amap = nullptr,
                                                const float *__restrict__ B2 = nullptr)
{
    constexpr int BM = T::BM, BN = T::BN, BK = T::BK, RW = T::RW;
    constexpr int SA = LdsOp<LA, BM, BK>::BYTES, SB = LdsOp<LB, BN, BK>::BYTES;
    char *lds = reinterpret_cast<char *>(smem);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wm = T::wm(), wn = T::wn(), rb = T::wk() * RW;
    if (rend <= rbeg) return;
    // whole stages; then one with a tail, if any (every stage is taken as one
    // where rows are shorter than a chunk)
    const bool narrow = !VEC && ((LA == OC && Mo < 4) || (LB == OC && No < 4));
    const int nfull = narrow ? 0 : (rend - rbeg) / BK;

    // Every prefetch is issued unconditionally: a stage past the end re-reads
    // the last whole stage's (in-bounds) addresses and is never used.  Loads
    // under a branch would leave the compiler unsure how many are outstanding
    // where the paths meet, and it would then wait for all of them, the
    // prefetch included, before every LDS store.
    auto stage = [&](int st) { return min(st, nfull - 1) * BK; };
    using LoadA = TileLoader<LA, BM, BK, VEC, T::THREADS, GA, false>;
    using LoadB = TileLoader<LB, BN, BK, VEC, T::THREADS, false, PB>;
    typename LoadA::Ptr pa;
    typename LoadB::Ptr pb;
    pa.init(A, lda, i0, Mo, rbeg, rend, tid, amap, nullptr);
    pb.init(B, ldb, j0, No, rbeg, rend, tid, nullptr, B2);

    // a b = ah bh + (ah bm + am bh) + (ah bl + am bm + al bh) + what lies below
    // 2^-25 of the product: six bf16 MFMAs, each product exact in fp32.  The
    // large terms have an accumulator of their own: rounding the small ones
    // into it as well would cost it six roundings per 16 steps instead of one.
    struct Frags { bf16x8 a[T::FM][3], b[T::FN][3]; };
    auto read = [&](Frags &f, const char *L) {
#pragma unroll
        for (int a = 0; a < T::FM; a++) read_frag<LA, BM, BK>(L, wm * T::WM + a * 32, rb, lane, f.a[a]);
#pragma unroll
        for (int b = 0; b < T::FN; b++) read_frag<LB, BN, BK>(L + SA, wn * T::WN + b * 32, rb, lane, f.b[b]);
    };
    auto compute = [&](const Frags &f) {
        constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB_[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int p = 0; p < 6; p++)
#pragma unroll
            for (int a = 0; a < T::FM; a++)
#pragma unroll
                for (int b = 0; b < T::FN; b++)
                    acc[a][b][p < 5] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[a][PA[p]], f.b[b][PB_[p]],
                                                                              acc[a][b][p < 5], 0, 0, 0);
    };

    // A stage passes through the register set st % NR (its fp32 values, loaded
    // NR - 1 steps ahead), LDS buffer st & 1 (its bf16 pieces) and fragment
    // set st & 1.  Step st reads stage st + 1's fragments, computes stage st
    // from the ones read a step earlier and, between its MFMAs, splits stage
    // st + 2 into the LDS buffer whose fragments are already in registers: no
    // wait stands between the step's barrier and its MFMAs.  Past the last
    // stage the same steps run on re-read data that nothing uses.
    if (nfull > 0) {
        constexpr int NR = T::NR;
        static_assert(NR % 2 == 0, "fragment sets alternate within a round");
        LoadA la[NR];
        LoadB lb[NR];
        Frags fr[2];
        auto fetch = [&](LoadA &a, LoadB &b, int st) {
            const int dr = stage(st);
            a.template load<false>(pa, rbeg + dr, dr, tid);
            a.prep(pa, rbeg + stage(st + NR), tid);   // the map rows of its next stage
            b.template load<false>(pb, rbeg + dr, dr, tid);
        };
        auto put = [&](LoadA &a, LoadB &b, int st) {
            a.align(pa, tid);
            b.align(pb, tid);
            char *L = lds + (st & 1) * (SA + SB);
            a.store(L, tid);
            b.store(L + SA, tid);
        };
#pragma unroll
        for (int k = 0; k < NR; k++) la[k].prep(pa, rbeg + stage(k), tid);
#pragma unroll
        for (int k = 0; k < NR; k++) fetch(la[k], lb[k], k);
        put(la[0], lb[0], 0);
        fetch(la[0], lb[0], NR);
        __syncthreads();
        read(fr[0], lds);
        put(la[1], lb[1], 1);
        auto step = [&](int st, int k) {
            __syncthreads();
            fetch(la[(k + 1) % NR], lb[(k + 1) % NR], st + 1 + NR);
            __builtin_amdgcn_sched_barrier(0);        // left alone the scheduler sinks the loads to their use
            read(fr[(k + 1) & 1], lds + ((st + 1) & 1) * (SA + SB));
            compute(fr[k & 1]);
            put(la[(k + 2) % NR], lb[(k + 2) % NR], st + 2);
            sched_step<T, 26 * (LoadA::PER + LoadB::PER) + 8, 3 * (LoadA::PER / LoadA::Ptr::W + LoadB::PER / LoadB::Ptr::W),
                       3 * (T::FM * (LA == OC ? 2 : 1) + T::FN * (LB == OC ? 2 : 1))>();
        };
        int st = 0;
        for (; st + NR <= nfull; st += NR) {
#pragma unroll
            for (int k = 0; k < NR; k++) step(st + k, k);
        }
        // The sums stay in their registers here: one-block waves copied all of
        // them at the end of every turn (33 moves behind the last MFMA).
#pragma unroll
        for (int n = 0; n < T::FM * T::FN * T::NCH; n++)
            asm("" : "+v"(acc[n / T::NCH / T::FN][n / T::NCH % T::FN][n % T::NCH]));
#pragma unroll
        for (int k = 0; k < NR - 1; k++)
            if (st + k < nfull) step(st + k, k);
        // The loads past the end have come in: left outstanding, each store of
        // an epilogue that takes their registers would wait for them, and with
        // them for the store before it.
        __builtin_amdgcn_s_waitcnt(0x0f70);           // vmcnt(0)
        __syncthreads();
    }
    for (int r0 = rbeg + nfull * BK; r0 < rend; r0 += BK) {
        LoadA a;
        LoadB b;
        Frags f;
        a.prep(pa, r0, tid);
        a.template load<true>(pa, r0, r0 - rbeg, tid);
        b.template load<true>(pb, r0, r0 - rbeg, tid);
        a.store(lds, tid);
        b.store(lds + SA, tid);
        __syncthreads();
        read(f, lds);
        compute(f);
        __syncthreads();
    }
}

// One segment's share of a 32x32 block that this wave owns, in plain fp32 on
// the fp32 matrix cores, operands straight from memory: steps [rbeg, rend) as
// the wave's reduction group takes them (RW of each BK), eight MFMAs of two
// steps per sixteen.  pa / pb: this lane's output index of A / B (lane & 31),
// at step 0.  GA: A's reduction rows go through the map.  Operands are taken
// times `scale`.
template <int LAY>
__device__ __forceinline__ const float *lane_base(const float *P, int o, int ld)
{
    return LAY == RC ? P + (size_t)o * ld : P + o;
}
template <class T, int LA, int LB, bool GA = false>
__device__ __forceinline__ void fp32_block(f32x16 &c, const float *__restrict__ pa, const float *__restrict__ pb,
                                           int lda, int ldb, int rbeg, int rend, float scale,
                                           const int *__restrict__ amap = nullptr)
{
    const int h8 = 8 * ((threadIdx.x & 63) >> 5);
    auto at_a = [&](int r) { return (LA == RC ? pa[r] : pa[(size_t)(GA ? amap[r] : r) * lda]) * scale; };
    auto at_b = [&](int r) { return (LB == RC ? pb[r] : pb[(size_t)r * ldb]) * scale; };
#pragma nounroll
    for (int r0 = rbeg + T::wk() * T::RW; r0 < rend; r0 += T::BK) {
        float a[8], b[8];
        const int r = r0 + h8;
        if (r0 + T::RW <= rend) {
#pragma unroll
            for (int k = 0; k < 8; k++) a[k] = at_a(r + k), b[k] = at_b(r + k);
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int rc = min(r + k, rend - 1);
                a[k] = at_a(rc);
                b[k] = at_b(rc);
                if (r + k >= rend) a[k] = b[k] = 0.f;
            }
        }
#pragma unroll
        for (int k = 0; k < 8; k++) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[k], b[k], c, 0, 0, 0);
    }
}

// Outputs that came out infinite or NaN, again in plain fp32.  An operand that
// is not finite (or from 2^112 on) has no split: its pieces turn every sum they
// enter into NaN where fp32 has infinities, or finite sums.  block(c, i, jt,
// scale): c += scale^2 times the wave's share of the 32x32 block in which this
// lane's rows of A and B are row i and tile column jt.  What is still not finite is summed once more at
// 2^-140: the fp32 MFMA rounds a product that is out of range to infinity, and
// two of them that cancel to NaN.  No wave waits for another here, and finite
// tiles only look.
// 8192 x 384 x 2048, fwd / dX / dW us: finite 81 / 99 / 95; one NaN in each
// operand 200 / 403 / 570, NaN everywhere 410 / 510 / 646 (one lane per output,
// 1436 / 4839 / 8101 and 5348 / 15192 / 17235).
//
// A reduction of one or two `steps` is summed here whatever its sums are: six
// piece products round a lone product worse than fp32 does (off by up to 9.6e-8
// of it, 6.0e-8 in fp32; two steps 1.29e-7 and 1.14e-7; from three on better).
template <class T, class Block>
__device__ __forceinline__ void tile_fix(f32x16 (&sum)[T::FM][T::FN], int i0, int Mo, int steps, Block block)
{
    auto finite = [](float x) { return fabsf(x) <= 3.402823466e38f; };
    unsigned need = 0;                                // blocks with a sum that is not finite
#pragma unroll
    for (int n = 0; n < T::FM * T::FN; n++) {
        float z = 0.f;                                // NaN if any is not
#pragma unroll
        for (int v = 0; v < 16; v++) z = fmaf(sum[n / T::FN][n % T::FN][v], 0.f, z);
        if (steps <= 2 || __any(z != z)) need |= 1u << n;
    }
    if (!need) return;
    const int o = threadIdx.x & 31;
#pragma nounroll
    for (int n = 0; n < T::FM * T::FN; n++) {
        if (!(need >> n & 1u)) continue;
        const int i = min(i0 + T::wm() * T::WM + n / T::FN * 32 + o, Mo - 1), jt = T::wn() * T::WN + n % T::FN * 32 + o;
#pragma nounroll
        for (float scale = 1.f, back = 1.f;; scale = 0x1p-70f, back = 0x1p70f) {
            f32x16 c = {};
            block(c, i, jt, scale);
            bool wild = false;
#pragma unroll
            for (int k = 0; k < T::FM * T::FN; k++)
                if (k == n) {
                    auto &x = sum[k / T::FN][k % T::FN];
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        if (!finite(x[v]) || (steps <= 2 && back == 1.f)) x[v] = c[v] * back * back;
                        wild |= !finite(x[v]);
                    }
                }
            if (back > 1.f || !__any(wild)) break;
        }
    }
}

// put(i, j, v, e) for every element (i, j) of the tile's valid part (i < Mo,
// j < No), v its sum and e = pre(i, j) what the epilogue reads from memory for
// it (pre sees clamped, valid indices).  A thread's reads are all issued
// before its first put: the compiler cannot move a read above another
// element's store, so read and stored one by one every element waited out a
// memory round trip, 16 in a row per 32x32 block (residual adds, m8: Wo 25.7 ->
// 20.7 us, W2 48.6 -> 42.8).
// 32x32 MFMA result layout: lane l, register v holds row 8*(v/4) + 4*(l/32) +
// v%4, column l%32.  With WK > 1 the wave groups' partial tiles go through
// `red` (LDS, WK*BM*BN floats, free once tile_accumulate has returned) and are
// summed in wave-group order, so the result does not depend on timing.
// STASH: every element's value (valid or not) is also left in red[f], f its
// fragment-order index (below), for a row-wise epilogue after the next
// barrier; red must hold TILE floats.
struct NoPre {
    struct E {};
    __device__ __forceinline__ E operator()(int, int) const { return E{}; }
};
template <class T, bool STASH = false, class Pre, class Put>
__device__ __forceinline__ void tile_epi(const f32x16 (&acc)[T::FM][T::FN], int Mo, int No, int i0, int j0,
                                         float *__restrict__ red, Pre pre, Put put)
{
    const int lane = threadIdx.x & 63;
    using E = decltype(pre(0, 0));
    if constexpr (T::WK == 1) {
        const int wm = T::wm(), wn = T::wn();
        const int h = lane >> 5, col = lane & 31;
        if constexpr (STASH) {
            const int g = T::wave() % (T::WGM * T::WGN);
#pragma unroll
            for (int a = 0; a < T::FM; a++)
#pragma unroll
                for (int b = 0; b < T::FN; b++)
#pragma unroll
                    for (int v = 0; v < 16; v++)
                        red[(((g * T::FM + a) * T::FN + b) * 16 + v) * 64 + lane] = acc[a][b][v];
        }
#pragma unroll
        for (int a = 0; a < T::FM; a++)
#pragma unroll
            for (int b = 0; b < T::FN; b++) {
                const int j = j0 + wn * T::WN + b * 32 + col, ib = i0 + wm * T::WM + a * 32 + 4 * h;
                E e[16];
#pragma unroll
                for (int v = 0; v < 16; v++) e[v] = pre(min(ib + 8 * (v >> 2) + (v & 3), Mo - 1), min(j, No - 1));
                // all in: else a path of the kernel that reads nothing would
                // wait before each of its stores for these registers, and so
                // for the store before it (64x64 mm 14.4 -> 15.7 us)
                if constexpr (!__is_empty(E)) __builtin_amdgcn_s_waitcnt(0x0f70);      // vmcnt(0)
                if (j >= No) continue;
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int i = ib + 8 * (v >> 2) + (v & 3);
                    if (i < Mo) put(i, j, acc[a][b][v], e[v]);
                }
            }
    } else {
        // fragment-order index of (wave-in-group g, a, b, v, lane) <-> element
        constexpr int IT = T::TILE / T::THREADS;
        static_assert(T::TILE % T::THREADS == 0, "whole rounds");
        auto row_of = [&](int f) {
            const int gg = (f >> 10) / (T::FN * T::FM), a = ((f >> 10) / T::FN) % T::FM, v = (f >> 6) & 15;
            return i0 + (gg / T::WGN) * T::WM + a * 32 + 8 * (v >> 2) + 4 * ((f >> 5) & 1) + (v & 3);
        };
        auto col_of = [&](int f) {
            const int gg = (f >> 10) / (T::FN * T::FM);
            return j0 + (gg % T::WGN) * T::WN + ((f >> 10) % T::FN) * 32 + (f & 31);
        };
        E e[IT];
#pragma unroll
        for (int q = 0; q < IT; q++) {
            const int f = threadIdx.x + q * T::THREADS;
            e[q] = pre(min(row_of(f), Mo - 1), min(col_of(f), No - 1));
        }
        const int g = T::wave() % (T::WGM * T::WGN);
        float *mine = red + T::wk() * T::TILE;
#pragma unroll
        for (int a = 0; a < T::FM; a++)
#pragma unroll
            for (int b = 0; b < T::FN; b++)
#pragma unroll
                for (int v = 0; v < 16; v++)
                    mine[(((g * T::FM + a) * T::FN + b) * 16 + v) * 64 + lane] = acc[a][b][v];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < IT; q++) {
            const int f = threadIdx.x + q * T::THREADS;
            float s = red[f];
#pragma unroll
            for (int k = 1; k < T::WK; k++) s += red[k * T::TILE + f];
            const int i = row_of(f), j = col_of(f);
            if (i < Mo && j < No) put(i, j, s, e[q]);
            if constexpr (STASH) red[f] = s;     // only this thread reads slot f of slice 0
        }
        __syncthreads();            // `red` aliases the stage buffers of the next tile
    }
}

// One output element of a tile: a streaming store for the Sched<T, 4 + ..>
// shapes (it goes past the L2, so the kernel's end does not wait to write
// back lines the next launch reads through another XCD's L2 anyway).
template <class T>
__device__ __forceinline__ void st_out(float *p, float v)
{
    if constexpr ((T::SCH & 4) != 0) __builtin_nontemporal_store(v, p);
    else *p = v;
}

// C (beta ? += : =) acc for the valid part of the tile.
template <class T>
__device__ __forceinline__ void tile_store(const f32x16 (&acc)[T::FM][T::FN], float *__restrict__ C, int ldc, int beta,
                                           int Mo, int No, int i0, int j0, float *__restrict__ red)
{
    if (beta)
        tile_epi<T>(acc, Mo, No, i0, j0, red, [&](int i, int j) { return C[(size_t)i * ldc + j]; },
                    [&](int i, int j, float v, float c) { st_out<T>(C + (size_t)i * ldc + j, c + v); });
    else
        tile_epi<T>(acc, Mo, No, i0, j0, red, NoPre(),
                    [&](int i, int j, float v, NoPre::E) { st_out<T>(C + (size_t)i * ldc + j, v); });
}

// C = acc (beta 0) and, for every 32-column block of each valid row, the dot
// product of the block with the same block of O:  out[i][j / 32] =
// sum_{c < 32} C[i][32 (j / 32) + c] O[i][32 (j / 32) + c] (O with C's row
// stride, out [Mo][No / 32]).  This is the attention backward's per-row term
// D = dO . O of each 32-wide head (tinylm.c:750-768) formed where dO is made
// (the O-projection backward's dX tile), in the dQ item's order: two 16-term
// fma chains, then their sum.  Needs No % 32 == 0 and TILE <= the LDS the
// tile's stages use (every shape but the 128 x 128 ones; the host checks).
template <class T>
__device__ __forceinline__ void tile_store_dot(const f32x16 (&acc)[T::FM][T::FN], float *__restrict__ C, int ldc, int Mo,
                                               int No, int i0, int j0, const float *__restrict__ O,
                                               float *__restrict__ out, float *__restrict__ red)
{
    if constexpr (T::TILE <= T::lds_max()) {
        tile_epi<T, true>(acc, Mo, No, i0, j0, red, NoPre(),
                          [&](int i, int j, float v, NoPre::E) { st_out<T>(C + (size_t)i * ldc + j, v); });
        __syncthreads();
        // eight lanes per (row, block), lane q holding float4 q of the block
        // (a wave's O loads: eight 128-byte row segments); each half's chain
        // passes through its four lanes in order, lane q continuing the sum
        // lane q - 1 ended with.  Every count here is a multiple of 64, so
        // whole waves take part in the shuffles.
        constexpr int NB = T::BN / 32;
        static_assert(T::BM * NB * 8 % 64 == 0, "whole waves");
        const int q = threadIdx.x & 7;
        for (int p8 = threadIdx.x; p8 < T::BM * NB * 8; p8 += T::THREADS) {
            const int p = p8 >> 3, row = p / NB, cb = p % NB;
            const int i = i0 + row, jb = j0 + cb * 32;
            // fragment-order index of (row, column 0 of block cb)
            const int rr = row % T::WM, a = rr / 32, r32 = rr % 32;
            const int v = 4 * (r32 >> 3) + (r32 & 3), hb = (r32 >> 2) & 1;
            const int b = ((cb * 32) % T::WN) / 32;
            const int g = (row / T::WM) * T::WGN + (cb * 32) / T::WN;
            const f32x4 x = *reinterpret_cast<const f32x4 *>(
                red + ((((g * T::FM + a) * T::FN + b) * 16 + v) * 64 + hb * 32) + 4 * q);
            const int ic = min(i, Mo - 1), jc = min(jb, No - 32);
            const f32x4 y = *reinterpret_cast<const f32x4 *>(O + (size_t)ic * ldc + jc + 4 * q);
            float d = 0.f;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const float in = __shfl_up(d, 1, 4);
                if ((q & 3) == s) {
                    float c = s ? in : 0.f;
                    c += x[0] * y[0];
                    c += x[1] * y[1];
                    c += x[2] * y[2];
                    c += x[3] * y[3];
                    d = c;
                }
            }
            const float h0 = __shfl_up(d, 4, 8);
            if (q == 7 && i < Mo && jb < No) out[(size_t)i * (No / 32) + jb / 32] = h0 + d;
        }
        __syncthreads();
    }
}

// 1 / (1 + e^-z) with the hardware exp2 and reciprocal (within a few ulp of
// the reference's expf and division; e^-z = inf gives 0, as there).
__device__ __forceinline__ float hw_sigmoid(float z)
{
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * -1.44269504088896341f));
}

// LDS of an expert-launch workgroup: the tile's stages or partials, and the
// SwiGLU epilogue's staged tile beside the partials.
template <class T>
__host__ __device__ constexpr int expert_lds()
{
    return T::mx(T::lds_max(), (T::WK > 1 ? T::WK * T::TILE : 0) + T::BM * (T::BN + 1));
}

// SwiGLU epilogue of a paired-column tile (TilePtr PB): the tile's columns
// alternate in groups of U between g = X W1 and u = X W3 of the output columns
// jh + [0, BN/2).  a = silu(g) u  (tinylm.c:786, :882) for i < Mo, j < No, and
// g, u too where Cg / Cu are given.  A wave of block pairs (FN even) holds g
// and u of an element in one lane; else the summed tile goes through LDS
// (after the WK partials, which it must not overlap).  With the pairs in
// registers the launch can run 128x128 tiles: m8 training step 7.64 -> 7.29
// ms, m3 1.905 -> 1.84 ms, both with the epilogues' reads issued together.
template <class T>
__device__ __forceinline__ void tile_swiglu(const f32x16 (&acc)[T::FM][T::FN], float *__restrict__ Ca,
                                            float *__restrict__ Cg, float *__restrict__ Cu, int ldc, int Mo,
                                            int No, int i0, int jh, float *__restrict__ red)
{
    auto emit = [&](int i, int j, float g, float u) {
        if (i >= Mo || j >= No) return;
        const size_t o = (size_t)i * ldc + j;
        st_out<T>(Ca + o, g * hw_sigmoid(g) * u);
        if (Cg) st_out<T>(Cg + o, g);
        if (Cu) st_out<T>(Cu + o, u);
    };
    constexpr int U = pair_unit(T::BN);
    if constexpr (T::WK == 1 && T::FN % 2 == 0 && U == 32) {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int a = 0; a < T::FM; a++)
#pragma unroll
            for (int b = 0; b < T::FN; b += 2)
#pragma unroll
                for (int v = 0; v < 16; v++)
                    emit(i0 + T::wm() * T::WM + a * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3),
                         jh + (T::wn() * T::WN + b * 32) / 2 + (lane & 31), acc[a][b][v], acc[a][b + 1][v]);
    } else {
        constexpr int H = T::BN / 2, LD = T::BN + 1;
        constexpr int OFF = T::WK > 1 ? T::WK * T::TILE : 0;
        static_assert(OFF + T::BM * LD <= expert_lds<T>(), "paired tile fits beside the partials");
        float *L = red + OFF;
        tile_epi<T>(acc, T::BM, T::BN, 0, 0, red, NoPre(),
                    [&](int i, int j, float v, NoPre::E) { L[i * LD + j] = v; });
        __syncthreads();
        for (int f = threadIdx.x; f < T::BM * H; f += T::THREADS) {
            const int x = f / H, c = f % H, t = c / U * 2 * U + c % U;
            emit(i0 + x, jh + c, L[x * LD + t], L[x * LD + t + U]);
        }
        __syncthreads();
    }
}

// The tile's sums: what the large products' and the small ones' accumulators hold
// (of operands times 2^16).
template <class T>
__device__ __forceinline__ void tile_sum(const f32x16 (&acc)[T::FM][T::FN][T::NCH], f32x16 (&sum)[T::FM][T::FN])
{
#pragma unroll
    for (int a = 0; a < T::FM; a++)
#pragma unroll
        for (int b = 0; b < T::FN; b++) sum[a][b] = (acc[a][b][0] + acc[a][b][1]) * 0x1p-32f;
}

template <int FM, int FN, int NCH>
__device__ __forceinline__ void zero_acc(f32x16 (&acc)[FM][FN][NCH])
{
#pragma unroll
    for (int a = 0; a < FM; a++)
#pragma unroll
        for (int b = 0; b < FN; b++)
#pragma unroll
            for (int c = 0; c < NCH; c++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[a][b][c][v] = 0.f;
}

// ------------------------------------------------------- single problem --
struct GemmArgs {
    const float *A;
    const float *B;
    float *C;
    int Mo, No, R;
    int lda, ldb, ldc;
    int beta;
    int tiles_n;     // tiles along No
    int tiles;       // tiles_m * tiles_n
    int splits;      // workgroups per tile along r
    int rps;         // r per split (multiple of BK)
    float *ws;       // splits x Mo x No partials (splits > 1)
};

template <class T, int LA, int LB, bool VEC>
__global__ __launch_bounds__(T::THREADS) void k_gemm(GemmArgs g)
{
    __shared__ __attribute__((aligned(16))) float smem[T::template lds<LA, LB>()];
    const int item = xcd_remap(blockIdx.x, gridDim.x);
    const int z = item / g.tiles, tile = item % g.tiles;
    const int i0 = (tile / g.tiles_n) * T::BM, j0 = (tile % g.tiles_n) * T::BN;
    const int rbeg = z * g.rps;
    const int rend = min(g.R, rbeg + g.rps);
    f32x16 acc[T::FM][T::FN][T::NCH], sum[T::FM][T::FN];
    zero_acc(acc);
    tile_accumulate<T, LA, LB, VEC>(smem, g.A, g.B, g.lda, g.ldb, i0, j0, g.Mo, g.No, rbeg, rend, acc);
    tile_sum<T>(acc, sum);
    tile_fix<T>(sum, i0, g.Mo, g.R, [&](f32x16 &c, int i, int jt, float scale) {
        fp32_block<T, LA, LB>(c, lane_base<LA>(g.A, i, g.lda), lane_base<LB>(g.B, min(j0 + jt, g.No - 1), g.ldb),
                              g.lda, g.ldb, rbeg, rend, scale);
    });
    // a split writes its partial (beta 0) into workspace slice z
    if (g.splits > 1)
        tile_store<T>(sum, g.ws + (size_t)z * g.Mo * g.No, g.No, 0, g.Mo, g.No, i0, j0, smem);
    else
        tile_store<T>(sum, g.C, g.ldc, g.beta, g.Mo, g.No, i0, j0, smem);
}

// C (beta ? += : =) sum_{z < splits} ws[z], in z order; Mo x No elements, the
// ones of [e0, e1) here, four to a thread where rows are whole float4s.  The
// slices' loads go out eight at a time (slices past the last re-read it and
// are not added): one by one, each waits out a memory round trip.  Against one
// value and one slice at a time: m8 training step 7.29 -> 6.62 ms, m3 1.85 ->
// 1.71, MoE layer 231 -> 219 us, (8192, 384, 2048) fwd + dX + dW 248 -> 236 us.
template <class V>
__device__ __forceinline__ void reduce_vec(const float *__restrict__ ws, float *__restrict__ C, int No, int ldc,
                                           int splits, int beta, size_t e0, size_t e1, size_t n)
{
    constexpr int W = sizeof(V) / 4;
    for (size_t e = e0 + W * threadIdx.x; e < e1; e += W * blockDim.x) {
        const size_t i = e / (size_t)No, j = e % (size_t)No;
        V *p = reinterpret_cast<V *>(C + i * (size_t)ldc + j);
        V c, s;
        if (beta) c = *p;
        for (int z0 = 0; z0 < splits; z0 += 8) {
            V x[8];
#pragma unroll
            for (int k = 0; k < 8; k++) x[k] = *reinterpret_cast<const V *>(ws + (size_t)min(z0 + k, splits - 1) * n + e);
            if (z0 == 0) s = x[0];
            else s += x[0];
#pragma unroll
            for (int k = 1; k < 8; k++)
                if (z0 + k < splits) s += x[k];
        }
        *p = beta ? c + s : s;
    }
}
__device__ __forceinline__ void reduce_range(const float *__restrict__ ws, float *__restrict__ C, int No, int ldc,
                                             int splits, int beta, size_t e0, size_t e1, size_t n)
{
    if (No % 4 == 0 && ldc % 4 == 0 && ((uintptr_t)C & 15) == 0 && ((uintptr_t)ws & 15) == 0)
        reduce_vec<f32x4>(ws, C, No, ldc, splits, beta, e0, e1, n);
    else
        reduce_vec<float>(ws, C, No, ldc, splits, beta, e0, e1, n);
}

// ------------------------------------------------------ grouped problems --
enum { PK_NN = 0, PK_NT = 1, PK_TN = 2, PK_RED = 3, PK_ZERO = 4, PK_COLSUM = 5 };
#define TLG_ZERO_CHUNK 4096          // floats a clear's work item sets to 0
#define TLG_MAXSEG 3
#define TLG_MAXPROB 16                // group_item pins 16 counts
#define TLG_RED_CHUNK 1024
#define TLG_ERED_CHUNK 2048            // elements per work item of an expert reduction

struct Seg { const float *A, *B; int R, lda, ldb; };
// The fields every work item reads lie in the first 160 bytes (C to items,
// then the segments), so a workgroup fetches them in a few scalar loads
// issued together.
struct Prob {
    float *C;
    const float *ws;      // PK_RED: partials; split GEMM: its partial slice base
    int Mo, No, ldc, beta;
    int kind, nseg;
    int tiles_n, tiles, splits, rps;
    int items;            // work items: tiles * splits, or reduction chunks
    Seg seg[TLG_MAXSEG];
    // Expert-batched problem (nexp > 0): the rows of a top-1 MoE layer are
    // grouped by expert, expert e owning rows [eoff[e], eoff[e+1]) of every
    // row operand.  NN / NT: the output rows are expert rows and the weight
    // operand B of expert e is B + e*es.  TN: the reduction runs over expert
    // rows in slices of rps, and the output of expert e is C + e*es.  `unit`
    // is the row extent of one item (BM for NN / NT, rps for TN).
    const int *eoff;
    long long es;
    int nexp, unit;
    // Fused forms of the MoE expert GEMMs (tinylm.c:876-888, :911-927):
    //   amap  A rows gathered through it (the sorted row -> token index)
    //   B2    NN: second weight of a column pair (W3 beside W1), SwiGLU
    //         epilogue; tiles_n then counts BN/2-column tiles
    //   epi   TLG_EPI_*: plain store, SwiGLU (C = a, X1 = g, X2 = u when
    //         given), SwiGLU backward (da from the tile, g / u in X1 / X2
    //         replaced by dg / du; C unused), or the top-1 combine (C = out,
    //         out[omap[i]] = fin[..] + gate[..] * tile row i; X1 = the rows
    //         themselves, sorted order, when given); on a dense NT problem
    //         ROWDOT: C stored, and X1 [Mo][No/32] the dot of each row's
    //         32-column blocks with those of `fin` (tile_store_dot)
    const int *amap, *omap;
    const float *B2;
    float *X1, *X2;
    const float *fin, *gate;
    int epi;
};
// items / devcount: filled from p[] by group_seal() before every launch (0
// past nprob), so the search for a workgroup's problem reads one contiguous
// block of counts instead of one problem struct after another.
struct GroupArgs {
    int nprob;
    int rows1;            // expert launches: > 0 = one expert owning rows [0, rows1)
    int items[TLG_MAXPROB];
    unsigned devcount;    // bit p: problem p's count is known only on the device (experts)
    Prob p[TLG_MAXPROB];
};

// Real work items of an expert-batched problem, from the device-resident
// row offsets: sum over experts of ceil(rows_e / unit) row units, times the
// column tiles (NN / NT) or the output tiles (TN).
__device__ __forceinline__ int expert_items(const Prob &P, const int *eo)
{
    int units = 0;
    for (int e = 0; e < P.nexp; e++) {
        const int c = eo[e + 1] - eo[e];
        units += c > 0 ? (c + P.unit - 1) / P.unit : 0;
    }
    return units * (P.kind == PK_TN ? P.tiles : P.tiles_n);
}

// Item -> (expert e, row unit t of that expert, first partial slot of e).
// Returns false when the item is past the experts' real work.
__device__ __forceinline__ bool expert_of(const Prob &P, const int *eo, int t, int *e_out, int *t_out,
                                          int *base, int *rows, int *slot0)
{
    int slot = 0;
    for (int e = 0; e < P.nexp; e++) {
        const int b = eo[e], c = eo[e + 1] - b;
        const int n = c > 0 ? (c + P.unit - 1) / P.unit : 0;
        if (t < n) { *e_out = e; *t_out = t; *base = b; *rows = c; *slot0 = slot; return true; }
        t -= n;
        slot += n;
    }
    return false;
}

// Accumulation of one expert tile, with its gather / pair form chosen at run
// time (uniform per problem): PB only for NN problems.
template <class T, int LA, int LB>
__device__ __forceinline__ void expert_acc(float *smem, const Prob &P, const Seg &s, const float *A,
                                           const float *B, const int *amap, int i0, int j0, int Mo, int No,
                                           int rbeg, int rend, f32x16 (&acc)[T::FM][T::FN][T::NCH])
{
    if constexpr (LA == RC && LB == OC) {
        if (P.B2) {
            const float *B2 = P.B2 + (B - s.B);
            if (amap)
                tile_accumulate<T, LA, LB, true, true, true>(smem, A, B, s.lda, s.ldb, i0, j0, Mo, No, rbeg,
                                                             rend, acc, amap, B2);
            else
                tile_accumulate<T, LA, LB, true, false, true>(smem, A, B, s.lda, s.ldb, i0, j0, Mo, No, rbeg,
                                                              rend, acc, nullptr, B2);
            return;
        }
    }
    if (amap)
        tile_accumulate<T, LA, LB, true, true>(smem, A, B, s.lda, s.ldb, i0, j0, Mo, No, rbeg, rend, acc, amap);
    else
        tile_accumulate<T, LA, LB, true>(smem, A, B, s.lda, s.ldb, i0, j0, Mo, No, rbeg, rend, acc);
}

template <class T, int LA, int LB>
__device__ __forceinline__ void expert_tile(float *smem, const Prob &P, int local, const int *eo)
{
    f32x16 acc[T::FM][T::FN][T::NCH], sum[T::FM][T::FN];
    int e, t, base, rows, slot0;
    if (P.kind != PK_TN) {
        if (!expert_of(P, eo, local / P.tiles_n, &e, &t, &base, &rows, &slot0)) return;
        // a paired tile covers BN/2 output columns
        const int i0 = t * T::BM, j0 = (local % P.tiles_n) * (P.B2 ? T::BN / 2 : T::BN);
        // combine: the tile rows' tokens and gates, staged before the
        // accumulation so the epilogue waits on one load level, not three
        __shared__ int s_tok[(LA == RC && LB == OC) ? T::BM : 1];
        __shared__ float s_gate[(LA == RC && LB == OC) ? T::BM : 1];
        if constexpr (LA == RC && LB == OC) {
            if (P.epi == TLG_EPI_COMBINE && (int)threadIdx.x < T::BM) {
                const int x = threadIdx.x, n = P.omap[base + min(i0 + x, rows - 1)];
                s_tok[x] = n;
                s_gate[x] = P.gate[n];
            }
        }
        zero_acc(acc);
        for (int k = 0; k < P.nseg; k++) {
            const Seg &s = P.seg[k];
            // gathered: rows of A through amap[base + x]; else A's expert rows
            const float *A = P.amap ? s.A : s.A + (size_t)base * s.lda;
            const int *amap = P.amap ? P.amap + base : nullptr;
            expert_acc<T, LA, LB>(smem, P, s, A, s.B + (size_t)e * P.es, amap, i0, j0, rows, P.No, 0, s.R,
                                  acc);
        }
        tile_sum<T>(acc, sum);
        tile_fix<T>(sum, i0, rows, P.seg[0].R, [&](f32x16 &c, int i, int jt, float scale) {
            // a paired tile's columns alternate between B and B2 (TilePtr PB)
            const bool pair = LA == RC && LB == OC && P.B2;
            constexpr int U = pair_unit(T::BN);
            const int j = min(j0 + (pair ? jt / (2 * U) * U + jt % U : jt), P.No - 1);
            const int am = P.amap ? P.amap[base + i] : base + i;
            for (int k = 0; k < P.nseg; k++) {
                const Seg &s = P.seg[k];
                const float *B = (pair && (jt & U) ? P.B2 : s.B) + (size_t)e * P.es;
                fp32_block<T, LA, LB>(c, lane_base<LA>(s.A, am, s.lda), lane_base<LB>(B, j, s.ldb), s.lda, s.ldb, 0,
                                      s.R, scale);
            }
        });
        const size_t cb = (size_t)base * P.ldc;
        switch (P.epi) {
        case TLG_EPI_SWIGLU:
            tile_swiglu<T>(sum, P.C + cb, P.X1 ? P.X1 + cb : nullptr, P.X2 ? P.X2 + cb : nullptr, P.ldc, rows,
                           P.No, i0, j0, smem);
            break;
        case TLG_EPI_SWIGLU_BWD: {
            // In place: g <- da u silu'(g), u <- da silu(g)  (tinylm.c:923-925)
            float *G = P.X1 + cb, *U = P.X2 + cb;
            const int ld = P.ldc;
            tile_epi<T>(sum, rows, P.No, i0, j0, smem,
                        [&](int i, int j) {
                            const size_t o = (size_t)i * ld + j;
                            return f32x2{G[o], U[o]};
                        },
                        [&](int i, int j, float d, f32x2 gu) {
                            const size_t o = (size_t)i * ld + j;
                            const float z = gu[0], sg = hw_sigmoid(z);
                            const float si = z * sg;
                            const float ds = sg + z * sg * (1.0f - sg);
                            st_out<T>(G + o, d * gu[1] * ds);
                            st_out<T>(U + o, d * si);
                        });
            break;
        }
        case TLG_EPI_COMBINE: {
            // out[n] = fin[n] + gate[n] y  for token n of sorted row i (:870, :886-888)
            if constexpr (LA == RC && LB == OC) {
                __syncthreads();          // the staged tokens, also when the reduction was empty
                const int ld = P.ldc;
                float *C = P.C;
                const float *fin = P.fin;
                float *Y = P.X1 ? P.X1 + cb : nullptr;      // the expert rows too, when kept
                tile_epi<T>(sum, rows, P.No, i0, j0, smem,
                            [&](int i, int j) { return fin[(size_t)s_tok[i - i0] * ld + j]; },
                            [&](int i, int j, float y, float x0) {
                                const int x = i - i0;
                                st_out<T>(C + (size_t)s_tok[x] * ld + j, fmaf(s_gate[x], y, x0));
                                if (Y) st_out<T>(Y + (size_t)i * ld + j, y);
                            });
            }
            break;
        }
        default:
            tile_store<T>(sum, P.C + cb, P.ldc, P.beta, rows, P.No, i0, j0, smem);
        }
    } else {
        if (!expert_of(P, eo, local / P.tiles, &e, &t, &base, &rows, &slot0)) return;
        const int tile = local % P.tiles;
        const int i0 = (tile / P.tiles_n) * T::BM, j0 = (tile % P.tiles_n) * T::BN;
        const int rbeg = base + t * P.unit, rend = min(base + rows, rbeg + P.unit);
        const Seg &s = P.seg[0];
        zero_acc(acc);
        // A's reduction rows are sorted rows; gathered ones map through amap
        expert_acc<T, LA, LB>(smem, P, s, s.A, s.B, P.amap, i0, j0, P.Mo, P.No, rbeg, rend, acc);
        tile_sum<T>(acc, sum);
        tile_fix<T>(sum, i0, P.Mo, rows, [&](f32x16 &c, int i, int jt, float scale) {
            const float *pa = lane_base<LA>(s.A, i, s.lda), *pb = lane_base<LB>(s.B, min(j0 + jt, P.No - 1), s.ldb);
            if (P.amap) fp32_block<T, LA, LB, true>(c, pa, pb, s.lda, s.ldb, rbeg, rend, scale, P.amap);
            else        fp32_block<T, LA, LB>(c, pa, pb, s.lda, s.ldb, rbeg, rend, scale);
        });
        tile_store<T>(sum, (float *)P.ws + (size_t)(slot0 + t) * P.Mo * P.No, P.No, 0, P.Mo, P.No, i0, j0,
                      smem);
    }
}

// Reduction of an expert TN problem: C_e (beta ? += : =) the sum of expert
// e's partial slots, in slot order.
__device__ __forceinline__ void expert_reduce(const Prob &P, int local, const int *eo)
{
    const size_t n = (size_t)P.Mo * P.No;
    const int chunks = (int)((n + TLG_ERED_CHUNK - 1) / TLG_ERED_CHUNK);
    const int e = local / chunks;
    int slot0 = 0;
    for (int k = 0; k < e; k++) {
        const int c = eo[k + 1] - eo[k];
        slot0 += c > 0 ? (c + P.unit - 1) / P.unit : 0;
    }
    const int c = eo[e + 1] - eo[e];
    const int ns = c > 0 ? (c + P.unit - 1) / P.unit : 0;
    const size_t e0 = (size_t)(local % chunks) * TLG_ERED_CHUNK;
    const size_t e1 = e0 + TLG_ERED_CHUNK < n ? e0 + TLG_ERED_CHUNK : n;
    float *C = P.C + (size_t)e * P.es;
    if (ns == 0) {
        if (!P.beta)
            for (size_t i = e0 + threadIdx.x; i < e1; i += blockDim.x) C[i] = 0.f;
        return;
    }
    reduce_range(P.ws + (size_t)slot0 * n, C, P.No, P.No, ns, P.beta, e0, e1, n);
}

template <class T, int LA, int LB, bool EXP>
__device__ __forceinline__ void group_tile(float *smem, const Prob &P, int local, const int *eo)
{
    if constexpr (EXP) {
        if (P.nexp) { expert_tile<T, LA, LB>(smem, P, local, eo); return; }
    }
    const int z = local / P.tiles, tile = local % P.tiles;
    const int i0 = (tile / P.tiles_n) * T::BM, j0 = (tile % P.tiles_n) * T::BN;
    f32x16 acc[T::FM][T::FN][T::NCH], sum[T::FM][T::FN];
    zero_acc(acc);
    if (P.splits > 1) {
        const Seg &s = P.seg[0];
        const int rbeg = z * P.rps, rend = min(s.R, rbeg + P.rps);
        tile_accumulate<T, LA, LB, true>(smem, s.A, s.B, s.lda, s.ldb, i0, j0, P.Mo, P.No, rbeg, rend, acc);
        tile_sum<T>(acc, sum);
        tile_fix<T>(sum, i0, P.Mo, s.R, [&](f32x16 &c, int i, int jt, float scale) {
            fp32_block<T, LA, LB>(c, lane_base<LA>(s.A, i, s.lda), lane_base<LB>(s.B, min(j0 + jt, P.No - 1), s.ldb),
                                  s.lda, s.ldb, rbeg, rend, scale);
        });
        tile_store<T>(sum, (float *)P.ws + (size_t)z * P.Mo * P.No, P.No, 0, P.Mo, P.No, i0, j0, smem);
        return;
    }
    for (int k = 0; k < P.nseg; k++) {
        const Seg &s = P.seg[k];
        tile_accumulate<T, LA, LB, true>(smem, s.A, s.B, s.lda, s.ldb, i0, j0, P.Mo, P.No, 0, s.R, acc);
    }
    tile_sum<T>(acc, sum);
    tile_fix<T>(sum, i0, P.Mo, P.seg[0].R, [&](f32x16 &c, int i, int jt, float scale) {
        for (int k = 0; k < P.nseg; k++) {
            const Seg &s = P.seg[k];
            fp32_block<T, LA, LB>(c, lane_base<LA>(s.A, i, s.lda), lane_base<LB>(s.B, min(j0 + jt, P.No - 1), s.ldb),
                                  s.lda, s.ldb, 0, s.R, scale);
        }
    });
    if (LA == RC && LB == OC && P.fin) {
        // mm with its residual add: C = R + acc (R in `fin`, C's layout)
        float *C = P.C;
        const float *Rr = P.fin;
        const int ld = P.ldc;
        tile_epi<T>(sum, P.Mo, P.No, i0, j0, smem, [&](int i, int j) { return Rr[(size_t)i * ld + j]; },
                    [&](int i, int j, float v, float r) { st_out<T>(C + (size_t)i * ld + j, r + v); });
        return;
    }
    if constexpr (LA == RC && LB == RC) {
        if (P.epi == TLG_EPI_ROWDOT) {
            tile_store_dot<T>(sum, P.C, P.ldc, P.Mo, P.No, i0, j0, P.fin, P.X1, smem);
            return;
        }
    }
    tile_store<T>(sum, P.C, P.ldc, P.beta, P.Mo, P.No, i0, j0, smem);
}

// Work-item mapping of a grouped launch.  The dispatcher deals workgroup b
// to XCD b % 8; XCD x takes an equal contiguous slice of EVERY problem's
// items (so each XCD's L2 sees neighbouring tiles of a problem, and every
// XCD gets the same mix of long and short items), problem by problem in
// list order (the host lists problems longest item first).  Workgroups past
// their XCD's share exit at once.
static_assert(TLG_MAXPROB == 16, "group_item pins exactly 16 item counts");
__device__ __forceinline__ int group_item(const GroupArgs &g, int b, int *local, const int *eo)
{
    const int x = b & 7;
    int slot = b >> 3;
    int cnt[TLG_MAXPROB];
#pragma unroll
    for (int p = 0; p < TLG_MAXPROB; p++) cnt[p] = g.items[p];
    const unsigned dev = g.devcount;
    // every count in flight at once: one round trip, then scalar arithmetic
    // (counts past nprob are 0, so nprob itself is not needed)
    asm volatile("" ::"s"(dev), "s"(cnt[0]), "s"(cnt[1]), "s"(cnt[2]), "s"(cnt[3]), "s"(cnt[4]), "s"(cnt[5]),
                 "s"(cnt[6]), "s"(cnt[7]), "s"(cnt[8]), "s"(cnt[9]), "s"(cnt[10]), "s"(cnt[11]), "s"(cnt[12]),
                 "s"(cnt[13]), "s"(cnt[14]), "s"(cnt[15]));
#pragma unroll
    for (int p = 0; p < TLG_MAXPROB; p++) {
        // expert-batched GEMMs: the real item count, known only on the device
        const int n = (dev >> p & 1u) ? expert_items(g.p[p], eo) : cnt[p];
        const int lo = (x * n) >> 3, hi = ((x + 1) * n) >> 3;
        if (slot < hi - lo) { *local = lo + slot; return p; }
        slot -= hi - lo;
    }
    return -1;
}

// `eo`: the expert row offsets of an expert-batched launch, staged in LDS
// (nullptr for dense launches, which have no expert problems).
// PK_COLSUM: C[0, No) (beta ? += : =) the sum of the `splits` partial rows
// ws[z][0, No) (a row-block reduction queued by tlg_defer_colsum).  Item
// `local` covers float4 columns [4 local, 4 local + 4), one wave per
// column at a time: lane l adds rows l, l + 64, ... in order, then a fixed
// butterfly, so the sum does not depend on timing.
#define TLG_COLSUM_CH 4
__device__ __forceinline__ void colsum(const Prob &P, int local)
{
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6, w = threadIdx.x >> 6;
    const int c4 = P.No >> 2, cend = min(TLG_COLSUM_CH * (local + 1), c4);
    for (int c = TLG_COLSUM_CH * local + w; c < cend; c += nw) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        for (int z = lane; z < P.splits; z += 64) s += reinterpret_cast<const f32x4 *>(P.ws + (size_t)z * P.No)[c];
        for (int o = 32; o > 0; o >>= 1) {
            s.x += __shfl_xor(s.x, o);
            s.y += __shfl_xor(s.y, o);
            s.z += __shfl_xor(s.z, o);
            s.w += __shfl_xor(s.w, o);
        }
        if (lane == 0) {
            f32x4 *out = reinterpret_cast<f32x4 *>(P.C) + c;
            *out = P.beta ? *out + s : s;
        }
    }
}

template <class T, bool EXP>
__device__ __forceinline__ void group_body(const GroupArgs &g, float *smem, const int *eo)
{
    int local = 0;
    const int p = group_item(g, blockIdx.x, &local, eo);
    if (p < 0) return;
    const Prob &P = g.p[p];
    // The fields a tile reads first, fetched together: one round trip to the
    // argument block before the tile's first loads, not one per field.
    asm volatile("" ::"s"(P.kind), "s"(P.nseg), "s"(P.Mo), "s"(P.No), "s"(P.tiles), "s"(P.tiles_n),
                 "s"(P.splits), "s"(P.rps), "s"(P.seg[0].A), "s"(P.seg[0].B), "s"(P.seg[0].R), "s"(P.seg[0].lda),
                 "s"(P.seg[0].ldb));
    switch (P.kind) {
    case PK_NN: group_tile<T, RC, OC, EXP>(smem, P, local, eo); break;
    case PK_NT: group_tile<T, RC, RC, EXP>(smem, P, local, eo); break;
    case PK_TN: group_tile<T, OC, OC, EXP>(smem, P, local, eo); break;
    case PK_COLSUM: colsum(P, local); break;
    case PK_ZERO: {
        const size_t n = (size_t)P.Mo * P.No, e0 = (size_t)local * TLG_ZERO_CHUNK;
        const size_t e1 = e0 + TLG_ZERO_CHUNK < n ? e0 + TLG_ZERO_CHUNK : n;
        for (size_t e = e0 + threadIdx.x; e < e1; e += blockDim.x) P.C[e] = 0.f;
        break;
    }
    default: {
        if constexpr (EXP) {
            if (P.nexp) { expert_reduce(P, local, eo); break; }
        }
        const size_t n = (size_t)P.Mo * P.No;
        const size_t e0 = (size_t)local * TLG_RED_CHUNK;
        const size_t e1 = e0 + TLG_RED_CHUNK < n ? e0 + TLG_RED_CHUNK : n;
        reduce_range(P.ws, P.C, P.No, P.ldc, P.splits, P.beta, e0, e1, n);
    }
    }
}

template <class T>
__global__ __launch_bounds__(T::THREADS) void k_group(GroupArgs g)
{
    __shared__ __attribute__((aligned(16))) float smem[T::lds_max()];
    group_body<T, false>(g, smem, nullptr);
}

// The same code for the expert-batched launches of the MoE layer, under its
// own name so profiles separate MoE launches from the dense grouped GEMMs.
// Every problem of such a launch shares one row-offset array; it is staged in
// LDS once, so finding a work item's expert costs no dependent global loads.
// The fused variants (gathered rows, paired columns, epilogues) are separate
// inlined code paths that share one register allocation: two waves per SIMD
// (64x64 tiles 171 VGPRs at four waves, 128x128 ones 245 at eight).
#define TLG_MAX_EXPERTS 64
template <class T>
__global__ __launch_bounds__(T::THREADS) void k_expert_group(GroupArgs g)
{
    __shared__ __attribute__((aligned(16))) float smem[expert_lds<T>()];
    __shared__ int eo[TLG_MAX_EXPERTS + 1];
    const int E = g.p[0].nexp;
    if (g.rows1 > 0) {
        if (threadIdx.x < 2) eo[threadIdx.x] = threadIdx.x ? g.rows1 : 0;
    } else {
        for (int i = threadIdx.x; i <= E; i += blockDim.x) eo[i] = g.p[0].eoff[i];
    }
    __syncthreads();
    group_body<T, true>(g, smem, eo);
}

// ---------------------------------------------------------------- shapes --
// Tile shapes: BM x BN output per workgroup, BK reduction steps per stage,
// WGM x WGN waves over the tile, WK wave groups along the reduction.
// X(index, BM, BN, BK, WGM, WK, NR, waves, instruction order and stores)
// Indices keep their meaning for the tuning hooks and their tables; a row that
// repeats another runs that one's kernels (tile_canon).
#define TLG_TILES(X) \
    X(0, 128, 128, 16, 2, 1, 2, 4, 0) \
    X(1, 128, 64, 16, 2, 1, 2, 4, 0) \
    X(2, 64, 128, 16, 2, 1, 2, 4, 0) \
    X(3, 64, 64, 16, 2, 1, 2, 4, 0) \
    X(4, 64, 64, 64, 1, 4, 2, 4, 0) \
    X(5, 64, 64, 32, 1, 2, 2, 4, 0) \
    X(6, 64, 128, 32, 1, 2, 2, 4, 0) \
    X(7, 128, 64, 32, 2, 2, 2, 4, 0) \
    X(8, 64, 64, 64, 1, 4, 2, 8, 0) \
    X(9, 128, 128, 16, 2, 1, 2, 8, 0) \
    X(10, 128, 128, 16, 2, 1, 2, 8, 0) \
    X(11, 128, 64, 16, 2, 1, 2, 4, 0) \
    X(12, 128, 64, 32, 2, 2, 2, 8, 0) \
    X(13, 32, 64, 32, 1, 2, 2, 4, 0) \
    X(14, 64, 32, 32, 2, 2, 2, 4, 0) \
    X(15, 32, 32, 64, 1, 4, 2, 4, 0) \
    X(16, 64, 64, 16, 2, 1, 2, 4, 0) \
    X(17, 64, 64, 16, 2, 1, 2, 4, 0) \
    X(18, 128, 64, 16, 2, 1, 4, 4, 1) \
    X(19, 128, 64, 16, 2, 1, 2, 4, 1) \
    X(20, 64, 64, 32, 2, 2, 2, 8, 0) \
    X(21, 64, 32, 64, 2, 4, 2, 8, 0) \
    X(22, 64, 64, 64, 1, 4, 2, 8, 0) \
    X(23, 128, 128, 16, 2, 1, 2, 8, 5) \
    X(24, 64, 64, 16, 2, 1, 2, 4, 1) \
    X(25, 64, 64, 32, 1, 2, 2, 4, 1) \
    X(26, 64, 32, 32, 2, 2, 2, 4, 1) \
    X(27, 64, 64, 32, 2, 2, 2, 8, 1) \
    X(28, 128, 64, 32, 2, 2, 2, 8, 5) \
    X(29, 32, 64, 32, 1, 2, 2, 4, 0) \
    X(30, 32, 32, 64, 1, 4, 2, 4, 0) \
    X(31, 128, 128, 16, 2, 1, 2, 4, 1) \
    X(32, 128, 64, 16, 2, 1, 2, 4, 1) \
    X(33, 128, 128, 16, 2, 1, 2, 8, 1) \
    X(34, 128, 64, 32, 2, 2, 2, 8, 1) \
    X(35, 64, 64, 16, 2, 1, 2, 4, 5) \
    X(36, 64, 64, 64, 1, 4, 2, 8, 1) \
    X(37, 64, 64, 32, 2, 2, 2, 8, 5) \
    X(38, 64, 64, 16, 2, 1, 2, 4, 4) \
    X(39, 64, 64, 16, 2, 1, 4, 4, 4) \
    X(40, 64, 32, 32, 2, 2, 2, 4, 4) \
    X(41, 64, 64, 64, 1, 4, 2, 8, 4) \
    X(42, 64, 64, 32, 2, 2, 2, 8, 4) \
    X(43, 32, 64, 32, 1, 2, 2, 4, 4) \
    X(44, 32, 32, 64, 1, 4, 2, 4, 4) \
    X(45, 128, 128, 16, 2, 1, 2, 4, 4) \
    X(46, 128, 64, 16, 2, 1, 2, 4, 4) \
    X(47, 128, 128, 16, 2, 1, 2, 8, 4) \
    X(48, 64, 64, 32, 1, 2, 2, 4, 4) \
    X(49, 64, 32, 64, 2, 4, 2, 8, 4) \
    X(50, 128, 64, 32, 2, 2, 2, 8, 4)
template <int BM, int BN, int BK, int WGM, int WK, int NR, int NW, int SCH>
struct TileOf { using type = Sched<Tile<BM, BN, BK, WGM, WK, NR, NW>, SCH>; };
template <int BM, int BN, int BK, int WGM, int WK, int NR, int NW>
struct TileOf<BM, BN, BK, WGM, WK, NR, NW, 0> { using type = Tile<BM, BN, BK, WGM, WK, NR, NW>; };

// The row whose kernels row i runs: 11, 22, 29 and 30 repeat the rows that they
// had another order of; 10 (128x128 tiles of 32-step stages, 713 registers
// spilled), 16 and 17 (two waves) and 19 stand in no rule or table and run the
// kept shape of their extents.
__host__ __device__ constexpr int tile_canon(int i)
{
    return i == 10 ? 9 : i == 11 ? 1 : i == 16 || i == 17 ? 3 : i == 19 ? 32 : i == 22 ? 8 : i == 29 ? 13 : i == 30 ? 15 : i;
}
// Shapes that grouped launches take (2 and 5 to 7 are single calls' alone).
__host__ __device__ constexpr bool tile_grouped(int i) { return i != 2 && (i < 5 || i > 7); }

// Shapes of the expert-batched launches: X(key, BM, BN, BK, WGM, WK, waves)
#define TLG_EXPERTS(X) \
    X(3, 64, 64, 16, 2, 1, 4) \
    X(9, 128, 128, 16, 4, 1, 8) \
    X(14, 64, 32, 32, 2, 2, 4) \
    X(15, 32, 32, 64, 1, 4, 4) \
    X(18, 64, 64, 32, 1, 2, 4) \
    X(22, 64, 64, 64, 1, 4, 8)

// Launches of the instances, compiled in parts (tlg_tiles.hip): each returns
// whether its part holds configuration `ci`.
#define TLG_GROUP_PARTS 5
#define TLG_SINGLE 16                 // single-call launches take the first 16 shapes
#define TLG_TILE_PARTS(X) X(0) X(1) X(2) X(3) X(4)
#define TLG_DECL(k) bool tlg_group_part##k(int ci, const GroupArgs &a, int grid, hipStream_t st);
TLG_TILE_PARTS(TLG_DECL)
#undef TLG_DECL
bool tlg_single_part0(int ci, TlgKind kind, bool vec, const GemmArgs &a, int grid, hipStream_t st);
bool tlg_single_part1(int ci, TlgKind kind, bool vec, const GemmArgs &a, int grid, hipStream_t st);
// key: an expert shape, + 200 with streaming stores
bool tlg_expert_part(int key, const GroupArgs &a, int grid, hipStream_t st);
#endif

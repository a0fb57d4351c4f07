// tlg_tiles.hip -- the tile kernels' instances (tlg_tile.h), compiled in parts
// so that a build runs in parallel: TLG_PART 0-4 hold the grouped launches'
// configurations (index modulo 5), 5 and 6 the single-call ones (modulo 2),
// 7 the expert-batched ones.
#include "tlg_tile.h"

#define TLG_CAT_(a, b) a##b
#define TLG_CAT(a, b) TLG_CAT_(a, b)

#if TLG_PART < TLG_GROUP_PARTS
template <int I, class T>
static bool launch_row(int ci, const GroupArgs &a, int grid, hipStream_t st)
{
    if constexpr (I % TLG_GROUP_PARTS == TLG_PART && tile_canon(I) == I && tile_grouped(I)) {
        if (ci == I) {
            hipLaunchKernelGGL((k_group<T>), dim3(grid), dim3(T::THREADS), 0, st, a);
            return true;
        }
    }
    return false;
}
bool TLG_CAT(tlg_group_part, TLG_PART)(int ci, const GroupArgs &a, int grid, hipStream_t st)
{
#define TLG_ROW(i, bm, bn, bk, wgm, wk, nr, nw, sch)                                                             \
    if (launch_row<i, TileOf<bm, bn, bk, wgm, wk, nr, nw, sch>::type>(ci, a, grid, st)) return true;
    TLG_TILES(TLG_ROW)
#undef TLG_ROW
    return false;
}

#elif TLG_PART < TLG_GROUP_PARTS + 2
#define TLG_SPART (TLG_PART - TLG_GROUP_PARTS)
template <class T, int LA, int LB>
static void launch_t(const GemmArgs &a, int grid, bool vec, hipStream_t st)
{
    if (vec) hipLaunchKernelGGL((k_gemm<T, LA, LB, true>), dim3(grid), dim3(T::THREADS), 0, st, a);
    else     hipLaunchKernelGGL((k_gemm<T, LA, LB, false>), dim3(grid), dim3(T::THREADS), 0, st, a);
}
template <int I, class T>
static bool launch_row(int ci, TlgKind kind, bool vec, const GemmArgs &a, int grid, hipStream_t st)
{
    if constexpr (I < TLG_SINGLE && I % 2 == TLG_SPART && tile_canon(I) == I) {
        if (ci == I) {
            if (kind == TLG_NN)      launch_t<T, RC, OC>(a, grid, vec, st);
            else if (kind == TLG_NT) launch_t<T, RC, RC>(a, grid, vec, st);
            else                     launch_t<T, OC, OC>(a, grid, vec, st);
            return true;
        }
    }
    return false;
}
#if TLG_SPART == 0
bool tlg_single_part0(int ci, TlgKind kind, bool vec, const GemmArgs &a, int grid, hipStream_t st)
#else
bool tlg_single_part1(int ci, TlgKind kind, bool vec, const GemmArgs &a, int grid, hipStream_t st)
#endif
{
#define TLG_ROW(i, bm, bn, bk, wgm, wk, nr, nw, sch)                                                             \
    if (launch_row<i, TileOf<bm, bn, bk, wgm, wk, nr, nw, 5>::type>(ci, kind, vec, a, grid, st)) return true;
    TLG_TILES(TLG_ROW)
#undef TLG_ROW
    return false;
}

#else
template <class T>
static void launch_t(const GroupArgs &a, int grid, hipStream_t st)
{
    hipLaunchKernelGGL((k_expert_group<T>), dim3(grid), dim3(T::THREADS), 0, st, a);
}
bool tlg_expert_part(int key, const GroupArgs &a, int grid, hipStream_t st)
{
#define TLG_ROW(k, bm, bn, bk, wgm, wk, nw)                                                                      \
    if (key == k) return launch_t<Sched<Tile<bm, bn, bk, wgm, wk, 2, nw>, 1>>(a, grid, st), true;             \
    if (key == 200 + k) return launch_t<Sched<Tile<bm, bn, bk, wgm, wk, 2, nw>, 5>>(a, grid, st), true;
    TLG_EXPERTS(TLG_ROW)
#undef TLG_ROW
    return false;
}
#endif

// hosttiles.hpp -- TEST-ONLY: the tiles of one launch, executed work-group by work-group and thread by thread
// (hostemu.cpp, hostfused.cpp).
#pragma once

#include "hc_stage.hpp"

#include <cfloat>
#include <cmath>
#include <memory>
#include <vector>

namespace hc {

template <class T, class RF> void run_tiles(const StageArgs<RF>& a)
{
    constexpr int TI = T::TILE_I, TJ = T::TILE_J;
    const int tiles_i = (a.m.ni + TI - 1) / TI, tiles_j = (a.m.nj + TJ - 1) / TJ;
    const int ntiles = tiles_i * tiles_j;
    auto sp = std::make_unique<typename T::Smem>();
    typename T::Smem& s = *sp;
    std::vector<unsigned int> flag(T::NT);
    for (int b = 0; b < ntiles; ++b) {
        const int t = xcd_tile(b, ntiles);
        const int i0 = (t / tiles_j) * TI, j0 = (t % tiles_j) * TJ;
        for (auto& f : flag) f = 0;
        std::vector<typename T::Geo> g0(T::NT);
        for (int tid = 0; tid < T::NT; ++tid) {
            T::load(a, s, i0, j0, tid, flag[tid]);
            T::prefetch(a, i0, j0, tid, g0[tid]);
        }
        for (int tid = 0; tid < T::NT; ++tid) T::qmetric(a, s, i0, j0, tid);
        for (int tid = 0; tid < T::NT; ++tid) T::faces(a, s, i0, j0, tid, flag[tid], g0[tid]);
        std::vector<double> red(T::NT);
        std::vector<typename T::CellIn> ci(T::NT);
        for (int tid = 0; tid < T::NT; ++tid) T::prefetch_cell(a, i0, j0, tid, ci[tid]);
        for (int tid = 0; tid < T::NT; ++tid) T::cells(a, s, i0, j0, tid, flag[tid], red[tid], ci[tid]);
        double m = 0.0;
        unsigned int f = 0;
        for (int tid = 0; tid < T::NT; ++tid) {
            m = fmax(m, red[tid]);
            f |= flag[tid];
        }
        if (a.mode == MODE_GLOBAL_STAGE0 && dbl_bits(m) > *a.maxslot) *a.maxslot = dbl_bits(m);
        *a.status |= f;
    }
    if (a.reset_max) *a.maxslot = dbl_bits(DBL_MIN);
}

// the fused Euler tile (hostfused.cpp): wide with 64-bit offsets, uniform on uniform geometry
void run_fused(int basis, int flux, int shape, bool wide, bool uniform, const StageArgs<double>& a);

}   // namespace hc

// hostfused.cpp -- TEST-ONLY: the fused Euler tile (hc_fused.hpp) of the host emulation, every basis, flux, shape
// and offset width that the library holds.  A file of its own, which compiles beside hostemu.cpp.
#include "hosttiles.hpp"

#include "hc_fused.hpp"
#include "hc_tiles.hpp"

namespace hc {

template <int BASIS, int FLUX, int K> static void run_shape(bool wide, bool uniform, const StageArgs<double>& a)
{
    constexpr TileShape S = TILESF[K], W = TILESW[K];
    if (wide) run_tiles<FusedTile<BASIS, FLUX, W.ti, W.tj, W.nt, unsigned long long, 0>>(a);
    else if (uniform) run_tiles<FusedTile<BASIS, FLUX, S.ti, S.tj, S.nt, unsigned, 1>>(a);
    else run_tiles<FusedTile<BASIS, FLUX, S.ti, S.tj, S.nt, unsigned, 0>>(a);
}

template <int BASIS, int FLUX> static void run_flux(int shape, bool wide, bool uniform, const StageArgs<double>& a)
{
    static_assert(NTILECFG == 3, "one run_shape per tile configuration");
    if (shape == 2) run_shape<BASIS, FLUX, 2>(wide, uniform, a);
    else if (shape == 1) run_shape<BASIS, FLUX, 1>(wide, uniform, a);
    else run_shape<BASIS, FLUX, 0>(wide, uniform, a);
}

template <int BASIS> static void run_basis(int flux, int shape, bool wide, bool uniform, const StageArgs<double>& a)
{
    switch (flux) {
    case 0: run_flux<BASIS, 0>(shape, wide, uniform, a); break;
    case 1: run_flux<BASIS, 1>(shape, wide, uniform, a); break;
    case 4: run_flux<BASIS, 4>(shape, wide, uniform, a); break;
    case 5: run_flux<BASIS, 5>(shape, wide, uniform, a); break;
    default: run_flux<BASIS, 6>(shape, wide, uniform, a); break;
    }
}

void run_fused(int basis, int flux, int shape, bool wide, bool uniform, const StageArgs<double>& a)
{
    if (basis == BASIS_CONSERVED) run_basis<BASIS_CONSERVED>(flux, shape, wide, uniform, a);
    else run_basis<BASIS_PRIMITIVE>(flux, shape, wide, uniform, a);
}

}   // namespace hc

// hc_kernel_inst.hip -- one instantiation of the stage kernel, selected with
// -DHC_LAW=<0|1> -DHC_BASIS=<0|1> -DHC_FLUX=<0..5> -DHC_PREC=<64|32>, in every tile shape
// of its precision.  The FP64 objects are compiled with -ffp-contract=off (bit-faithful
// arithmetic), the mixed ones with contraction allowed.
#if defined(HC_PREC) && HC_PREC == 32
#define HC_MIXED_OBJECT
#endif
#include "hc_fused.hpp"
#include "hc_launch.hpp"

#if !defined(HC_LAW) || !defined(HC_BASIS) || !defined(HC_FLUX) || !defined(HC_PREC)
#error "hc_kernel_inst.hip needs HC_LAW, HC_BASIS, HC_FLUX and HC_PREC"
#endif

#define HC_NAME4(L, B, F, P) hc_stage_L##L##_B##B##_F##F##_P##P
#define HC_NAME(L, B, F, P) HC_NAME4(L, B, F, P)
#define HC_UNAME3(L, B, P) hc_upd_L##L##_B##B##_P##P
#define HC_UNAME(L, B, P) HC_UNAME3(L, B, P)

#if HC_PREC == 64
using RF = double;
#else
using RF = float;
#endif

template <class T, int WPE, class A> static hipError_t launch(const A& L, hipStream_t st)
{
    hipLaunchKernelGGL((hc::k_stage<T, RF, WPE>), dim3(L.ntiles), dim3(T::NT), 0, st, L);
    return hipGetLastError();
}

// UNI: the uniform-geometry kernel of the shape
template <int K, int UNI, class A> static hipError_t launch_shape(const A& L, hipStream_t st)
{
    if constexpr (HC_PREC == 64 && hc::fused_euler(HC_LAW, HC_FLUX)) {
        constexpr hc::TileShape S = hc::TILESF[K];
        // 64-bit offsets only where a mesh needs them, and then in one shape and without the
        // uniform-geometry variant (in every shape they were 30 of 150 fused kernels)
        constexpr hc::TileShape W = hc::TILESW[K];
        if (L.fused && L.wide)
            return launch<hc::FusedTile<HC_BASIS, HC_FLUX, W.ti, W.tj, W.nt, unsigned long long, 0>, 4>(L, st);
        // Five waves per SIMD where they can be had.  15x16 holds 58 KB of LDS, two groups a CU: four.  The
        // folded general tile would spill 20 registers for the fifth, which gains nothing (1000x901 AUSM+up
        // 1265 us for 6 steps at four waves, 1261 - 1271 at five; 144x96 one-stage 408 for 50, 410 at five)
        constexpr int W64 = S.nt > 256 ? 4 : 5, WF64 = UNI ? W64 : 4;
        if (L.fused && L.upd_in)
            return launch<hc::FusedTile<HC_BASIS, HC_FLUX, S.ti, S.tj, S.nt, unsigned, UNI, 1>, WF64>(L, st);
        if (L.fused) return launch<hc::FusedTile<HC_BASIS, HC_FLUX, S.ti, S.tj, S.nt, unsigned, UNI>, W64>(L, st);
    }
    // centre staging has nothing to stage on uniform geometry, so a shape that differs from another
    // only by it shares that shape's kernel
    constexpr hc::TileShape S = hc::tile_shapes(HC_PREC == 32, HC_LAW, HC_FLUX, false, false)[K];
    // FP64 in the reference's order takes 91 - 97 VGPRs where the cell phase's inputs are loaded late: five
    // waves per SIMD ask for 96 (AUSM+up in the primitive basis holds them early, at four): the 512x1024
    // gradient 5190 -> 5104 us; the variants that fold an update would spill there and keep four
    constexpr int CST = UNI ? 0 : S.cst;
    constexpr bool EARLY = HC_LAW == 1 && HC_FLUX == 4 && HC_BASIS == 1;
    constexpr int WPE = S.gpf == 0 ? 1 : HC_PREC == 64 && HC_LAW == 1 && !EARLY && !UNI ? 5 : 4;
    if (L.upd_in)
        return launch<hc::StageTile<HC_LAW, HC_BASIS, HC_FLUX, RF, S.ti, S.tj, S.nt, CST, S.gpf, UNI, 1>, (S.gpf != 0 ? 4 : 1)>(L, st);
    return launch<hc::StageTile<HC_LAW, HC_BASIS, HC_FLUX, RF, S.ti, S.tj, S.nt, CST, S.gpf, UNI>, WPE>(L, st);
}

hipError_t HC_NAME(HC_LAW, HC_BASIS, HC_FLUX, HC_PREC)(const hc::LaunchArgs<RF>& L, int cfg, int uni, hipStream_t st)
{
    static_assert(hc::NTILECFG == 3, "one launch_shape per tile configuration");
    if (L.ntiles <= 0) return hipSuccess;
    if (uni) {
        switch (cfg) {
        case 0: return launch_shape<0, 1>(L, st);
        case 1: return launch_shape<1, 1>(L, st);
        case 2: return launch_shape<2, 1>(L, st);
        default: return hipErrorInvalidValue;
        }
    }
    switch (cfg) {
    case 0: return launch_shape<0, 0>(L, st);
    case 1: return launch_shape<1, 0>(L, st);
    case 2: return launch_shape<2, 0>(L, st);
    default: return hipErrorInvalidValue;
    }
}

#if HC_FLUX == 0
hipError_t HC_UNAME(HC_LAW, HC_BASIS, HC_PREC)(const hc::LaunchArgs<RF>& L, const hc::UpdChunk* chunks, int nchunks,
                                                hipStream_t st)
{
    if (nchunks <= 0) return hipSuccess;
    hipLaunchKernelGGL((hc::k_stage0_update<HC_LAW, HC_BASIS, RF>), dim3((unsigned)nchunks), dim3(256), 0, st, L,
                       chunks);
    return hipGetLastError();
}
#endif

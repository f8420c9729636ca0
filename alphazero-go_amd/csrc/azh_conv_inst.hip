// One compiled instance of the 3x3 convolutions: board size AZH_CONV_N and
// the tower's workgroup shape of index AZH_CONV_TILING for the chunks of input
// channels AZH_CONV_CH (1, 2, or 0 for more; with 0 the stem's shape of that
// index too), all given on the compiler line, or with AZH_RESIDENT_TOWER the
// board-resident tower of board size AZH_CONV_N. The build compiles this file once per
// instance, so the fully unrolled kernels build in parallel.
#include "azh_resident.hpp"

#if !defined(AZH_CONV_N) || (!defined(AZH_CONV_TILING) && !defined(AZH_RESIDENT_TOWER))
#error "AZH_CONV_N and AZH_CONV_TILING (or AZH_RESIDENT_TOWER) must be defined"
#endif

namespace azh {

#if defined(AZH_RESIDENT_TOWER)
template hipError_t launchResidentTowerT<AZH_CONV_N>(const ResidentTower&, int, hipStream_t);
#else
#if AZH_CONV_CH == 0
constexpr ConvTiling kStem = kConvTilings[AZH_CONV_TILING];
template hipError_t launchStemT<AZH_CONV_N, kStem.coPerWave, kStem.wavesCo, kStem.wavesPg, kStem.pgPerWave>(
    const float*, const float*, const float*, const float*, const float*, float*, const BoardScales&, int, int, int,
    bool, hipStream_t);
#endif
constexpr ConvTiling kTower = kTowerTilings[AZH_CONV_TILING];
template hipError_t launchTowerT<AZH_CONV_N, kTower.coPerWave, kTower.wavesCo, kTower.wavesPg, kTower.pgPerWave,
                                 AZH_CONV_CH>(
    const float*, const TowerWeights&, const float*, float*, const BoardScales&, int, int, int, bool, hipStream_t);
#endif

} // namespace azh

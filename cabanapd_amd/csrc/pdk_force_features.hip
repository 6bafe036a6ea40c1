// pdk_force_features.hip -- the row-window force pass of specimens with
// several materials, a temperature and / or a plastic stretch, with a slice's
// rows shared by several waves and on lattices with missing sites
// (pdk_rows.hpp).
#include "pdk_rows.hpp"

namespace pdk
{
namespace
{
template <int MODEL, int FEAT, int W, bool HOLE>
ForceFn pickForm( const PDArgs& a )
{
    const bool mixed = a.precision == PDK_MIXED;
    if constexpr ( ( FEAT & kFeatEP ) == 0 ) // ElasticPerfectlyPlastic exists with fracture only
        if ( !a.fracture )
            return mixed ? kForceRowsF<MODEL, false, kMixed, FEAT, W, HOLE>
                         : kForceRowsF<MODEL, false, kF64, FEAT, W, HOLE>;
    return mixed ? kForceRowsF<MODEL, true, kMixed, FEAT, W, HOLE> : kForceRowsF<MODEL, true, kF64, FEAT, W, HOLE>;
}
template <int MODEL, int FEAT>
ForceFn pickWaves( const PDArgs& a, int waves, bool hole )
{
    switch ( waves )
    {
    case 8: return hole ? pickForm<MODEL, FEAT, 8, true>( a ) : pickForm<MODEL, FEAT, 8, false>( a );
    case 4: return hole ? pickForm<MODEL, FEAT, 4, true>( a ) : pickForm<MODEL, FEAT, 4, false>( a );
    default: return pickForm<MODEL, FEAT, 1, true>( a );
    }
}
} // namespace

ForceFn splitForceRowsFeat( const PDArgs& a, int waves, bool hole )
{
    switch ( rowFeatures( a ) )
    {
    case kFeatMT:
        return a.model == kLPS ? pickWaves<kLPS, kFeatMT>( a, waves, hole ) : pickWaves<kPMB, kFeatMT>( a, waves, hole );
    case kFeatTH: return pickWaves<kPMB, kFeatTH>( a, waves, hole );
    case kFeatEP: return pickWaves<kPMB, kFeatEP>( a, waves, hole );
    default: return pickWaves<kPMB, kFeatTH | kFeatEP>( a, waves, hole );
    }
}

} // namespace pdk

// pdk_force_split.hip -- the row-window force pass and LPS state pass with a
// slice's rows shared by several waves, and on lattices with missing sites
// (pdk_rows.hpp), for one material without temperature or plastic stretch.
#include "pdk_rows.hpp"

namespace pdk
{
namespace
{
// (split launches have a wave or two per SIMD: the row's slots together)
template <int MODEL, int W, bool HOLE>
ForceFn pickForm( const PDArgs& a )
{
    constexpr int G = W > 1 ? kSplitSlots : 1;
    const bool mixed = a.precision == PDK_MIXED;
    if ( a.fracture )
        return mixed ? kForceRows<MODEL, true, kMixed, false, W, HOLE, G>
                     : kForceRows<MODEL, true, kF64, false, W, HOLE, G>;
    return mixed ? kForceRows<MODEL, false, kMixed, false, W, HOLE, G>
                 : kForceRows<MODEL, false, kF64, false, W, HOLE, G>;
}
template <int MODEL>
ForceFn pickWaves( const PDArgs& a, int waves, bool hole )
{
    switch ( waves )
    {
    case 8: return hole ? pickForm<MODEL, 8, true>( a ) : pickForm<MODEL, 8, false>( a );
    case 4: return hole ? pickForm<MODEL, 4, true>( a ) : pickForm<MODEL, 4, false>( a );
    default: return pickForm<MODEL, 1, true>( a );
    }
}
template <int W, bool HOLE>
LpsFn pickLpsForm( const PDArgs& a )
{
    const bool mixed = a.precision == PDK_MIXED;
    if ( a.fracture )
        return mixed ? kLpsStateRows<true, kMixed, false, W, HOLE> : kLpsStateRows<true, kF64, false, W, HOLE>;
    return mixed ? kLpsStateRows<false, kMixed, false, W, HOLE> : kLpsStateRows<false, kF64, false, W, HOLE>;
}
} // namespace

ForceFn splitForceRows( const PDArgs& a, int waves, bool hole )
{
    return a.model == kLPS ? pickWaves<kLPS>( a, waves, hole ) : pickWaves<kPMB>( a, waves, hole );
}

LpsFn splitLpsRows( const PDArgs& a, int waves, bool hole )
{
    switch ( waves )
    {
    case 8: return hole ? pickLpsForm<8, true>( a ) : pickLpsForm<8, false>( a );
    case 4: return hole ? pickLpsForm<4, true>( a ) : pickLpsForm<4, false>( a );
    default: return pickLpsForm<1, true>( a );
    }
}

} // namespace pdk

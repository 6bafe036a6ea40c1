// pdk_contact.hip -- DEM contact step: Hertz and Hertz-JKR pair forces over a
// cell-binned contact list on current positions.
//
// Reference: Force<HertzianModel> (force/CabanaPD_Contact.hpp:109-172) with
// HertzianModel (force_models/CabanaPD_Hertzian.hpp:58-87) or
// HertzianJKRModel (force_models/CabanaPD_HertzianJKR.hpp:82-176), the list
// rebuild of Neighbor::update (CabanaPD_Neighbor.hpp:106-132) and
// VelocityVerlet<Contact> (CabanaPD_Integrate.hpp:147-193).
//
// Extension beyond the reference (which has one radius and equal masses):
// with per-particle radii the pair uses R* = R_i R_j / (R_i + R_j), overlap
// R_i + R_j - r and effective mass m_i m_j / (m_i + m_j).  Uniform specs use
// the reference's expressions unchanged.
#include <algorithm>
#include <cmath>
#include <vector>

#include "pdk_rows.hpp"
#include "pdk_serving.hpp"

namespace pdk
{
namespace
{
constexpr double kPi = 3.141592653589793238462643383279502884;

struct PairK
{
    double Rs, coeff_h_n, delta_tear, two_r, ms;
};

// Correctly rounded powers of the contact models (the reference evaluates
// Kokkos::pow, within an ulp of the exact value).  Built from IEEE operations
// only -- + - * /, sqrt, fma, frexp/ldexp -- in the same order as the
// oracle's, so both return the same bits.  Double-double arithmetic (exact
// products through fma, after Dekker) carries each power to ~2^-100 relative
// before the final rounding, which is then the correct rounding unless the
// exact value lies within ~2^-100 of a rounding boundary (Muller et al.,
// Handbook of Floating-Point Arithmetic, on correct rounding).
__device__ __forceinline__ double crSq( double x )
{
    return x * x;
}
__device__ double crCube( double x )
{
#pragma clang fp contract( off )
    if ( !( fabs( x ) < 1e100 ) || x == 0.0 )
        return x * x * x; // overflow, infinities, NaN and signed zeros as pow
    const double ph = x * x, pl = fma( x, x, -ph );
    const double qh = ph * x, ql = fma( ph, x, -qh );
    return qh + ( ql + pl * x );
}
__device__ __forceinline__ double crHalf( double x )
{
    return x == 0.0 ? 0.0 : sqrt( x ); // +0 at -0, as pow
}
// x^1.5: sqrt with its exact remainder x - sq^2, times x in double-double.
__device__ double crPow32( double x )
{
#pragma clang fp contract( off )
    if ( !( x > 0.0 ) )
        return x == 0.0 ? 0.0 : sqrt( -1.0 );
    if ( isinf( x ) )
        return x;
    const double sq = sqrt( x );
    const double rem = fma( -sq, sq, x );
    const double sl = rem / ( 2.0 * sq );
    const double ph = x * sq, pl = fma( x, sq, -ph );
    return ph + ( pl + x * sl );
}
// ln x for x > 0 to ~1e-16 relative: e ln 2 + 2 atanh(z), z = (m-1)/(m+1),
// m in [1/sqrt 2, sqrt 2), the atanh series to z^23.
__device__ double crLog( double x )
{
#pragma clang fp contract( off )
    int e = 0;
    double m = frexp( x, &e );
    if ( m < 0.70710678118654752440 )
    {
        m = 2.0 * m;
        e = e - 1;
    }
    const double z = ( m - 1.0 ) / ( m + 1.0 );
    const double z2 = z * z;
    double sum = 1.0 / 23.0;
    for ( int k = 21; k >= 1; k -= 2 )
        sum = sum * z2 + 1.0 / k;
    return static_cast<double>( e ) * 0.69314718055994530942 + 2.0 * z * sum;
}
// x^y with y the double nearest 1/3, y = (1 - 2^-54) / 3: cbrt(x) as a
// double-double (Newton from a cubic start, the last step with the exact
// double-double cube), times x^(-2^-54/3) = 1 - t + t^2/2, t = ln(x)/(3 2^54).
__device__ double crThird( double x )
{
#pragma clang fp contract( off )
    if ( x != x || x < 0.0 )
        return sqrt( -1.0 );
    if ( x == 0.0 )
        return 0.0;
    if ( isinf( x ) )
        return x;
    int e = 0;
    const double m0 = frexp( x, &e ); // x = m0 2^e, m0 in [0.5, 1)
    int r = e % 3;
    if ( r < 0 )
        r += 3;
    const double m = ldexp( m0, r ); // in [0.5, 4), e - r divisible by 3
    const int q = ( e - r ) / 3;
    // Newton for c^3 = m from a cubic start (cbrt on [0.5, 1), relative
    // error below 1.4e-4, times 2^(r/3)): three steps reach ~1 ulp
    double c = 0.44019728644131806 + m0 * ( 0.9266652504745495 + m0 * ( -0.5110337078357359 + m0 * 0.1442771968559388 ) );
    c = c * ( r == 0 ? 1.0 : ( r == 1 ? 1.2599210498948732 : 1.5874010519681994 ) );
    for ( int it = 0; it < 3; it++ )
        c = c - ( c * c * c - m ) / ( 3.0 * c * c );
    const double ph = c * c, pl = fma( c, c, -ph );
    const double qh = ph * c, ql = fma( ph, c, -qh );
    const double res = ( ( m - qh ) - ql ) - pl * c;
    const double cl = res / ( 3.0 * ph );
    const double t = crLog( x ) * ( 1.0 / 54043195528445952.0 );
    const double k = -t + 0.5 * ( t * t );
    const double chi = ldexp( c, q ), clo = ldexp( cl, q );
    return chi + ( clo + chi * k );
}

// cbrt(x) to 1.4e-4 relative for finite x > 0: the cubic start of crThird
// (the exponent (1 - 2^-54) / 3 of the exact power changes the value by less
// than 1.3e-14 relative, which the bound absorbs).
__device__ __forceinline__ double cbrtEstimate( double x )
{
#pragma clang fp contract( off )
    int e = 0;
    const double m0 = frexp( x, &e );
    int r = e % 3;
    if ( r < 0 )
        r += 3;
    const int q = ( e - r ) / 3;
    double c = 0.44019728644131806 + m0 * ( 0.9266652504745495 + m0 * ( -0.5110337078357359 + m0 * 0.1442771968559388 ) );
    c = c * ( r == 0 ? 1.0 : ( r == 1 ? 1.2599210498948732 : 1.5874010519681994 ) );
    return ldexp( c, q );
}

__device__ double jkrPatchRadius( const PDArgs& A, double Rs, double delta_n )
{
#pragma clang fp contract( off )
    // force_models/CabanaPD_HertzianJKR.hpp:141-176
    const double nu = A.nu, E = A.E, Gamma = A.Gamma;
    double c0 = crSq( Rs * delta_n );
    double c1 = -4.0 * ( 1.0 - crSq( nu ) ) * kPi * Gamma * crSq( Rs ) / E;
    double c2 = -2.0 * Rs * delta_n;
    double P = -crSq( c2 ) / 12.0 - c0;
    double Q = -crCube( c2 ) / 108.0 + c0 * c2 / 3.0 - crSq( c1 ) / 8.0;
    double U = crThird( -Q / 2.0 + crHalf( fmax( 0.0, crSq( Q ) / 4.0 + crCube( P ) / 27.0 ) ) );
    double sv = 0.0;
    if ( P != 0.0 )
        sv = -5.0 / 6.0 * c2 + U - P / ( 3.0 * U );
    else
        sv = -5.0 / 6.0 * c2 - crThird( Q );
    double w = crHalf( fmax( 0.0, c2 + 2.0 * sv ) );
    double lambda = c1 / ( 2.0 * w + 1e-14 );
    return 1.0 / 2.0 * ( w + crHalf( fmax( 0.0, crSq( w ) - 4.0 * ( c2 + sv + lambda ) ) ) );
}

template <bool JKR>
__device__ double normalForce( const PDArgs& A, const PairK& pk, double r, double vn, double vol )
{
#pragma clang fp contract( off )
    if constexpr ( !JKR )
    {
        const double delta_n = ( r - pk.two_r );
        double coeff = 0.0;
        if ( delta_n < 0.0 )
            coeff = fmin( 0.0, -pk.coeff_h_n * crPow32( fabs( delta_n ) ) );
        coeff /= vol;
        double Sn = 0.0;
        if ( delta_n < 0.0 )
            Sn = 2.0 * A.Es * sqrt( pk.Rs * fabs( delta_n ) );
        coeff -= A.coeff_h_d * sqrt( Sn * pk.ms ) * vn / vol;
        return coeff;
    }
    else
    {
        const double delta_n = ( pk.two_r - r );
        double coeff = 0.0;
        if ( delta_n >= pk.delta_tear )
        {
            double a = jkrPatchRadius( A, pk.Rs, delta_n );
            double a3 = crCube( a );
            coeff = -1.0 * ( pk.coeff_h_n * a3 - crHalf( 8.0 * A.Gamma * kPi * A.Es * a3 ) );
            double Sn = 2.0 * A.Es * a;
            coeff -= A.coeff_h_d * sqrt( Sn * pk.ms ) * vn;
            if ( delta_n <= 0.0 && vn <= 0.0 )
                coeff = 0.0;
        }
        coeff /= vol;
        return coeff;
    }
}

// ---------------------------------------------------------------------------
// Pair records: what a pair force reads of its neighbour, in three 32-byte
// records (position and radius; displacement and mass; velocity) instead of
// twelve gathered doubles.  The neighbours of a wavefront are scattered, so a
// gather costs one cache line a lane and array: 64 lanes touched about 300
// lines per slot.  rec_x follows the upload; rec_u and rec_v are written by the
// pass that advances u and v.  The mass is the product rho V that the pair
// formed before.  Where memory has no room for them (PairRecords) the arrays
// are gathered (REC = false), with the same results.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__( 256 ) void kContactPack( const PDArgs* __restrict__ specs, int32_t parity )
{
#pragma clang fp contract( off )
    const PDArgs& A = *specs;
    const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t n = A.n;
    if ( p >= n )
        return;
    const double* u = A.U[parity];
    A.rec_x[p] = make_double4( A.x[p], A.x[n + p], A.x[2 * n + p], A.radius ? A.radius[p] : 0.0 );
    A.rec_u[p] = make_double4( u[p], u[n + p], u[2 * n + p], A.rho[p] * A.vol[p] );
    A.rec_v[p] = make_double4( A.v[p], A.v[n + p], A.v[2 * n + p], 0.0 );
}

// Hertz-JKR: a listed pair farther apart than its tear distance exerts
// nothing, and the patch radius (a cube root, four square roots, a dozen
// divisions) is most of the pass (VALU bound, 71 % of its cycles).  Each lane
// first marks the pairs that may reach (a squared distance against a bound),
// then evaluates the marked ones in list order: a wavefront runs the patch as
// often as its busiest lane has touching neighbours, not once per listed slot.  A skipped pair adds zero times its unit normal, which
// leaves the sum as it is (pairs that are not at a finite distance are not
// skipped).  Undamped or not, Hertz evaluates every listed pair: its zero
// depends on the velocities being finite.
// (Hertz-JKR, 442k polydisperse spheres, 12 listed neighbours of which about
// 3 touch: 139 -> 127 us; 71 % of the cycles issue VALU work.  Marking by the
// estimated tear distance of each pair instead of the bound: 140.)
template <bool POLY, bool JKR, bool REC>
__global__ __launch_bounds__( kBlock ) void kContact( const PDArgs* __restrict__ specs, int32_t epi, int32_t parity )
{
#pragma clang fp contract( off )
    const PDArgs& A = *specs;
    const int lane = threadIdx.x & ( kSlice - 1 );
    const int64_t slice = xcdRemap( blockIdx.x, gridDim.x ) * kSlicesPerBlock + threadIdx.x / kSlice;
    if ( slice >= A.nslices )
        return;
    const int64_t n = A.n;
    const int64_t p = slice * kSlice + lane;
    if ( p >= n )
        return; // no cross-lane operations in this kernel
    const double4* __restrict__ rec_x = A.rec_x;
    const double4* __restrict__ rec_u = A.rec_u;
    const double4* __restrict__ rec_v = A.rec_v;
    const double* __restrict__ x = A.x;
    const double* __restrict__ u = A.U[parity];
    const double* __restrict__ v = A.v;
    auto loadX = [&]( int64_t j ) {
        if constexpr ( REC )
            return rec_x[j];
        else
            return make_double4( x[j], x[n + j], x[2 * n + j], POLY ? A.radius[j] : 0.0 );
    };
    auto loadU = [&]( int64_t j ) {
        if constexpr ( REC )
            return rec_u[j];
        else
            return make_double4( u[j], u[n + j], u[2 * n + j], POLY ? A.rho[j] * A.vol[j] : 0.0 );
    };
    auto loadV = [&]( int64_t j ) {
        if constexpr ( REC )
            return rec_v[j];
        else
            return make_double4( v[j], v[n + j], v[2 * n + j], 0.0 );
    };
    const double4 xi = loadX( p ), ui = loadU( p ), vi = loadV( p );
    const double vol_i = A.vol[p];
    const double rho_i = A.rho[p];
    const double mi = ui.w;
    const double Ri = xi.w;
    const int32_t mycnt = A.cnt[p];
    const int64_t base = A.slice_ptr[slice];
    const int32_t* __restrict__ colp = A.col + base * kSlice + lane;
    PairK pk;
    pk.Rs = A.Rs;
    pk.coeff_h_n = A.coeff_h_n;
    pk.delta_tear = A.delta_tear;
    pk.two_r = A.two_r;
    pk.ms = ( rho_i * vol_i ) / 2.0;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    // The estimated tear distance of a polydisperse JKR pair and whether it
    // decides on which side of it dn lies: an estimate within 3e-4 relative
    // decides unless dn lies within 1e-3 of it.
    auto tearEstimate = [&]( double Rs, double dn, double& xa, double& dte ) {
        xa = 9.0 / 2.0 * A.Gamma * kPi / A.Es * crSq( Rs );
        // (pow(6, -1/3) of the host's libm, as the oracle evaluates it)
        const double a0e = cbrtEstimate( xa );
        dte = -1.0 / 2.0 * A.jkr_c6 * crSq( a0e ) / Rs;
        return xa > 0.0 && xa < 1e300 && fabs( dte ) > 1e-290 && fabs( dte ) < 1e290 &&
               fabs( dn - dte ) > 1e-3 * fabs( dte );
    };
    auto pairForce = [&]( const double4 xj, const double4 uj, const double4 vj ) {
        const double rx = ( xj.x - xi.x ) + ( uj.x - ui.x );
        const double ry = ( xj.y - xi.y ) + ( uj.y - ui.y );
        const double rz = ( xj.z - xi.z ) + ( uj.z - ui.z );
        // |r| and the normal from one reciprocal root where that gives the
        // general code's bits (pdk_rows.hpp: ordinary magnitudes, and not the
        // one mantissa whose reciprocal it misses)
        const double r2 = rx * rx + ry * ry + rz * rz;
        const Root64 rr = rootRecip( r2 );
        double r = rr.r, nx = divBy( rx, r, rr.y ), ny = divBy( ry, r, rr.y ), nz = divBy( rz, r, rr.y );
        auto plain = []( double a ) { return a == 0.0 || fabs( a ) >= 0x1p-300; };
        if ( !( r2 >= 0x1p-400 && r2 <= 0x1p400 ) || !plain( rx ) || !plain( ry ) || !plain( rz ) ||
             lowWord( r ) == 0xffffffffu )
        {
            r = sqrt( r2 );
            nx = rx / r;
            ny = ry / r;
            nz = rz / r;
        }
        const double vx = vj.x - vi.x, vy = vj.y - vi.y, vz = vj.z - vi.z;
        const double vn = vx * nx + vy * ny + vz * nz;
        if constexpr ( POLY )
        {
            const double Rj = xj.w;
            pk.Rs = Ri * Rj / ( Ri + Rj );
            pk.two_r = Ri + Rj;
            if constexpr ( JKR )
            {
                pk.coeff_h_n = 4.0 / 3.0 * A.Es / pk.Rs;
                // The tear distance only places delta_n = 2R - r on one side
                // of it (normalForce): only where the estimate does not
                // decide is the correctly rounded value formed.  The
                // decision, and with it every force, is that of the exact value.
                const double dn = pk.two_r - r;
                double xa, dte;
                if ( tearEstimate( pk.Rs, dn, xa, dte ) )
                    pk.delta_tear = dn >= dte ? -INFINITY : INFINITY;
                else
                {
                    const double a0 = crThird( xa );
                    pk.delta_tear = -1.0 / 2.0 * A.jkr_c6 * crSq( a0 ) / pk.Rs;
                }
            }
            else
                pk.coeff_h_n = 4.0 / 3.0 * A.Es * sqrt( pk.Rs );
            const double mj = uj.w;
            pk.ms = mi * mj / ( mi + mj );
        }
        const double fn = normalForce<JKR>( A, pk, r, vn, vol_i );
        fx += fn * nx;
        fy += fn * ny;
        fz += fn * nz;
        double ftx = 0.0, fty = 0.0, ftz = 0.0;
        if constexpr ( JKR )
        {
            // force_models/CabanaPD_HertzianJKR.hpp:114-129
            // Without friction or normal force every term is a signed zero,
            // which leaves the sum unchanged: skip the three tanh.
            const double fna = fabs( fn );
            const double mu = A.mu_f;
            if ( mu != 0.0 && fna != 0.0 )
            {
                const double vtx = vx - vn * nx, vty = vy - vn * ny, vtz = vz - vn * nz;
                const double vt = sqrt( vtx * vtx + vty * vty + vtz * vtz );
                ftx = ( vt > 0 ) ? fabs( mu * tanh( 10 * vtx ) ) * fna * vtx / vt : 0.0;
                fty = ( vt > 0 ) ? fabs( mu * tanh( 10 * vty ) ) * fna * vty / vt : 0.0;
                ftz = ( vt > 0 ) ? fabs( mu * tanh( 10 * vtz ) ) * fna * vtz / vt : 0.0;
            }
        }
        fx += ftx;
        fy += fty;
        fz += ftz;
    };
    if constexpr ( JKR )
    {
        // Beyond contact a pair reaches as far as its tear distance, at most
        // that of R* = R_i (it grows with R*, and R* = R_i R_j / (R_i + R_j) <
        // R_i); with a margin over every rounding of the distances.
        double reach = -pk.delta_tear;
        if constexpr ( POLY )
        {
            const double a0e = cbrtEstimate( 9.0 / 2.0 * A.Gamma * kPi / A.Es * crSq( Ri ) );
            reach = 1.0 / 2.0 * A.jkr_c6 * crSq( a0e ) / Ri;
        }
        reach = fabs( reach ) * 1.01 + 0x1p-30 * ( POLY ? Ri : pk.two_r );
        // the ids of the marked pairs, kNear a lane
        constexpr int kNear = 16;
        __shared__ int32_t near[kNear][kBlock];
        int32_t q = 0;
        while ( q < mycnt )
        {
            int marked = 0;
            while ( q < mycnt && marked <= kNear - 4 )
            {
                // four slots at a time: their loads in flight together
                int32_t j[4];
                double4 xj[4], uj[4];
                const int c = mycnt - q < 4 ? mycnt - q : 4;
#pragma unroll
                for ( int k = 0; k < 4; k++ )
                    j[k] = colp[( q + ( k < c ? k : 0 ) ) * kSlice];
#pragma unroll
                for ( int k = 0; k < 4; k++ )
                {
                    xj[k] = loadX( j[k] );
                    uj[k] = loadU( j[k] );
                }
#pragma unroll
                for ( int k = 0; k < 4; k++ )
                {
                    const double rx = ( xj[k].x - xi.x ) + ( uj[k].x - ui.x );
                    const double ry = ( xj[k].y - xi.y ) + ( uj[k].y - ui.y );
                    const double rz = ( xj[k].z - xi.z ) + ( uj[k].z - ui.z );
                    const double r2 = rx * rx + ry * ry + rz * rz;
                    // (comparisons that are false for NaN keep the pair)
                    const double far = ( POLY ? Ri + xj[k].w : pk.two_r ) + reach;
                    const bool skip = r2 > far * far && r2 < 1e300;
                    if ( k < c && !skip )
                        near[marked++][threadIdx.x] = j[k];
                }
                q += c;
            }
            for ( int m = 0; m < marked; m++ )
            {
                const int32_t j = near[m][threadIdx.x];
                pairForce( loadX( j ), loadU( j ), loadV( j ) );
            }
        }
    }
    else
        for ( int32_t q = 0; q < mycnt; q++ )
        {
            const int32_t j = colp[q * kSlice];
            pairForce( loadX( j ), loadU( j ), loadV( j ) );
        }
    if ( epi != kEpiStoreOnly )
    {
        if ( A.body )
        {
            fx = fx + A.body[p];
            fy = fy + A.body[n + p];
            fz = fz + A.body[2 * n + p];
        }
        if ( A.bc_kind >= 0 && A.bcflag[p] )
        {
            if ( A.bc_kind == PDK_BC_FORCE_VALUE )
                fx = fy = fz = A.bc_value;
            else
            {
                fx = fx + A.bc_value;
                fy = fy + A.bc_value;
                fz = fz + A.bc_value;
            }
        }
    }
    // (the velocities are left alone: other waves of this launch read those of
    // their neighbours)
    A.f[p] = fx;
    A.f[n + p] = fy;
    A.f[2 * n + p] = fz;
}

// VelocityVerlet<Contact>::initialHalfStep (CabanaPD_Integrate.hpp:154-193),
// with FINAL preceded by the final half step of the step before (:128-134):
// the half kicks, the drift into the other displacement buffer, the pair
// records (REC) and the block maxima of |u - u_build|.
template <bool FINAL, bool REC>
__global__ __launch_bounds__( 256 ) void kContactAdvance( const PDArgs* __restrict__ specs, int32_t parity,
                                                          double* __restrict__ partial )
{
#pragma clang fp contract( off )
    __shared__ double red[256];
    const PDArgs& A = *specs;
    const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t n = A.n;
    double mx = 0.0;
    if ( p < n )
    {
        const double half_dt_m = A.half_dt / A.rho[p];
        const double* u = A.U[parity];
        double* un = A.U[parity ^ 1];
        double dd[3], uu[3], vv[3];
#pragma unroll
        for ( int d = 0; d < 3; d++ )
        {
            const double f = A.f[d * n + p];
            vv[d] = A.v[d * n + p];
            if constexpr ( FINAL )
                vv[d] = vv[d] + half_dt_m * f;
            vv[d] = vv[d] + half_dt_m * f;
            A.v[d * n + p] = vv[d];
            uu[d] = u[d * n + p] + A.dt * vv[d];
            un[d * n + p] = uu[d];
            dd[d] = uu[d] - A.u_neigh[d * n + p];
        }
        mx = sqrt( dd[0] * dd[0] + dd[1] * dd[1] + dd[2] * dd[2] );
        if constexpr ( REC )
        {
            A.rec_u[p] = make_double4( uu[0], uu[1], uu[2], A.rho[p] * A.vol[p] );
            A.rec_v[p] = make_double4( vv[0], vv[1], vv[2], 0.0 );
        }
    }
    red[threadIdx.x] = mx;
    __syncthreads();
    for ( int w = 128; w > 0; w >>= 1 )
    {
        if ( (int)threadIdx.x < w )
            red[threadIdx.x] = fmax( red[threadIdx.x], red[threadIdx.x + w] );
        __syncthreads();
    }
    if ( threadIdx.x == 0 )
        partial[blockIdx.x] = red[0];
}

// Maximum of the per-block maxima, written to pinned host memory (one block;
// a launch of its own: finishing in the last block of kContactAdvance needs a
// device-wide release per block, which took that pass from 14 to 88 us).
__global__ __launch_bounds__( 1024 ) void kMaxReduce( const double* __restrict__ partial, int64_t nb,
                                                      double* __restrict__ out )
{
    __shared__ double red[1024];
    double mx = 0.0;
    for ( int64_t b = threadIdx.x; b < nb; b += 1024 )
        mx = fmax( mx, partial[b] );
    red[threadIdx.x] = mx;
    __syncthreads();
    for ( int w = 512; w > 0; w >>= 1 )
    {
        if ( (int)threadIdx.x < w )
            red[threadIdx.x] = fmax( red[threadIdx.x], red[threadIdx.x + w] );
        __syncthreads();
    }
    if ( threadIdx.x == 0 )
        *out = red[0];
}

// VelocityVerlet::finalHalfStep (CabanaPD_Integrate.hpp:128-134) as its own
// pass, after a contact pass whose pair forces read the velocities.
__global__ __launch_bounds__( 256 ) void kContactFinal( const PDArgs* __restrict__ specs )
{
#pragma clang fp contract( off )
    const PDArgs& A = *specs;
    const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t n = A.n;
    if ( p >= n )
        return;
    const double half_dt_m = A.half_dt / A.rho[p];
    for ( int d = 0; d < 3; d++ )
        A.v[d * n + p] = A.v[d * n + p] + half_dt_m * A.f[d * n + p];
}

using ContactFn = void ( * )( const PDArgs*, int32_t, int32_t );
template <bool REC>
ContactFn pickContactForm( const PDArgs& a )
{
    const bool jkr = a.model == PDK_MODEL_HERTZ_JKR;
    if ( a.polydisperse )
        return jkr ? kContact<true, true, REC> : kContact<true, false, REC>;
    return jkr ? kContact<false, true, REC> : kContact<false, false, REC>;
}
ContactFn pickContact( const PDArgs& a )
{
    return a.rec_x ? pickContactForm<true>( a ) : pickContactForm<false>( a );
}
thread_local char g_contact_name[64];

} // namespace

const char* contactKernelName( const PDArgs& a )
{
    auto text = []( bool b ) { return b ? "true" : "false"; };
    std::snprintf( g_contact_name, sizeof( g_contact_name ), "kContact<%s, %s, %s>", text( a.polydisperse != 0 ),
                   text( a.model == PDK_MODEL_HERTZ_JKR ), text( a.rec_x != nullptr ) );
    return g_contact_name;
}

// The pair records (if any) of the current state.
void launchContactPack( const PDArgs* args_dev, const PDArgs& a, int32_t parity, hipStream_t st )
{
    if ( a.n == 0 || !a.rec_x )
        return;
    hipLaunchKernelGGL( kContactPack, dim3( static_cast<unsigned>( ( a.n + 255 ) / 256 ) ), dim3( 256 ), 0, st,
                        args_dev, parity );
    PDK_HIP( hipGetLastError() );
}

void launchContactForce( const PDArgs* args_dev, const PDArgs& a, int32_t epilogue_mode, int32_t parity,
                         hipStream_t st )
{
    if ( a.nslices == 0 )
        return;
    const unsigned g = static_cast<unsigned>( ( a.nslices + kSlicesPerBlock - 1 ) / kSlicesPerBlock );
    hipLaunchKernelGGL( pickContact( a ), dim3( g ), dim3( kBlock ), 0, st, args_dev, epilogue_mode,
                        parity );
    PDK_HIP( hipGetLastError() );
}

void launchContactFinal( const PDArgs* args_dev, const PDArgs& a, hipStream_t st )
{
    if ( a.n == 0 )
        return;
    hipLaunchKernelGGL( kContactFinal, dim3( static_cast<unsigned>( ( a.n + 255 ) / 256 ) ), dim3( 256 ), 0, st,
                        args_dev );
    PDK_HIP( hipGetLastError() );
}

void contactBuild( pdk_spec_s* s, bool initial )
{
    ContactState cs = contactState( s );
    contactBuildImpl( s, initial, cs.max_disp, cs.since_build );
}

namespace
{
// The list rebuilt between steps; short of memory, without the pair records.
void rebuildList( pdk_spec_s* s, const ContactState& cs, PairRecords& rec )
{
    specTimed( s, 3, [&] {
        try
        {
            contactBuildImpl( s, false, cs.max_disp, cs.since_build );
        }
        catch ( const MemError& )
        {
            if ( !rec.drop() )
                throw;
            contactBuildImpl( s, false, cs.max_disp, cs.since_build );
        }
    } );
}
} // namespace

// Neighbor::update then the contact pass, storing f (init / computeForce).
void contactForceStore( pdk_spec_s* s )
{
    ContactState cs = contactState( s );
    PairRecords rec( s );
    if ( *cs.max_disp > cs.extend )
        rebuildList( s, cs, rec );
    SpecView v = view( s );
    specTimed( s, 0, [&] {
        launchContactPack( v.dargs, *v.h, *v.cur, v.st );
        launchContactForce( v.dargs, *v.h, kEpiStoreOnly, *v.cur, v.st );
    } );
}

void contactStep( pdk_spec_s* s, int32_t nsteps )
{
    ContactState cs = contactState( s );
    PairRecords rec( s );
    if ( rec.fresh() )
    {
        SpecView v = view( s );
        launchContactPack( v.dargs, *v.h, *v.cur, v.st );
    }
    for ( int32_t k = 0; k < nsteps; k++ )
    {
        if ( rec.wanted() )
            rec.drop();
        SpecView v = view( s );
        const int64_t nb = ( v.n + 255 ) / 256;
        if ( cs.partial->bytes() < static_cast<size_t>( nb ) * sizeof( double ) )
            cs.partial->alloc( nb * sizeof( double ), cs.acct );
        double* part = cs.partial->as<double>();
        specTimed( s, 4, [&] {
            const dim3 g( static_cast<unsigned>( nb ) );
            // the final half step of the step before rides along
            const bool records = v.h->rec_x != nullptr;
            auto advance = k == 0 ? ( records ? kContactAdvance<false, true> : kContactAdvance<false, false> )
                                  : ( records ? kContactAdvance<true, true> : kContactAdvance<true, false> );
            hipLaunchKernelGGL( advance, g, dim3( 256 ), 0, v.st, v.dargs, *v.cur, part );
            hipLaunchKernelGGL( kMaxReduce, dim3( 1 ), dim3( 1024 ), 0, v.st, part, nb, cs.disp_dev );
            PDK_HIP( hipGetLastError() );
        } );
        *v.cur ^= 1;
        // The host decides on a rebuild (CabanaPD_Neighbor.hpp:116-119) from
        // the largest displacement, which the pass wrote to pinned memory.
        // Unless the periodic rebuild is due, the force pass (which writes f
        // only) is launched with the current list before the host waits for
        // that value, so the GPU is not left idle meanwhile; if the
        // displacement calls for a rebuild, the list is rebuilt and the force
        // pass runs again over the new list, which overwrites f.  The results
        // are those of deciding first.
        PDK_HIP( hipEventRecord( cs.disp_ready, v.st ) );
        *cs.since_build += 1;
        const bool periodic = cs.rebuild_every > 0 && *cs.since_build >= cs.rebuild_every;
        auto force = [&] {
            v = view( s );
            specTimed( s, 0, [&] { launchContactForce( v.dargs, *v.h, kEpiApplyOnly, *v.cur, v.st ); } );
        };
        if ( !periodic )
            force();
        PDK_HIP( hipEventSynchronize( cs.disp_ready ) );
        const double mx = *cs.disp_pinned;
        *cs.max_disp = mx;
        if ( mx > cs.extend || periodic )
        {
            rebuildList( s, cs, rec );
            force();
        }
    }
    SpecView v = view( s );
    specTimed( s, 4, [&] { launchContactFinal( v.dargs, *v.h, v.st ); } );
}

} // namespace pdk

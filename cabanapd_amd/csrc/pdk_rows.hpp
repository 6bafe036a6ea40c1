// pdk_rows.hpp -- bond arithmetic and the row-window bond passes (force and
// LPS state), shared by the translation units that instantiate them:
// pdk_force.hip (one wave per slice), pdk_force_split.hip and
// pdk_force_features.hip (split slices, lattices with missing sites).
//
// Mapping: one wavefront per 64-row slice of the sliced CSR, one lane per
// particle, a serial loop over the lane's bonds, no atomics -- the reference's
// SerialOpTag traversal (CabanaPD_Neighbor.hpp:31,134-151) laid out for
// 64-wide wavefronts: each slot row of 64 neighbor ids is one coalesced 256 B
// load and the broken-bond word of a slot row is one uniform 8 B load.
//
// Precision forms:
//   FP64  : the reference's expressions, operand order and rounding
//           (contraction off, correctly rounded sqrt/div).  Rows are summed
//           in the oracle's order, so f/u/v match the oracle bit for bit.
//   MIXED : bond geometry in FP32 from FP64 differences (no large-coordinate
//           cancellation: xi = x_j - x_i and eta = u_j - u_i are formed in
//           FP64 and rounded once), stretch s = (2 xi.eta + eta.eta) /
//           (|xi| (|xi+eta| + |xi|)), bond forces accumulated in FP64.  A
//           bond whose FP32 stretch lies inside a guard band around s0 is
//           re-tested with the FP64 expression, so break decisions equal the
//           FP64 decisions for the same state.
#ifndef PDK_ROWS_HPP
#define PDK_ROWS_HPP

#include <cmath>
#include <type_traits>

#include "pdk_internal.hpp"

namespace pdk
{
namespace
{
// Values equal the ABI's model kinds.  The linearized models take the force
// model of their parent (LinearPMB: PMB, LinearLPS: LPS) and change only the
// bond geometry of the force and energy passes.
enum ModelT : int
{
    kPMB = 0,
    kLPS = 1,
    kLinPMB = 4,
    kLinLPS = 5
};
template <int M>
constexpr bool kIsLps = ( M == kLPS || M == kLinLPS );
template <int M>
constexpr bool kIsLin = ( M == kLinPMB || M == kLinLPS );
enum PrecT : int
{
    kF64 = 0,
    kMixed = 1
};

struct Bond64
{
    double xi, r, s, rx, ry, rz;
};

// getDistance (CabanaPD_Force.hpp:74-93), operation for operation.
__device__ __forceinline__ void getDistance64( double xi0, double xi1, double xi2, double ui0,
                                               double ui1, double ui2, double xj0, double xj1,
                                               double xj2, double uj0, double uj1, double uj2,
                                               Bond64& b )
{
#pragma clang fp contract( off )
    const double xi_x = xj0 - xi0;
    const double eta_u = uj0 - ui0;
    const double xi_y = xj1 - xi1;
    const double eta_v = uj1 - ui1;
    const double xi_z = xj2 - xi2;
    const double eta_w = uj2 - ui2;
    b.rx = xi_x + eta_u;
    b.ry = xi_y + eta_v;
    b.rz = xi_z + eta_w;
    b.r = sqrt( b.rx * b.rx + b.ry * b.ry + b.rz * b.rz );
    b.xi = sqrt( xi_x * xi_x + xi_y * xi_y + xi_z * xi_z );
    b.s = ( b.r - b.xi ) / b.xi;
}

// BaseFractureModel CriticalStretchTag (CabanaPD_ForceModels.hpp:123-128).
__device__ __forceinline__ bool criticalStretch64( double r, double xi, double bcc )
{
#pragma clang fp contract( off )
    return r * r >= bcc * xi * xi;
}

// TemperatureDependent (CabanaPD_ForceModels.hpp:203-211): the bond's
// temp_avg; the stretch becomes s - alpha * temp_avg.
__device__ __forceinline__ double thermalAvg( const PDArgs& A, double Ti, double Tj )
{
#pragma clang fp contract( off )
    return 0.5 * ( Ti + Tj ) - A.temp0;
}
// ThermalFractureModel CriticalStretchTag coefficient (CabanaPD_ForceModels.hpp:246-255).
__device__ __forceinline__ double thermalBcc( const PDArgs& A, double temp_avg )
{
#pragma clang fp contract( off )
    return ( 1.0 + A.s0 + A.alpha * temp_avg ) * ( 1.0 + A.s0 + A.alpha * temp_avg );
}
// EPP ForceCoeffTag (force_models/CabanaPD_PMB.hpp:104-121): update the bond's
// plastic stretch (written only when it changes) and return s - s_p.
__device__ __forceinline__ double plasticStretch( double* slot, double s, double sY )
{
#pragma clang fp contract( off )
    double sp = *slot;
    if ( s >= sp + sY )
    {
        sp = s - sY;
        *slot = sp;
    }
    else if ( s <= sp - sY )
    {
        sp = s + sY;
        *slot = sp;
    }
    return s - sp;
}
// The same with the slot's stored plastic stretch already loaded (sp).
__device__ __forceinline__ double plasticStretchAt( double* slot, double sp, double s, double sY )
{
#pragma clang fp contract( off )
    if ( s >= sp + sY )
    {
        sp = s - sY;
        *slot = sp;
    }
    else if ( s <= sp - sY )
    {
        sp = s + sY;
        *slot = sp;
    }
    return s - sp;
}
// EPP EnergyTag stretch term (force_models/CabanaPD_PMB.hpp:123-146).
__device__ __forceinline__ double plasticEnergyTerm( double s, double sp, double sY )
{
#pragma clang fp contract( off )
    if ( s >= sp + sY )
        return sY * ( 2.0 * s - sY );
    if ( s <= sp - sY )
        return sY * ( -2.0 * s - sY );
    return s * s;
}

struct Bond32
{
    float s, rinv, rx, ry, rz, xi;
};

// Mixed-form bond geometry from the FP64 bond vector r = xi + (u_j - u_i)
// (the reference bond xi of the stencil entry, or x_j - x_i, plus the
// displacement difference, so no large coordinate cancels): the stretch
// numerator |r|^2 - |xi|^2 in FP64 as one FMA chain seeded with -|xi|^2 (the
// FP64 square of the reference bond), then 1/|r| and
//   s = (|r|^2 - |xi|^2) / (|xi| (|r| + |xi|))
// in FP32, with |r|^2 = |xi|^2 + numerator.  The numerator is exact to FP64
// rounding for any rotation of the bond (no xi.eta against eta.eta
// cancellation in FP32), so the FP32 stretch is within a few ulp of s.  The
// force passes accumulate the bond force along the FP64 r.
__device__ __forceinline__ void mixedBond( double r0, double r1, double r2, double xi2d, float xi, Bond32& b )
{
    const float num = static_cast<float>( fma( r0, r0, fma( r1, r1, fma( r2, r2, -xi2d ) ) ) );
    const float r2f = fmaf( xi, xi, num );
    b.rinv = __builtin_amdgcn_rsqf( r2f );
    b.s = num * __builtin_amdgcn_rcpf( fmaf( r2f, b.rinv, xi ) * xi );
    b.rx = static_cast<float>( r0 );
    b.ry = static_cast<float>( r1 );
    b.rz = static_cast<float>( r2 );
    b.xi = xi;
}

// Wave-uniform read through the scalar data cache (p must be the same in
// every lane).  Used for the stencil tables, which no kernel writes, and for
// the per-slot bond-mask words, which a wave reads before it writes them (a
// vector store) and which no other wave of the launch touches; the scalar
// cache starts every kernel dispatch invalidated.
template <class T>
__device__ __forceinline__ T scalarLoad( const T* p )
{
    return *( const __attribute__( ( address_space( 4 ) ) ) T* )( p );
}
__device__ __forceinline__ float4 scalarLoad4( const float4* p )
{
    const auto* f = ( const __attribute__( ( address_space( 4 ) ) ) float* )( p );
    return make_float4( f[0], f[1], f[2], f[3] );
}
// Raw buffer access for the row windows: an SGPR resource (uniform base and
// byte size), a VGPR byte offset (the lane) and an SGPR byte offset (the
// window start), so no address arithmetic runs on the vector ALUs.  Offsets
// at or past the size read 0 (hardware range check), which also covers
// windows that start before id 0 (their negative offsets wrap to values
// above the size for any specimen of fewer than 2^28 particles).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t bufferOf( const void* base, uint32_t bytes )
{
    // base is wave-uniform; readfirstlane keeps the resource in SGPRs
    const uint64_t b = reinterpret_cast<uint64_t>( base );
    const uint32_t lo = __builtin_amdgcn_readfirstlane( static_cast<uint32_t>( b ) );
    const uint32_t hi = __builtin_amdgcn_readfirstlane( static_cast<uint32_t>( b >> 32 ) );
    void* ub = reinterpret_cast<void*>( ( static_cast<uint64_t>( hi ) << 32 ) | lo );
    // dword 3 of a raw (untyped) buffer resource on gfx9-family GPUs
    return __builtin_amdgcn_make_buffer_rsrc( ub, 0, static_cast<int>( __builtin_amdgcn_readfirstlane( bytes ) ),
                                              0x00020000 );
}
__device__ __forceinline__ double bufferLoad64( __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff )
{
    return __builtin_bit_cast( double, __builtin_amdgcn_raw_buffer_load_b64( r, voff, soff, 0 ) );
}
__device__ __forceinline__ uint8_t bufferLoad8( __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff )
{
    return __builtin_amdgcn_raw_buffer_load_b8( r, voff, soff, 0 );
}

__device__ __forceinline__ int4 scalarLoad4( const int4* p )
{
    const auto* f = ( const __attribute__( ( address_space( 4 ) ) ) int* )( p );
    return make_int4( f[0], f[1], f[2], f[3] );
}

// getLinearizedDistance (CabanaPD_Force.hpp:114-138), operation for
// operation: stretch linearized in eta, force along the reference bond.
// Stored so that the force passes' coeff * rx / r is coeff * xi_x / xi.
__device__ __forceinline__ void getLinearizedDistance64( double xi0, double xi1, double xi2, double ui0,
                                                         double ui1, double ui2, double xj0, double xj1,
                                                         double xj2, double uj0, double uj1, double uj2,
                                                         Bond64& b )
{
#pragma clang fp contract( off )
    const double xi_x = xj0 - xi0;
    const double eta_u = uj0 - ui0;
    const double xi_y = xj1 - xi1;
    const double eta_v = uj1 - ui1;
    const double xi_z = xj2 - xi2;
    const double eta_w = uj2 - ui2;
    b.xi = sqrt( xi_x * xi_x + xi_y * xi_y + xi_z * xi_z );
    b.s = ( xi_x * eta_u + xi_y * eta_v + xi_z * eta_w ) / ( b.xi * b.xi );
    b.rx = xi_x;
    b.ry = xi_y;
    b.rz = xi_z;
    b.r = b.xi;
}

// Mixed form of the linearized stretch: s = xi.eta / |xi|^2 in FP32 from the
// FP64 differences; direction and 1/r are those of the reference bond.
__device__ __forceinline__ void linearized32( float gx, float gy, float gz, float xi, float xinv, double ui0,
                                              double ui1, double ui2, double uj0, double uj1, double uj2, Bond32& b )
{
    const float ex = static_cast<float>( uj0 - ui0 );
    const float ey = static_cast<float>( uj1 - ui1 );
    const float ez = static_cast<float>( uj2 - ui2 );
    b.rx = gx;
    b.ry = gy;
    b.rz = gz;
    b.xi = xi;
    b.rinv = xinv;
    b.s = ( gx * ex + gy * ey + gz * ez ) * ( xinv * xinv );
}

// Bond geometry of the force and energy passes for the model.
template <int MODEL>
__device__ __forceinline__ void bond64( double xi0, double xi1, double xi2, double ui0, double ui1, double ui2,
                                        double xj0, double xj1, double xj2, double uj0, double uj1, double uj2,
                                        Bond64& b )
{
    if constexpr ( kIsLin<MODEL> )
        getLinearizedDistance64( xi0, xi1, xi2, ui0, ui1, ui2, xj0, xj1, xj2, uj0, uj1, uj2, b );
    else
        getDistance64( xi0, xi1, xi2, ui0, ui1, ui2, xj0, xj1, xj2, uj0, uj1, uj2, b );
}
// Linearized stretch of the mixed form, bond vector gathered (x_j - x_i)
// or from the stencil table (g = (xi_x, xi_y, xi_z, |xi|), xinv = 1/|xi|).
__device__ __forceinline__ void linearized32g( double xi0, double xi1, double xi2, double ui0, double ui1,
                                               double ui2, double xj0, double xj1, double xj2, double uj0,
                                               double uj1, double uj2, Bond32& b )
{
    const float gx = static_cast<float>( xj0 - xi0 );
    const float gy = static_cast<float>( xj1 - xi1 );
    const float gz = static_cast<float>( xj2 - xi2 );
    const float g2 = gx * gx + gy * gy + gz * gz;
    const float xinv = __builtin_amdgcn_rsqf( g2 );
    linearized32( gx, gy, gz, g2 * xinv, xinv, ui0, ui1, ui2, uj0, uj1, uj2, b );
}

// ---------------------------------------------------------------------------
// The FP64 bond arithmetic without the range handling of the compiler's
// square root and division (the row-window passes).  A bond takes two roots
// and four divisions by them; the compiler's forms scale each operand into
// range, iterate and fix up the special cases, every division from a
// reciprocal of its own (117 VALU instructions per slot of the PMB pass).
// Here one reciprocal square root starts both the root and the reciprocal of
// the root (Goldschmidt's iteration, then Newton's), and the divisions by one
// divisor share it, each corrected by its exact remainder (Markstein):
// the same iterations, so the results are the correctly rounded ones, the
// same bits.  That holds
//   - for operands whose intermediate values neither overflow nor lose bits
//     to underflow: PDArgs::plain_low (lattice, constants) and the rows'
//     own test of the staged values (rowPlain) see to that, together with
//     the coefficient's bound of 2^600;
//   - for roots that are neither zero, infinite nor NaN: those make the
//     stretch NaN, and with it the coefficient;
//   - for divisors other than 2^k (2 - 2^-52), the one mantissa whose
//     reciprocal Newton's iteration misses by an ulp: lowWord
//     finds every divisor whose low word is all ones.
// A row in which a lane fails one of them is evaluated again by the general
// code, from the sums as they were before the row.
// (1e8 random roots and quotients, half of them with mantissas within 16 ulp
// of a power of two, were compared with IEEE results once, with no difference
// but for the excluded divisors; the extreme-value tests compare specimens whose
// bonds are of such lengths with the oracle.  The PMB fracture slot takes 75
// VALU instructions; 25 steps of the 1.44M-particle plate with their download
// 28.2 -> 23.6 ms, 50 steps of a 41^3 cube 4.23 -> 3.52 ms, with the LPS model
// 8.50 -> 7.48.)
// ---------------------------------------------------------------------------
constexpr int kPlainHigh = 100;  // staged u and T: zero or 2^-plain_low <= |.| < 2^100
constexpr int kPlainExpAB = 200; // staged lpsA, lpsB: zero or 2^-200 <= |.| < 2^200

struct Root64
{
    double r, y; // correctly rounded sqrt(a), and 1 / r to within an ulp
};
__device__ __forceinline__ Root64 rootRecip( double a )
{
#pragma clang fp contract( off )
    const double y0 = __builtin_amdgcn_rsq( a );
    const double g0 = a * y0;
    const double h0 = 0.5 * y0;
    const double e = fma( -h0, g0, 0.5 );
    const double g1 = fma( g0, e, g0 );
    const double h1 = fma( h0, e, h0 );
    const double g2 = fma( fma( -g1, g1, a ), h1, g1 );
    Root64 o;
    o.r = fma( fma( -g2, g2, a ), h1, g2 );
    const double y = h1 + h1;
    o.y = fma( y, fma( -o.r, y, 1.0 ), y );
    return o;
}
// The reciprocal of a divisor that is no root (a particle's m).
__device__ __forceinline__ double recip64( double b )
{
    double y = __builtin_amdgcn_rcp( b );
    y = fma( y, fma( -b, y, 1.0 ), y );
    return fma( y, fma( -b, y, 1.0 ), y );
}
// a / b, y = 1 / b to within an ulp
__device__ __forceinline__ double divBy( double a, double b, double y )
{
#pragma clang fp contract( off )
    const double q = a * y;
    return fma( fma( -b, q, a ), y, q );
}
__device__ __forceinline__ uint32_t lowWord( double a )
{
    return static_cast<uint32_t>( __builtin_bit_cast( uint64_t, a ) );
}
// Every finite nonzero argument has magnitude in [2^-(lim+1), 2^lim) (infinities and
// NaN pass: they reach the coefficient as NaN).
__device__ __forceinline__ void expRange( double a, int& lo, int& hi )
{
    const int e = __builtin_amdgcn_frexp_exp( a );
    lo = min( lo, e );
    hi = max( hi, e );
}

struct Fast64
{
    double xi, r, s, rx, ry, rz, yxi, yr;
};
// getDistance64 with shared reciprocals.
__device__ __forceinline__ void getDistanceFast( double xi0, double xi1, double xi2, double ui0, double ui1,
                                                 double ui2, double xj0, double xj1, double xj2, double uj0,
                                                 double uj1, double uj2, Fast64& b )
{
#pragma clang fp contract( off )
    const double xi_x = xj0 - xi0;
    const double eta_u = uj0 - ui0;
    const double xi_y = xj1 - xi1;
    const double eta_v = uj1 - ui1;
    const double xi_z = xj2 - xi2;
    const double eta_w = uj2 - ui2;
    b.rx = xi_x + eta_u;
    b.ry = xi_y + eta_v;
    b.rz = xi_z + eta_w;
    const Root64 r = rootRecip( b.rx * b.rx + b.ry * b.ry + b.rz * b.rz );
    const Root64 x = rootRecip( xi_x * xi_x + xi_y * xi_y + xi_z * xi_z );
    b.r = r.r;
    b.yr = r.y;
    b.xi = x.r;
    b.yxi = x.y;
    b.s = divBy( b.r - b.xi, b.xi, b.yxi );
}

// Uniform per-wave access to the spec of this wave's slice.
struct WaveCtx
{
    const PDArgs* A;
    int64_t slice;
    int32_t epi;
    int32_t cur;
};

// SPLIT: the block's waves share one slice (its lattice rows in turn), else
// every wave of the block has a slice of its own.
template <bool SPLIT = false>
__device__ __forceinline__ bool waveSetup( const PDArgs* __restrict__ specs,
                                           const int32_t* __restrict__ tile_spec,
                                           const int64_t* __restrict__ tile_slice, int32_t epi,
                                           int32_t parity, int64_t launch, WaveCtx& w )
{
    // uniform per wavefront; readfirstlane lets the compiler keep it (and the
    // addresses derived from it) in scalar registers
    const int wave = __builtin_amdgcn_readfirstlane( static_cast<int>( threadIdx.x / kSlice ) );
    const int64_t t = xcdRemap( blockIdx.x, gridDim.x );
    if ( tile_spec == nullptr )
    {
        w.A = specs;
        w.slice = SPLIT ? t : t * kSlicesPerBlock + wave;
        w.epi = epi;
        w.cur = parity;
    }
    else
    {
        // the tile tables are written by the host before the launch
        const int64_t tile = SPLIT ? t / kSlicesPerBlock : t;
        w.A = specs + scalarLoad( tile_spec + tile );
        w.slice = scalarLoad( tile_slice + tile ) + ( SPLIT ? t - tile * kSlicesPerBlock : wave );
        // launch < 0: step -1 - launch of a replayed graph, whose first step's
        // index is the device counter (written by an earlier kernel of the
        // stream; the scalar cache starts every dispatch invalidated)
        const int64_t L = launch >= 0 ? launch : scalarLoad( scalarLoad( &w.A->launch_ctr ) ) + ( -1 - launch );
        w.cur = static_cast<int32_t>( L & 1 ) ^ w.A->parity_offset;
        w.epi = ( L + 1 < w.A->end_launch ) ? kEpiFinalInitial : kEpiFinal;
    }
    return w.slice < w.A->nslices;
}

// Force BC and body term (CabanaPD_Boundary.hpp:94-157, CabanaPD_BodyTerm.hpp:46-63),
// then the velocity-Verlet halves (CabanaPD_Integrate.hpp:100-109, 128-134).
__device__ __forceinline__ void epilogue( const PDArgs& A, int64_t p, int32_t epi, int32_t cur,
                                          double fx, double fy, double fz )
{
#pragma clang fp contract( off )
    const int64_t n = A.n;
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
            {
                fx = A.bc_value;
                fy = A.bc_value;
                fz = A.bc_value;
            }
            else
            {
                fx = fx + A.bc_value;
                fy = fy + A.bc_value;
                fz = fz + A.bc_value;
            }
        }
    }
    A.f[p] = fx;
    A.f[n + p] = fy;
    A.f[2 * n + p] = fz;
    if ( epi == kEpiStoreOnly )
        return;
    const double half_dt_m = A.half_dt / A.rho[p];
    double vx = A.v[p], vy = A.v[n + p], vz = A.v[2 * n + p];
    vx = vx + half_dt_m * fx;
    vy = vy + half_dt_m * fy;
    vz = vz + half_dt_m * fz;
    if ( epi == kEpiFinalInitial )
    {
        vx = vx + half_dt_m * fx;
        vy = vy + half_dt_m * fy;
        vz = vz + half_dt_m * fz;
        const double* u = A.U[cur];
        double* un = A.U[cur ^ 1];
        un[p] = u[p] + A.dt * vx;
        un[n + p] = u[n + p] + A.dt * vy;
        un[2 * n + p] = u[2 * n + p] + A.dt * vz;
    }
    A.v[p] = vx;
    A.v[n + p] = vy;
    A.v[2 * n + p] = vz;
}

// The epilogue of component d alone (the waves of a split slice hold one each).
__device__ __forceinline__ void epilogueOf( const PDArgs& A, int64_t p, int32_t epi, int32_t cur, int d, double f )
{
#pragma clang fp contract( off )
    const int64_t q = d * A.n + p;
    if ( epi != kEpiStoreOnly )
    {
        if ( A.body )
            f = f + A.body[q];
        if ( A.bc_kind >= 0 && A.bcflag[p] )
            f = A.bc_kind == PDK_BC_FORCE_VALUE ? A.bc_value : f + A.bc_value;
    }
    A.f[q] = f;
    if ( epi == kEpiStoreOnly )
        return;
    const double half_dt_m = A.half_dt / A.rho[p];
    double v = A.v[q];
    v = v + half_dt_m * f;
    if ( epi == kEpiFinalInitial )
    {
        v = v + half_dt_m * f;
        A.U[cur ^ 1][q] = A.U[cur][q] + A.dt * v;
    }
    A.v[q] = v;
}

// ---------------------------------------------------------------------------
// Split slices (W waves per slice, small specimens).  With one wave per slice
// a specimen of 64 k particles puts one wave on each SIMD, and a step lasts as
// long as one wave's chain of slots (about 1200 cycles each in FP64: LDS
// reads, two roots, four divisions, nothing to overlap them with).  Here the
// block's W waves take the slice's lattice rows in turn, W rows per round:
// each wave leaves its row's bond terms in LDS, and after a barrier waves 0,
// 1 and 2 add one force component each, in slot order, so every sum takes the
// same terms in the same order as with one wave and has the same bits.
// ---------------------------------------------------------------------------
// Rows of at most kSplitSlots slots (horizons up to three spacings); shorter
// rows fill up with -0.0, which leaves every sum as it is, so that the sums
// run without a branch.
constexpr int kSplitSlots = 5;
template <int W, int ND, int NF>
struct SplitTerms
{
    double d[W][kSplitSlots][ND > 0 ? ND : 1][kSlice];
    float f[NF > 0 ? W : 1][NF > 0 ? kSplitSlots : 1][NF > 0 ? NF : 1][kSlice];
};
// Add a round's terms in slot order: value k of every slot.
template <int W, int ND, int NF>
__device__ __forceinline__ double addRound( const SplitTerms<W, ND, NF>& T, int lane, int k, double sum )
{
#pragma clang fp contract( off )
    double d[W * kSplitSlots];
#pragma unroll
    for ( int v = 0; v < W; v++ )
#pragma unroll
        for ( int t = 0; t < kSplitSlots; t++ )
            d[v * kSplitSlots + t] = T.d[v][t][k][lane];
    if constexpr ( NF > 0 )
    {
        // mixed force pass: factor 0 of the slot times its value
#pragma unroll
        for ( int v = 0; v < W; v++ )
#pragma unroll
            for ( int t = 0; t < kSplitSlots; t++ )
                sum = fma( static_cast<double>( T.f[v][t][0][lane] ), d[v * kSplitSlots + t], sum );
    }
    else
    {
#pragma unroll
        for ( int q = 0; q < W * kSplitSlots; q++ )
            sum += d[q];
    }
    return sum;
}

// ---------------------------------------------------------------------------
// The same force pass with the neighbor data staged in LDS (stencil-slot form
// on lattice rows).  For a lattice row r = (dy, dz) of the stencil, slots
// q0 .. q0+c-1 of the 64 lanes of a slice have their neighbors at the
// contiguous ids g .. g+63+c-1 (g = first id of the slice + the row's offset):
// the wave loads that window once with coalesced loads, stores it in its LDS
// buffer, and slot q0+t of lane L reads window[L + t].  The window of the next
// row is loaded while the current row is evaluated.  Per slot, one
// wave-uniform 64-bit word (scalar load) gates the lanes: the intact word
// under fracture (breaks and pre-notches only clear bits, so it is a subset
// of the existence word) or the existence word.  Evaluation order and
// arithmetic are kForce's, so results are identical.
// ---------------------------------------------------------------------------
// Waves per SIMD the register allocator must leave room for (the attribute
// below): 6 for the PMB passes (80 VGPRs, one spill outside the loops;
// measured 6 % faster on the fracture plate than the unconstrained
// allocation at 5 waves); LPS (models 1 and 5) stays unconstrained, since
// forcing it spills inside the slot loop (mixed LPS at 6 waves: 8 VGPRs
// spilled, 0.349 -> 0.354 ms on a 128^3 cube).
// W: waves per slice (1, or a split slice).  HOLE: a lattice with missing
// sites: the neighbour window of (slice, row) and each lane's place in it come
// from the build's tables (PDArgs::hole_win, hole_pos), and a lane's place
// moves on by one with every neighbour that exists.  Two vector instructions
// and a scalar load a slot more than on full lattices, where the gathers of the
// compact form read 5 bytes of ids a bond and took a wavefront's neighbour
// data from three to twelve scattered loads: 100 mixed steps of a 423k-particle
// perforated plate 26.5 -> 11.0 ms, 100 FP64 elastic-plastic steps of a 29k
// dogbone 14.2 -> 5.3 ms (4.3 with slots together).
// G: slots evaluated together (1: one after the other).  Five in split
// launches, in both precisions.  With one wave per slice five gave 47 -> 41 us
// in FP64 on small specimens and nothing from 2000 slices on; the mixed form got
// slower.
template <int MODEL, bool FRAC, int PREC, bool GEN, int W = 1, bool HOLE = false, int G = 1>
__global__ __launch_bounds__( W == 1 ? kBlock : W * kSlice ) __attribute__( ( amdgpu_waves_per_eu( ( MODEL == 1 || MODEL == 5 || G > 1 ) ? 1 : 6, 8 ) ) ) void
kForceRows( const PDArgs* __restrict__ specs,
                                                        const int32_t* __restrict__ tile_spec,
                                                        const int64_t* __restrict__ tile_slice,
                                                        int32_t epi, int32_t parity, int64_t launch,
                                                        int32_t accumulate )
{
#pragma clang fp contract( off )
    constexpr int kW = kSlice + kRowMaxSlots - 1;  // window width
    constexpr int NX = ( PREC == kF64 ) ? 3 : 0;    // staged x components
    // mixed form (non-linear stretch): the bond vector r = xi + (u_j - u_i)
    // in FP64 from the slot's FP64 stencil offset xi; the windows hold u only
    constexpr bool XV = ( PREC == kMixed ) && !kIsLin<MODEL>;
    constexpr int NAB = kIsLps<MODEL> ? 2 : 0;  // staged lpsA, lpsB
    constexpr bool FAST = ( PREC == kF64 ) && !kIsLin<MODEL>; // shared reciprocals where they give the same bits
    constexpr int KV = 3 + NX + NAB;                // staged vol (GEN)
    constexpr int KNF = KV + 1;                     // staged no-fail flag (GEN)
    constexpr int NC = KV + ( GEN ? 2 : 0 );
    // channel stride: PMB mixed rows pad each channel to 128 values, so the
    // second window half is stored by every lane (no per-row store masks);
    // values past the row's window are never read
    constexpr bool PAD = HOLE || ( ( PREC == kMixed ) && !kIsLps<MODEL> && !GEN );
    constexpr int kWS = PAD ? 2 * kSlice : kW;
    constexpr int NBUF = ( W == 1 && !HOLE ) ? 2 : 1;
    __shared__ double win[W == 1 ? kSlicesPerBlock : W][NBUF][NC][kWS];
    WaveCtx w;
    if ( !waveSetup<( W > 1 )>( specs, tile_spec, tile_slice, epi, parity, launch, w ) )
        return; // one wave per slice: waves are independent; split: the whole block leaves
    const PDArgs& A = *w.A;
    const int wv = __builtin_amdgcn_readfirstlane( static_cast<int>( threadIdx.x / kSlice ) );
    const int lane = threadIdx.x & ( kSlice - 1 );
    const int64_t n = scalarLoad( &A.n );
    const int64_t p0 = w.slice * kSlice;
    const int64_t p = p0 + lane;
    const bool valid = p < n;
    const int64_t pc = valid ? p : p0;
    // Base pointers, the row table and the slice table through scalar loads
    // (the argument block and the tables are written by the host only), so
    // window addresses are an SGPR base plus the lane offset.
    const double* __restrict__ x = scalarLoad( &A.x );
    const double* __restrict__ u = scalarLoad( &A.U[w.cur] );
    const int4* __restrict__ rows = scalarLoad( &A.rows );
    // particle i: reference position (FP64 form) and displacement
    double xi0 = 0.0, xi1 = 0.0, xi2 = 0.0;
    if constexpr ( PREC == kF64 )
    {
        xi0 = x[pc];
        xi1 = x[n + pc];
        xi2 = x[2 * n + pc];
    }
    const double ui0 = u[pc], ui1 = u[n + pc], ui2 = u[2 * n + pc];
    // Per-slot lane masks of the slice: the intact words (a subset of the
    // existence words, so they alone gate the fracture forms) or, without
    // fracture, the existence words.  Lanes past n hold no bonds.
    // (the argument block and the slice table are written by the host only)
    const int64_t row0 = scalarLoad( scalarLoad( &A.slice_ptr ) + w.slice );
    uint64_t* __restrict__ bits = scalarLoad( &A.intact ) + row0;
    const uint64_t* __restrict__ mwords = FRAC ? bits : scalarLoad( &A.exist ) + row0;
    const float4* __restrict__ sten = scalarLoad( &A.stencil );
    const float4* __restrict__ saux = scalarLoad( &A.stencil_aux );
    const double* __restrict__ sxiv = scalarLoad( &A.stencil_xiv );
    const bool nf_i = FRAC ? ( A.nofail[pc] != 0 ) : false;
    // Loop-invariant scalars held in registers (the args block lives in
    // global memory, which the bit-word stores could alias).
    const double c = A.c;
    const double bcc = A.bcc;
    const float c32 = static_cast<float>( A.c );
    const double s0near = A.s0 - 0x1p-30 * ( 1.0 + A.s0 );
    const double volu = A.vol_value;
    const float s0f = A.s0f;
    const float bandK = A.bandK;
    // lower edge of the decision path: every stretch within bandK of s0 or
    // above it lies at or above s0 - 2 bandK
    const float s0lo = s0f - 2.0f * bandK;
    // uniform volume: c vol (PMB) or vol (LPS) scales each FP32 row sum
    const double rscale = GEN ? 1.0 : A.row_scale;
    const int infl1 = A.influence;
    // lanes whose particle may break bonds (every lane of the wave is active here)
    const uint64_t nfi_ok = FRAC ? __ballot( !nf_i ) : 0ull;
    double Ai = 0.0, Bi = 0.0;
    if constexpr ( kIsLps<MODEL> )
    {
        Ai = A.lpsA[pc]; // theta_coeff * theta_i / m_i
        Bi = A.lpsB[pc]; // s_coeff / m_i
    }

    double fx = 0.0, fy = 0.0, fz = 0.0;
    if ( W == 1 && accumulate && valid )
    {
        fx = A.f[p];
        fy = A.f[n + p];
        fz = A.f[2 * n + p];
    }
    // XV: the bond forces fr r (FP32 fr, FP64 bond vector r) summed in FP64
    double sx = 0.0, sy = 0.0, sz = 0.0;

    const double* src[KV];
    src[0] = u;
    src[1] = u + n;
    src[2] = u + 2 * n;
    if constexpr ( NX )
    {
        src[3] = x;
        src[4] = x + n;
        src[5] = x + 2 * n;
    }
    if constexpr ( NAB )
    {
        src[3 + NX] = scalarLoad( &A.lpsA );
        src[4 + NX] = scalarLoad( &A.lpsB );
    }
    const double* __restrict__ volp = scalarLoad( &A.vol );
    const uint8_t* __restrict__ nfp = scalarLoad( &A.nofail );
    double v0[NC], v1[NC];
#pragma unroll
    for ( int k = 0; k < NC; k++ )
        v1[k] = 0.0;
    // Row tables exist only for n < 2^28 (byte sizes and offsets fit 32 bits).
    const int32_t p032 = static_cast<int32_t>( p0 );
    const uint32_t nbytes = static_cast<uint32_t>( n ) * 8u;
    __amdgpu_buffer_rsrc_t rs[KV + ( GEN ? 1 : 0 )];
#pragma unroll
    for ( int k = 0; k < KV; k++ )
        rs[k] = bufferOf( src[k], nbytes );
    const __amdgpu_buffer_rsrc_t rnf = bufferOf( nfp, GEN ? static_cast<uint32_t>( n ) : 0u );
    if constexpr ( GEN )
        rs[KV] = bufferOf( volp, nbytes );
    const uint32_t lane8 = static_cast<uint32_t>( lane ) * 8u;
    auto loadAt = [&]( double* dst, uint32_t vo, uint32_t so ) {
#pragma unroll
        for ( int k = 0; k < KV; k++ )
            dst[k] = bufferLoad64( rs[k], vo, so );
        if constexpr ( GEN )
        {
            dst[KV] = bufferLoad64( rs[KV], vo, so );
            dst[KNF] = ( FRAC && bufferLoad8( rnf, vo >> 3, so >> 3 ) != 0 ) ? 1.0 : 0.0;
        }
    };
    // 64 window values starting at id g (uniform) into dst.
    auto loadHalf = [&]( double* dst, int32_t g ) {
        // g >= 0: lane offset + uniform start; g < 0: per-lane offsets, the
        // negative ones wrap out of range and read 0
        loadAt( dst, g >= 0 ? lane8 : static_cast<uint32_t>( g + lane ) * 8u,
                g >= 0 ? static_cast<uint32_t>( g ) * 8u : 0u );
    };
    auto loadIds = [&]( double* dst, int32_t id ) { loadAt( dst, static_cast<uint32_t>( id ) * 8u, 0u ); };
    // Window of row r: ids g .. g + 63 (every lane) and g + 64 .. g + 64 + c - 2
    // (lanes < c - 1); with holes, ids and length from the build's table.
    const int nrows = scalarLoad( &A.nrows );
    const int64_t hole0 = HOLE ? w.slice * nrows : 0;
    const int4* __restrict__ hwin = HOLE ? scalarLoad( &A.hole_win ) + hole0 : nullptr;
    const uint8_t* __restrict__ hpos = HOLE ? scalarLoad( &A.hole_pos ) + hole0 * kSlice + lane : nullptr;
    int4 wnext{};      // (HOLE) window and place of the row being loaded
    int32_t pnext = 0;
    auto loadRow = [&]( int r ) {
        const int4 R = scalarLoad4( rows + r );
        if constexpr ( HOLE )
        {
            wnext = scalarLoad4( hwin + r );
            pnext = hpos[r * kSlice];
            loadIds( v0, lane + ( lane < wnext.y ? wnext.x : wnext.z ) );
            if ( lane + kSlice < wnext.w )
                loadIds( v1, lane + kSlice + ( lane + kSlice < wnext.y ? wnext.x : wnext.z ) );
            return;
        }
        const int32_t g = p032 + R.z; // uniform
        loadHalf( v0, g );
        if ( lane < R.y - 1 )
            loadHalf( v1, g + kSlice );
    };

    // FAST: the range test of a row's staged values and of particle i's own
    const int plain_low = FAST ? scalarLoad( &A.plain_low ) : 0;
    const bool plain = plain_low != 0;
    int own_lo = 0, own_hi = 0;
    if constexpr ( FAST )
    {
        expRange( ui0, own_lo, own_hi );
        expRange( ui1, own_lo, own_hi );
        expRange( ui2, own_lo, own_hi );
    }
    auto rowPlain = [&]() {
        int lo = own_lo, hi = own_hi;
#pragma unroll
        for ( int q = 0; q < 3; q++ )
        {
            expRange( v0[q], lo, hi );
            expRange( v1[q], lo, hi );
        }
        bool out = lo < -plain_low || hi > kPlainHigh;
        if constexpr ( NAB )
        {
            int la = 0, ha = 0;
#pragma unroll
            for ( int q = 3 + NX; q < 5 + NX; q++ )
            {
                expRange( v0[q], la, ha );
                expRange( v1[q], la, ha );
            }
            expRange( Ai, la, ha );
            expRange( Bi, la, ha );
            out = out || la < -kPlainExpAB || ha > kPlainExpAB;
        }
        return __ballot( out ) == 0;
    };
    // split: the bond terms, three FP64 values and (mixed) one FP32 factor
    __shared__ SplitTerms<W == 1 ? 1 : W, W == 1 ? 0 : 3, ( PREC == kMixed && W > 1 ) ? 1 : 0> T;
    auto put = [&]( int t, double a, double b, double c3 ) {
        if constexpr ( W > 1 )
        {
            T.d[wv][t][0][lane] = a;
            T.d[wv][t][1][lane] = b;
            T.d[wv][t][2][lane] = c3;
        }
    };
    auto putFactor = [&]( int t, float fr ) {
        if constexpr ( W > 1 && PREC == kMixed )
            T.f[wv][t][0][lane] = fr;
    };
    auto evalRow = [&]( const int r ) __attribute__( ( always_inline ) ) {
        const int4 R = scalarLoad4( rows + r );
        double* __restrict__ wb = &win[wv][NBUF == 2 ? r & 1 : 0][0][0];
        const int4 hw = wnext;
        const int32_t pos0 = pnext;
        if constexpr ( NBUF == 1 )
        {
            // the previous row's window reads stay above this row's stores
            __builtin_amdgcn_fence( __ATOMIC_RELEASE, "wavefront" );
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "wavefront" );
        }
#pragma unroll
        for ( int k = 0; k < NC; k++ )
        {
            wb[k * kWS + lane] = v0[k];
            if ( PAD || lane < R.y - 1 )
                wb[k * kWS + kSlice + lane] = v1[k];
        }
        // a tiny (or huge) displacement in the row: only bonds without force
        // may take the shared reciprocals
        const double limit = FAST && rowPlain() ? 0x1p600 : 0.0;
        // LDS operations of one wavefront complete in order; the fences keep
        // the compiler from moving the window reads above the stores.
        __builtin_amdgcn_fence( __ATOMIC_RELEASE, "wavefront" );
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "wavefront" );
        if ( r + W < nrows )
            loadRow( r + W );
        int32_t pos = pos0; // the lane's place in the window (HOLE)
        const uint64_t* __restrict__ ex_r = HOLE ? scalarLoad( &A.exist ) + row0 + R.x : nullptr;
        auto window = [&]( int t ) { return HOLE ? wb + pos : wb + lane + t; };
        auto moveOn = [&]( int t ) {
            if constexpr ( HOLE )
                pos += __builtin_amdgcn_inverse_ballot_w64( scalarLoad( ex_r + t ) ) ? 1 : 0;
        };
        float px = 0.0f, py = 0.0f, pz = 0.0f; // FP32 sum of this row's bond forces (mixed form)
        // the row's slots q = R.x + t through row base pointers, so the
        // unrolled slots address their words and table entries with
        // immediate offsets (no per-slot 64-bit address arithmetic)
        const uint64_t* __restrict__ mw_r = mwords + R.x;
        uint64_t* __restrict__ bits_r = bits + R.x;
        const float4* __restrict__ st_r = sten + R.x;
        const float4* __restrict__ sa_r = saux + R.x;
        const double* __restrict__ xv_r = sxiv + 4 * R.x;
        // XV: xi_y - u_i,y and xi_z - u_i,z, one value each for the row (the
        // slots of a lattice row differ in xi_x only)
        double ay = 0.0, az = 0.0;
        if constexpr ( XV )
        {
            ay = scalarLoad( xv_r + kXiY ) - ui1;
            az = scalarLoad( xv_r + kXiZ ) - ui2;
        }
        // The wave-uniform data of slot t: its intact word (fracture) or
        // existence word, its FP32 stencil entries and (XV) its FP64 offset
        // and |xi|^2 (one 32-byte record).  Loading slot t + 1's data while
        // slot t computes measured slower on the fracture plate (0.209 vs
        // 0.202 ms): the register copies between slots cost more scalar
        // issue than the hidden load latency saved.
        // (the 48-byte records of the other row passes, one scalar load for
        // all of a slot's values, measured 2.8 % slower here: the 32-byte FP64
        // record and the FP32 table entry are two loads but stay within one
        // scalar-cache line each)
        struct SlotK
        {
            uint64_t ww;
            float4 g, ga;
            double x0, x2d;
        };
        auto loadK = [&]( const int t ) __attribute__( ( always_inline ) ) {
            SlotK K{};
            K.ww = scalarLoad( mw_r + t );
            if constexpr ( PREC == kMixed )
            {
                K.g = scalarLoad4( st_r + t );
                K.ga = scalarLoad4( sa_r + t ); // (1/|xi|, |xi|^2, infl |xi|, infl |xi|^2)
                if constexpr ( XV )
                {
                    const double* xv = xv_r + 4 * t;
                    K.x0 = scalarLoad( xv + kXiX );
                    K.x2d = scalarLoad( xv + kXi2 );
                }
            }
            return K;
        };
        auto slot = [&]( const int t, const SlotK& K ) __attribute__( ( always_inline ) ) {
            const uint64_t ww = K.ww;
            // A slot with no live bond in the wave (the slots past a face of
            // the specimen, fully broken slots) adds nothing: the LPS passes
            // skip it (measured 8 % faster on the 128^3 LPS fracture cube; the
            // branch made the PMB plate pass 3 % slower, so PMB evaluates
            // and masks).  The FP64 form skips through its exec mask.
            if constexpr ( PREC == kMixed && kIsLps<MODEL> )
                if ( ww == 0 )
                {
                    if constexpr ( W > 1 )
                    {
                        put( t, 0.0, 0.0, 0.0 );
                        putFactor( t, 0.0f );
                    }
                    moveOn( t );
                    return;
                }
            // The window always holds readable values; bonds that do not
            // exist are masked out below.
            const double* __restrict__ wr = window( t );
            const double uj0 = wr[0], uj1 = wr[kWS], uj2 = wr[2 * kWS];
            // candidates for the break test: intact, neither end no-fail
            // (LPS tests nofail(i) twice, force/CabanaPD_LPS.hpp:417-418)
            uint64_t cand = 0;
            if constexpr ( FRAC )
            {
                cand = ww & nfi_ok;
                if constexpr ( !kIsLps<MODEL> && GEN )
                    cand &= __ballot( wr[KNF * kWS] == 0.0 );
            }
            // Masks below are wave-uniform (ballots in converged code).
            uint64_t brkm = 0; // bonds that break in this pass
            if constexpr ( PREC == kF64 )
            {
                bool brk = false;
                double cx = -0.0, cy = -0.0, cz = -0.0; // what adds nothing to any sum
                if ( __builtin_amdgcn_inverse_ballot_w64( ww ) )
                {
                    const double vj = GEN ? wr[KV * kWS] : volu;
                    Bond64 b;
                    bond64<MODEL>( xi0, xi1, xi2, ui0, ui1, ui2, wr[3 * kWS], wr[4 * kWS], wr[5 * kWS], uj0, uj1,
                                   uj2, b );
                    if constexpr ( FRAC )
                        brk = criticalStretch64( b.r, b.xi, bcc ) && __builtin_amdgcn_inverse_ballot_w64( cand );
                    if ( !brk )
                    {
                        double coeff;
                        if constexpr ( !kIsLps<MODEL> )
                            coeff = c * b.s * vj;
                        else
                        {
                            const double infl = infl1 ? 1.0 / b.xi : 1.0;
                            coeff = ( Ai + wr[( 3 + NX ) * kWS] + b.s * ( Bi + wr[( 4 + NX ) * kWS] ) ) * infl * b.xi * vj;
                        }
                        cx = coeff * b.rx / b.r;
                        cy = coeff * b.ry / b.r;
                        cz = coeff * b.rz / b.r;
                        if constexpr ( W == 1 )
                        {
                            fx += cx;
                            fy += cy;
                            fz += cz;
                        }
                    }
                }
                if constexpr ( W > 1 )
                    put( t, cx, cy, cz );
                if constexpr ( FRAC )
                    brkm = __ballot( brk );
            }
            else
            {
                const float4 g = K.g;
                const float4 ga = K.ga;
                Bond32 b;
                double r0 = 0.0, r1 = 0.0, r2 = 0.0; // XV: the FP64 bond vector
                if constexpr ( XV )
                {
                    r0 = ( uj0 - ui0 ) + K.x0;
                    r1 = uj1 + ay;
                    r2 = uj2 + az;
                    mixedBond( r0, r1, r2, K.x2d, g.w, b );
                }
                else
                    linearized32( g.x, g.y, g.z, g.w, ga.x, ui0, ui1, ui2, uj0, uj1, uj2, b );
                if constexpr ( FRAC )
                {
                    // FP32 decision, except within bandK of s0 where the
                    // reference's FP64 test decides.  One compare first:
                    // only a wave with a candidate at or above s0 - 2 bandK
                    // (rare: bonds near breaking) takes the decision path.
                    if ( __ballot( b.s >= s0lo ) & cand )
                    {
                    const uint64_t inb = __ballot( fabsf( b.s - s0f ) <= bandK ) & cand;
                    brkm = __ballot( b.s > s0f ) & cand & ~inb;
                    if ( inb )
                    {
                        bool crit = false;
                        if ( __builtin_amdgcn_inverse_ballot_w64( inb ) )
                        {
                            // neighbor j = p + R.z + t: uniform base + lane; the
                            // reference positions of i and j are loaded here
                            // (rare path; the compiler barrier keeps the loads of
                            // x_i from being hoisted into registers held for the
                            // whole pass), the displacements are the registers
                            // and the window
                            __asm__ volatile( "" ::: "memory" );
                            // (with holes: the id at the lane's place)
                            const int64_t jo = HOLE ? static_cast<int64_t>( pos - lane + ( pos < hw.y ? hw.x : hw.z ) ) : p0 + R.z + t;
                            const double* __restrict__ xj = x + jo;
                            const double* __restrict__ xp = x + p0;
                            Bond64 e;
                            getDistance64( xp[lane], ( xp + n )[lane], ( xp + 2 * n )[lane], ui0, ui1, ui2, xj[lane],
                                           ( xj + n )[lane], ( xj + 2 * n )[lane], uj0, uj1, uj2, e );
                            crit = criticalStretch64( e.r, e.xi, bcc );
                        }
                        brkm |= __ballot( crit ) & inb;
                    }
                    }
                }
                // dead lanes (absent, broken or breaking bonds) add exactly
                // zero: their window values are finite, fr is selected to 0
                const bool live = __builtin_amdgcn_inverse_ballot_w64( ww & ~brkm );
                float fr;
                if constexpr ( !kIsLps<MODEL> )
                    fr = ( GEN ? ( c32 * static_cast<float>( wr[KV * kWS] ) ) * b.s : b.s ) * b.rinv;
                else
                {
                    const float coeff = static_cast<float>( Ai + wr[( 3 + NX ) * kWS] ) +
                                        b.s * static_cast<float>( Bi + wr[( 4 + NX ) * kWS] );
                    fr = ( GEN ? ( coeff * ga.z ) * static_cast<float>( wr[KV * kWS] ) : coeff * ga.z ) * b.rinv;
                }
                fr = live ? fr : 0.0f;
                if constexpr ( W > 1 )
                {
                    put( t, r0, r1, r2 );
                    putFactor( t, fr );
                }
                else if constexpr ( XV )
                {
                    const double frd = static_cast<double>( fr );
                    sx = fma( frd, r0, sx );
                    sy = fma( frd, r1, sy );
                    sz = fma( frd, r2, sz );
                }
                else
                {
                    px = fmaf( fr, b.rx, px );
                    py = fmaf( fr, b.ry, py );
                    pz = fmaf( fr, b.rz, pz );
                }
            }
            if constexpr ( FRAC )
            {
                // wave-uniform test first (rare: a bond of the wave breaks),
                // then one lane writes the word
                if ( __builtin_expect( brkm != 0, 0 ) )
                {
                    if ( lane == 0 )
                        bits_r[t] = ww & ~brkm;
                }
            }
            moveOn( t );
        };
        // FP64 with shared reciprocals: the lanes whose bond the general code
        // has to evaluate (nothing of such a lane is kept; a bond that breaks
        // in another lane is recorded, and breaks again if the row is
        // evaluated again).
        auto slotFast = [&]( const int t, const double lim ) __attribute__( ( always_inline ) ) {
            const uint64_t ww = scalarLoad( mw_r + t );
            const double* __restrict__ wr = window( t );
            bool brk = false, gen = false;
            double cx = -0.0, cy = -0.0, cz = -0.0;
            if ( __builtin_amdgcn_inverse_ballot_w64( ww ) )
            {
                const double vj = GEN ? wr[KV * kWS] : volu;
                Fast64 b;
                getDistanceFast( xi0, xi1, xi2, ui0, ui1, ui2, wr[3 * kWS], wr[4 * kWS], wr[5 * kWS], wr[0], wr[kWS],
                                 wr[2 * kWS], b );
                if constexpr ( FRAC )
                {
                    // a bond below s0 by more than rounding cannot break: the
                    // reference's test runs only in a wave with a stretch near
                    // s0 or above it
                    if ( __ballot( b.s >= s0near ) )
                    {
                        bool ok = !nf_i;
                        if constexpr ( !kIsLps<MODEL> && GEN )
                            ok = ok && wr[KNF * kWS] == 0.0;
                        brk = criticalStretch64( b.r, b.xi, bcc ) && ok;
                    }
                }
                double coeff;
                if constexpr ( !kIsLps<MODEL> )
                    coeff = c * b.s * vj;
                else
                {
                    const double infl = infl1 ? 1.0 / b.xi : 1.0;
                    coeff = ( Ai + wr[( 3 + NX ) * kWS] + b.s * ( Bi + wr[( 4 + NX ) * kWS] ) ) * infl * b.xi * vj;
                }
                gen = !( fabs( coeff ) <= lim ) || max( lowWord( b.r ), lowWord( b.xi ) ) == 0xffffffffu;
                brk = brk && !gen;
                if ( !brk )
                {
                    cx = divBy( coeff * b.rx, b.r, b.yr );
                    cy = divBy( coeff * b.ry, b.r, b.yr );
                    cz = divBy( coeff * b.rz, b.r, b.yr );
                    if constexpr ( W == 1 )
                    {
                        fx += cx;
                        fy += cy;
                        fz += cz;
                    }
                }
            }
            if constexpr ( W > 1 )
                put( t, cx, cy, cz );
            moveOn( t );
            if constexpr ( FRAC )
            {
                const uint64_t brkm = __ballot( brk );
                if ( __builtin_expect( brkm != 0, 0 ) )
                {
                    if ( lane == 0 )
                        bits_r[t] = ww & ~brkm;
                }
            }
            return __ballot( gen );
        };
        // NG slots at once, every lane evaluating (the window holds readable
        // values; absent bonds are left out of the sums): NG independent
        // chains overlap where the launch has a wave or two per SIMD.  The
        // arithmetic of each bond is slot's / slotFast's.
        auto group = [&]( auto ng, const int t0, const double lim ) __attribute__( ( always_inline ) ) {
            constexpr int NG = decltype( ng )::value;
            uint64_t ww[NG], brkm[NG];
            const double* wr[NG];
            uint64_t bad = 0, near = 0;
#pragma unroll
            for ( int g = 0; g < NG; g++ )
            {
                ww[g] = scalarLoad( mw_r + t0 + g );
                brkm[g] = 0;
                wr[g] = window( t0 + g );
                moveOn( t0 + g );
            }
            if constexpr ( PREC == kF64 )
            {
                Fast64 b[NG];
                double coeff[NG];
#pragma unroll
                for ( int g = 0; g < NG; g++ )
                    getDistanceFast( xi0, xi1, xi2, ui0, ui1, ui2, wr[g][3 * kWS], wr[g][4 * kWS], wr[g][5 * kWS],
                                     wr[g][0], wr[g][kWS], wr[g][2 * kWS], b[g] );
#pragma unroll
                for ( int g = 0; g < NG; g++ )
                {
                    const double vj = GEN ? wr[g][KV * kWS] : volu;
                    if constexpr ( FRAC )
                        near |= __ballot( b[g].s >= s0near ) & ww[g];
                    if constexpr ( !kIsLps<MODEL> )
                        coeff[g] = c * b[g].s * vj;
                    else
                    {
                        const double infl = infl1 ? 1.0 / b[g].xi : 1.0;
                        coeff[g] = ( Ai + wr[g][( 3 + NX ) * kWS] + b[g].s * ( Bi + wr[g][( 4 + NX ) * kWS] ) ) * infl *
                                   b[g].xi * vj;
                    }
                    const uint64_t gen = __ballot( !( fabs( coeff[g] ) <= lim ) ||
                                                   max( lowWord( b[g].r ), lowWord( b[g].xi ) ) == 0xffffffffu ) &
                                         ww[g];
                    bad |= gen;
                }
                if constexpr ( FRAC )
                    if ( near )
                    {
#pragma unroll
                        for ( int g = 0; g < NG; g++ )
                        {
                            uint64_t cand = ww[g] & nfi_ok;
                            if constexpr ( !kIsLps<MODEL> && GEN )
                                cand &= __ballot( wr[g][KNF * kWS] == 0.0 );
                            // (the row is evaluated again where bad: no break is recorded now)
                            brkm[g] = bad ? 0 : __ballot( criticalStretch64( b[g].r, b[g].xi, bcc ) ) & cand;
                        }
                    }
#pragma unroll
                for ( int g = 0; g < NG; g++ )
                {
                    const double cx = divBy( coeff[g] * b[g].rx, b[g].r, b[g].yr );
                    const double cy = divBy( coeff[g] * b[g].ry, b[g].r, b[g].yr );
                    const double cz = divBy( coeff[g] * b[g].rz, b[g].r, b[g].yr );
                    const bool live = __builtin_amdgcn_inverse_ballot_w64( ww[g] & ~brkm[g] );
                    put( t0 + g, live ? cx : -0.0, live ? cy : -0.0, live ? cz : -0.0 );
                }
            }
            else
            {
                Bond32 b[NG];
                double r0[NG], r1[NG], r2[NG];
                float4 ga[NG];
#pragma unroll
                for ( int g = 0; g < NG; g++ )
                {
                    const SlotK K = loadK( t0 + g );
                    ga[g] = K.ga;
                    r0[g] = ( wr[g][0] - ui0 ) + K.x0;
                    r1[g] = wr[g][kWS] + ay;
                    r2[g] = wr[g][2 * kWS] + az;
                    mixedBond( r0[g], r1[g], r2[g], K.x2d, K.g.w, b[g] );
                    if constexpr ( FRAC )
                        near |= __ballot( b[g].s >= s0lo ) & ww[g];
                }
                if constexpr ( FRAC )
                    bad = near; // a bond near s0 or above it: one slot after the other (the caller)
                if ( !bad )
                {
#pragma unroll
                    for ( int g = 0; g < NG; g++ )
                    {
                        float fr;
                        if constexpr ( !kIsLps<MODEL> )
                            fr = ( GEN ? ( c32 * static_cast<float>( wr[g][KV * kWS] ) ) * b[g].s : b[g].s ) * b[g].rinv;
                        else
                        {
                            const float coeff = static_cast<float>( Ai + wr[g][( 3 + NX ) * kWS] ) +
                                                b[g].s * static_cast<float>( Bi + wr[g][( 4 + NX ) * kWS] );
                            fr = ( GEN ? ( coeff * ga[g].z ) * static_cast<float>( wr[g][KV * kWS] )
                                       : coeff * ga[g].z ) *
                                 b[g].rinv;
                        }
                        fr = __builtin_amdgcn_inverse_ballot_w64( ww[g] ) ? fr : 0.0f;
                        put( t0 + g, r0[g], r1[g], r2[g] );
                        putFactor( t0 + g, fr );
                    }
                }
            }
            if constexpr ( FRAC && PREC == kF64 )
            {
#pragma unroll
                for ( int g = 0; g < NG; g++ )
                    if ( __builtin_expect( brkm[g] != 0, 0 ) )
                    {
                        if ( lane == 0 )
                            bits_r[t0 + g] = ww[g] & ~brkm[g];
                    }
            }
            return bad;
        };
        // Mixed forms: the slots of a row (at most kRowMaxSlots) unrolled, so
        // the window reads take immediate offsets and the PMB pass fits 70
        // VGPRs without spills (7 % faster on the fracture plate, 2 % on the
        // LPS cube; unrolling the FP64 form measured slower)
        if constexpr ( PREC == kMixed && G > 1 )
        {
            for ( int t = 0; t < R.y; )
            {
                const int left = R.y - t;
                const int32_t pos_t = pos;
                uint64_t again;
                int done;
                if ( left >= 5 )
                {
                    done = 5;
                    again = group( std::integral_constant<int, 5>{}, t, 0.0 );
                }
                else if ( left >= 3 )
                {
                    done = 3;
                    again = group( std::integral_constant<int, 3>{}, t, 0.0 );
                }
                else
                {
                    done = 1;
                    again = group( std::integral_constant<int, 1>{}, t, 0.0 );
                }
                if ( again )
                {
                    pos = pos_t;
                    for ( int g = 0; g < done; g++ )
                        slot( t + g, loadK( t + g ) );
                }
                t += done;
            }
        }
        else if constexpr ( PREC == kMixed )
        {
#pragma unroll
            for ( int t = 0; t < kRowMaxSlots; t++ )
                if ( t < R.y )
                    slot( t, loadK( t ) );
        }
        else
        {
            if constexpr ( FAST )
            {
                if ( plain )
                {
                    const double fx0 = fx, fy0 = fy, fz0 = fz;
                    uint64_t bad = 0;
                    if constexpr ( G > 1 )
                    {
                        int t = 0;
                        for ( ; t + 5 <= R.y; t += 5 )
                            bad |= group( std::integral_constant<int, 5>{}, t, limit );
                        for ( ; t + 3 <= R.y; t += 3 )
                            bad |= group( std::integral_constant<int, 3>{}, t, limit );
                        for ( ; t < R.y; t++ )
                            bad |= group( std::integral_constant<int, 1>{}, t, limit );
                    }
                    else
                        for ( int t = 0; t < R.y; t++ )
                            bad |= slotFast( t, limit );
                    if ( __builtin_expect( bad == 0, 1 ) )
                        return;
                    fx = fx0;
                    fy = fy0;
                    fz = fz0;
                    pos = pos0;
                }
            }
            for ( int t = 0; t < R.y; t++ )
                slot( t, loadK( t ) );
        }
        if constexpr ( PREC == kMixed && !XV )
        {
            fx = fma( rscale, static_cast<double>( px ), fx );
            fy = fma( rscale, static_cast<double>( py ), fy );
            fz = fma( rscale, static_cast<double>( pz ), fz );
        }
    };
    if constexpr ( W > 1 )
    {
        static_assert( !kIsLin<MODEL>, "the linearized forms are not split" );
        if ( wv < nrows )
            loadRow( wv );
        // component c is added by wave c mod W
        double sum[3] = { 0.0, 0.0, 0.0 };
#pragma unroll
        for ( int c = 0; c < 3; c++ )
            if ( PREC == kF64 && c % W == wv && accumulate && valid )
                sum[c] = A.f[c * n + p];
        for ( int rb = 0; rb < nrows; rb += W )
        {
            int filled = 0;
            if ( rb + wv < nrows )
            {
                evalRow( rb + wv );
                filled = scalarLoad( &rows[rb + wv].y );
            }
            for ( int t = filled; t < kSplitSlots; t++ )
            {
                put( t, -0.0, -0.0, -0.0 );
                putFactor( t, 1.0f ); // 1 x -0.0: nothing
            }
            __syncthreads();
#pragma unroll
            for ( int c = 0; c < 3; c++ )
                if ( c % W == wv )
                    sum[c] = addRound( T, lane, c, sum[c] );
            __syncthreads();
        }
        if ( !valid )
            return;
#pragma unroll
        for ( int c = 0; c < 3; c++ )
            if ( c % W == wv )
            {
                if constexpr ( PREC == kMixed )
                    sum[c] = fma( rscale, sum[c], accumulate ? A.f[c * n + p] : 0.0 );
                epilogueOf( A, p, w.epi, w.cur, c, sum[c] );
            }
        return;
    }
    loadRow( 0 );
    for ( int r = 0; r < nrows; r++ )
        evalRow( r );
    if constexpr ( XV )
    {
        fx = fma( rscale, sx, fx );
        fy = fma( rscale, sy, fy );
        fz = fma( rscale, sz, fz );
    }
    if ( !valid )
        return;
    epilogue( A, p, w.epi, w.cur, fx, fy, fz );
}

// ---------------------------------------------------------------------------
// The row-window force pass for specimens with per-particle features: several
// materials (pair tables), TemperatureDependent (per-particle temperature) and
// ElasticPerfectlyPlastic (per-bond plastic stretch).  FEAT is a set of
// kFeat* bits.  The window channels are u, x (FP64 form), lpsA/lpsB (LPS),
// the volume, a tag (2 x material + no-fail flag) and the temperature; the
// plastic stretch of slot q sits at splas[(row0 + q) * 64 + lane].  Per bond
// the arithmetic and the order of the sums are those of the gather pass
// (kForce with the slot layout), so both forms give identical results.
// ---------------------------------------------------------------------------
enum : int
{
    kFeatMT = 1, // pair tables (multi-material)
    kFeatTH = 2, // temperature-dependent stretch
    kFeatEP = 4  // elastic-perfectly-plastic bonds
};

// Waves per SIMD the register allocator must leave room for: 6 for the mixed
// PMB instances with several materials or a plastic stretch (measured 8 % and
// 10 % faster on the fracture plate than at 4-5 waves); the temperature
// instances spill at 6 and stay unconstrained.
// (W, HOLE: as kForceRows)
template <int MODEL, bool FRAC, int PREC, int FEAT, int W = 1, bool HOLE = false>
__global__ __launch_bounds__( W == 1 ? kBlock : W * kSlice ) __attribute__( ( amdgpu_waves_per_eu( ( W == 1 && PREC == kMixed && !kIsLps<MODEL> && ( FEAT == kFeatMT || FEAT == kFeatEP ) ) ? 6 : 1, 8 ) ) ) void kForceRowsF( const PDArgs* __restrict__ specs,
                                                         const int32_t* __restrict__ tile_spec,
                                                         const int64_t* __restrict__ tile_slice,
                                                         int32_t epi, int32_t parity, int64_t launch,
                                                         int32_t accumulate )
{
#pragma clang fp contract( off )
    constexpr bool MT = ( FEAT & kFeatMT ) != 0;
    constexpr bool TH = ( FEAT & kFeatTH ) != 0 && !kIsLps<MODEL>;
    constexpr bool EP = ( FEAT & kFeatEP ) != 0 && !kIsLps<MODEL>;
    constexpr int kW = HOLE ? 2 * kSlice : kSlice + kRowMaxSlots - 1; // window width
    constexpr int NX = ( PREC == kF64 ) ? 3 : 0;  // staged x components
    constexpr int NAB = kIsLps<MODEL> ? 2 : 0;    // staged lpsA, lpsB
    constexpr int KV = 3 + NX + NAB;              // volume
    constexpr int KT = KV + 1;                    // tag: 2 x material + no-fail flag
    constexpr bool TAG = MT || ( FRAC && !kIsLps<MODEL> );
    constexpr int KH = KT + ( TAG ? 1 : 0 );      // temperature
    constexpr int NC = KH + ( TH ? 1 : 0 );
    // one buffer per wave: the next row's window waits in registers until
    // the current row's reads are done
    __shared__ double win[W == 1 ? kSlicesPerBlock : W][NC][kW];
    // several materials: the pair tables (c, bond_break_coeff, FP32 s0 and
    // band) of the block's spec, indexed 4 a + b
    __shared__ double tab_c[MT ? 16 : 1], tab_bcc[MT ? 16 : 1];
    __shared__ float tab_s0[MT ? 16 : 1], tab_band[MT ? 16 : 1];
    WaveCtx w;
    const bool active = waveSetup<( W > 1 )>( specs, tile_spec, tile_slice, epi, parity, launch, w );
    if constexpr ( MT )
    {
        // every wave of a block belongs to one spec
        if ( threadIdx.x < 16 )
        {
            tab_c[threadIdx.x] = w.A->mat_c[threadIdx.x];
            tab_bcc[threadIdx.x] = w.A->mat_bcc[threadIdx.x];
            tab_s0[threadIdx.x] = w.A->mat_s0f[threadIdx.x];
            tab_band[threadIdx.x] = w.A->mat_bandK[threadIdx.x];
        }
        __syncthreads();
    }
    if ( !active )
        return; // one wave per slice: waves are otherwise independent; split: the whole block leaves
    const PDArgs& A = *w.A;
    const int wv = __builtin_amdgcn_readfirstlane( static_cast<int>( threadIdx.x / kSlice ) );
    const int lane = threadIdx.x & ( kSlice - 1 );
    const int64_t n = scalarLoad( &A.n );
    const int64_t p0 = w.slice * kSlice;
    const int64_t p = p0 + lane;
    const bool valid = p < n;
    const int64_t pc = valid ? p : p0;
    const double* __restrict__ x = scalarLoad( &A.x );
    const double* __restrict__ u = scalarLoad( &A.U[w.cur] );
    const int4* __restrict__ rows = scalarLoad( &A.rows );
    double xi0 = 0.0, xi1 = 0.0, xi2 = 0.0;
    if constexpr ( PREC == kF64 )
    {
        xi0 = x[pc];
        xi1 = x[n + pc];
        xi2 = x[2 * n + pc];
    }
    const double ui0 = u[pc], ui1 = u[n + pc], ui2 = u[2 * n + pc];
    const int64_t row0 = scalarLoad( scalarLoad( &A.slice_ptr ) + w.slice );
    uint64_t* __restrict__ bits = scalarLoad( &A.intact ) + row0;
    const uint64_t* __restrict__ mwords = FRAC ? bits : scalarLoad( &A.exist ) + row0;
    const double* __restrict__ srec = scalarLoad( &A.stencil_rec );
    const uint8_t* __restrict__ nfp = scalarLoad( &A.nofail );
    const uint8_t* __restrict__ mtp = MT ? scalarLoad( &A.mtype ) : nullptr;
    const double* __restrict__ tmpp = TH ? scalarLoad( &A.temp ) : nullptr;
    double* __restrict__ spl = EP ? scalarLoad( &A.splas ) + row0 * kSlice + lane : nullptr;
    const bool nf_i = FRAC ? ( nfp[pc] != 0 ) : false;
    const int ti4 = MT ? 4 * static_cast<int>( mtp[pc] ) : 0;
    const double Ti = TH ? tmpp[pc] : 0.0;
    const double c = A.c;
    const double bcc = A.bcc;
    const float c32 = static_cast<float>( A.c );
    const float s0f = A.s0f;
    const float bandK = A.bandK;
    const int infl1 = A.influence;
    // uniform volume: c vol (PMB, one material) or vol (LPS) scales the sum
    // (as in the gather pass)
    const bool fold = A.vol_uniform != 0 && !( FRAC && A.any_nofail != 0 ) && !( MT && !kIsLps<MODEL> );
    const double rscale = ( PREC == kMixed && fold ) ? A.row_scale : 1.0;
    double Ai = 0.0, Bi = 0.0;
    if constexpr ( kIsLps<MODEL> )
    {
        Ai = A.lpsA[pc]; // theta_coeff * theta_i / m_i
        Bi = A.lpsB[pc]; // s_coeff / m_i
    }
    double fx = 0.0, fy = 0.0, fz = 0.0;
    if ( W == 1 && accumulate && valid )
    {
        fx = A.f[p];
        fy = A.f[n + p];
        fz = A.f[2 * n + p];
    }
    double sx = 0.0, sy = 0.0, sz = 0.0; // mixed form: the bond forces fr r summed in FP64

    const double* src[KV + 1];
    src[0] = u;
    src[1] = u + n;
    src[2] = u + 2 * n;
    if constexpr ( NX )
    {
        src[3] = x;
        src[4] = x + n;
        src[5] = x + 2 * n;
    }
    if constexpr ( NAB )
    {
        src[3 + NX] = scalarLoad( &A.lpsA );
        src[4 + NX] = scalarLoad( &A.lpsB );
    }
    src[KV] = scalarLoad( &A.vol );
    // row tables exist only for n < 2^28 (byte sizes and offsets fit 32 bits)
    const int32_t p032 = static_cast<int32_t>( p0 );
    const uint32_t nbytes = static_cast<uint32_t>( n ) * 8u;
    __amdgpu_buffer_rsrc_t rs[KV + 1];
#pragma unroll
    for ( int k = 0; k <= KV; k++ )
        rs[k] = bufferOf( src[k], nbytes );
    const __amdgpu_buffer_rsrc_t rnf = bufferOf( nfp, static_cast<uint32_t>( n ) );
    const __amdgpu_buffer_rsrc_t rmt = bufferOf( MT ? mtp : nfp, static_cast<uint32_t>( n ) );
    const __amdgpu_buffer_rsrc_t rth = bufferOf( TH ? tmpp : src[0], nbytes );
    const uint32_t lane8 = static_cast<uint32_t>( lane ) * 8u;
    double v0[NC], v1[NC];
#pragma unroll
    for ( int k = 0; k < NC; k++ )
        v1[k] = 0.0;
    auto loadAt = [&]( double* dst, uint32_t vo, uint32_t so ) {
#pragma unroll
        for ( int k = 0; k <= KV; k++ )
            dst[k] = bufferLoad64( rs[k], vo, so );
        if constexpr ( TAG )
        {
            int tag = 0;
            if constexpr ( FRAC && !kIsLps<MODEL> )
                tag = bufferLoad8( rnf, vo >> 3, so >> 3 ) != 0 ? 1 : 0;
            if constexpr ( MT )
                tag += 2 * static_cast<int>( bufferLoad8( rmt, vo >> 3, so >> 3 ) );
            dst[KT] = static_cast<double>( tag );
        }
        if constexpr ( TH )
            dst[KH] = bufferLoad64( rth, vo, so );
    };
    auto loadHalf = [&]( double* dst, int32_t g ) {
        // g >= 0: lane offset + uniform start; g < 0: per-lane offsets, the
        // negative ones wrap out of range and read 0
        loadAt( dst, g >= 0 ? lane8 : static_cast<uint32_t>( g + lane ) * 8u,
                g >= 0 ? static_cast<uint32_t>( g ) * 8u : 0u );
    };
    auto loadIds = [&]( double* dst, int32_t id ) { loadAt( dst, static_cast<uint32_t>( id ) * 8u, 0u ); };
    const int nrows = scalarLoad( &A.nrows );
    const int64_t hole0 = HOLE ? w.slice * nrows : 0;
    const int4* __restrict__ hwin = HOLE ? scalarLoad( &A.hole_win ) + hole0 : nullptr;
    const uint8_t* __restrict__ hpos = HOLE ? scalarLoad( &A.hole_pos ) + hole0 * kSlice + lane : nullptr;
    int4 wnext{};      // (HOLE) window and place of the row being loaded
    int32_t pnext = 0;
    auto loadRow = [&]( int r ) {
        const int4 R = scalarLoad4( rows + r );
        if constexpr ( HOLE )
        {
            wnext = scalarLoad4( hwin + r );
            pnext = hpos[r * kSlice];
            loadIds( v0, lane + ( lane < wnext.y ? wnext.x : wnext.z ) );
            if ( lane + kSlice < wnext.w )
                loadIds( v1, lane + kSlice + ( lane + kSlice < wnext.y ? wnext.x : wnext.z ) );
            return;
        }
        const int32_t g = p032 + R.z; // uniform
        loadHalf( v0, g );
        if ( lane < R.y - 1 )
            loadHalf( v1, g + kSlice );
    };

    // FP64: rows of ordinary values take the shared reciprocals (see kForceRows)
    constexpr bool FAST = ( PREC == kF64 ) && !( TH && EP && W == 1 );
    const int plain_low = FAST ? scalarLoad( &A.plain_low ) : 0;
    const bool plain = plain_low != 0;
    int own_lo = 0, own_hi = 0;
    if constexpr ( FAST )
    {
        expRange( ui0, own_lo, own_hi );
        expRange( ui1, own_lo, own_hi );
        expRange( ui2, own_lo, own_hi );
        expRange( Ti, own_lo, own_hi );
    }
    auto rowPlain = [&]() {
        int lo = own_lo, hi = own_hi;
#pragma unroll
        for ( int q = 0; q < 3; q++ )
        {
            expRange( v0[q], lo, hi );
            expRange( v1[q], lo, hi );
        }
        if constexpr ( TH )
        {
            expRange( v0[KH], lo, hi );
            expRange( v1[KH], lo, hi );
        }
        bool out = lo < -plain_low || hi > kPlainHigh;
        if constexpr ( NAB )
        {
            int la = 0, ha = 0;
#pragma unroll
            for ( int q = 3 + NX; q < 5 + NX; q++ )
            {
                expRange( v0[q], la, ha );
                expRange( v1[q], la, ha );
            }
            expRange( Ai, la, ha );
            expRange( Bi, la, ha );
            out = out || la < -kPlainExpAB || ha > kPlainExpAB;
        }
        return __ballot( out ) == 0;
    };
    double* __restrict__ wb = &win[wv][0][0];
    // split: the bond terms, three FP64 values and (mixed) one FP32 factor
    __shared__ SplitTerms<W == 1 ? 1 : W, W == 1 ? 0 : 3, ( PREC == kMixed && W > 1 ) ? 1 : 0> T;
    auto put = [&]( int t, double a, double b, double c3 ) {
        if constexpr ( W > 1 )
        {
            T.d[wv][t][0][lane] = a;
            T.d[wv][t][1][lane] = b;
            T.d[wv][t][2][lane] = c3;
        }
    };
    auto putFactor = [&]( int t, float fr ) {
        if constexpr ( W > 1 && PREC == kMixed )
            T.f[wv][t][0][lane] = fr;
    };
    auto evalRow = [&]( const int r ) __attribute__( ( always_inline ) ) {
        const int4 R = scalarLoad4( rows + r );
        const int4 hw = wnext;
        const int32_t pos0 = pnext;
        // the previous row's window reads stay above this row's stores (a
        // lane's read of a position another lane overwrites)
        __builtin_amdgcn_fence( __ATOMIC_RELEASE, "wavefront" );
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "wavefront" );
#pragma unroll
        for ( int k = 0; k < NC; k++ )
        {
            wb[k * kW + lane] = v0[k];
            if ( HOLE || lane < R.y - 1 )
                wb[k * kW + kSlice + lane] = v1[k];
        }
        const double limit = FAST && rowPlain() ? 0x1p600 : 0.0;
        __builtin_amdgcn_fence( __ATOMIC_RELEASE, "wavefront" );
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "wavefront" );
        if ( r + W < nrows )
            loadRow( r + W );
        int32_t pos = pos0; // the lane's place in the window (HOLE)
        const uint64_t* __restrict__ ex_r = HOLE ? scalarLoad( &A.exist ) + row0 + R.x : nullptr;
        auto window = [&]( int t ) { return HOLE ? wb + pos : wb + lane + t; };
        auto moveOn = [&]( int t ) {
            if constexpr ( HOLE )
                pos += __builtin_amdgcn_inverse_ballot_w64( scalarLoad( ex_r + t ) ) ? 1 : 0;
        };
        auto slot = [&]( const int t ) __attribute__( ( always_inline ) ) {
            const int32_t q = R.x + t;
            const uint64_t ww = scalarLoad( mwords + q );
            const double* __restrict__ wr = window( t );
            const bool live = __builtin_amdgcn_inverse_ballot_w64( ww );
            int mj = 0;
            bool nf_j = false;
            if constexpr ( TAG )
            {
                const int tag = static_cast<int>( wr[KT * kW] );
                mj = tag >> 1;
                nf_j = ( tag & 1 ) != 0;
            }
            if constexpr ( kIsLps<MODEL> )
                nf_j = nf_i; // LPS tests nofail(i) twice (force/CabanaPD_LPS.hpp:417-418)
            // ElasticPerfectlyPlastic: the slot's plastic stretch is loaded
            // up front (every lane has an entry), so its latency overlaps the
            // bond arithmetic; it is written back only where it changes
            double spv = 0.0;
            if constexpr ( EP )
                spv = spl[q * kSlice];
            if constexpr ( PREC == kF64 )
            {
                bool brk = false;
                double cx = -0.0, cy = -0.0, cz = -0.0; // what adds nothing to any sum
                if ( live )
                {
                    const double uj0 = wr[0], uj1 = wr[kW], uj2 = wr[2 * kW];
                    const double vj = wr[KV * kW];
                    const double tj = TH ? wr[KH * kW] : 0.0;
                    Bond64 b;
                    bond64<MODEL>( xi0, xi1, xi2, ui0, ui1, ui2, wr[3 * kW], wr[4 * kW], wr[5 * kW], uj0, uj1, uj2,
                                   b );
                    double temp_avg = 0.0;
                    if constexpr ( TH )
                    {
                        temp_avg = thermalAvg( A, Ti, tj );
                        b.s = b.s - ( A.alpha * temp_avg );
                    }
                    if constexpr ( FRAC )
                    {
                        const double bcc_ij = TH ? thermalBcc( A, temp_avg ) : ( MT ? tab_bcc[ti4 + mj] : bcc );
                        if ( criticalStretch64( b.r, b.xi, bcc_ij ) && !nf_i && !nf_j )
                            brk = true;
                    }
                    if ( !brk )
                    {
                        double coeff;
                        if constexpr ( !kIsLps<MODEL> )
                        {
                            const double sd = EP ? plasticStretchAt( spl + q * kSlice, spv, b.s, A.sY ) : b.s;
                            coeff = ( MT ? tab_c[ti4 + mj] : c ) * sd * vj;
                        }
                        else
                        {
                            const double infl = infl1 ? 1.0 / b.xi : 1.0;
                            coeff = ( Ai + wr[( 3 + NX ) * kW] + b.s * ( Bi + wr[( 4 + NX ) * kW] ) ) * infl * b.xi *
                                    vj;
                        }
                        cx = coeff * b.rx / b.r;
                        cy = coeff * b.ry / b.r;
                        cz = coeff * b.rz / b.r;
                        if constexpr ( W == 1 )
                        {
                            fx += cx;
                            fy += cy;
                            fz += cz;
                        }
                    }
                }
                if constexpr ( W > 1 )
                    put( t, cx, cy, cz );
                if constexpr ( FRAC )
                {
                    // wave-uniform test first (rare: a bond of the wave
                    // breaks), then one lane writes the word
                    const uint64_t m = __ballot( brk ) & ww;
                    if ( __builtin_expect( m != 0, 0 ) )
                    {
                        if ( lane == 0 )
                            bits[q] = ww & ~m;
                    }
                }
            }
            else
            {
                // every lane evaluates (window values are finite for every
                // lane); bonds that do not exist, are broken or break add
                // exactly zero.  r = xi + (u_j - u_i) from the slot's FP64
                // stencil record.
                const double* rr = srec + kRecStride * q;
                const double uj0 = wr[0], uj1 = wr[kW], uj2 = wr[2 * kW];
                const double r0 = ( uj0 - ui0 ) + scalarLoad( rr + kRecXiX );
                const double r1 = uj1 + ( scalarLoad( rr + kRecXiY ) - ui1 );
                const double r2 = uj2 + ( scalarLoad( rr + kRecXiZ ) - ui2 );
                const float xil = scalarLoad( reinterpret_cast<const float*>( rr + kRecF ) ); // |xi|
                Bond32 b;
                mixedBond( r0, r1, r2, scalarLoad( rr + kRecXi2 ), xil, b );
                double temp_avg = 0.0;
                float ath = 0.0f;
                const float s_mech = b.s;
                if constexpr ( TH )
                {
                    temp_avg = thermalAvg( A, Ti, wr[KH * kW] );
                    ath = static_cast<float>( A.alpha * temp_avg );
                    b.s = b.s - ath;
                }
                uint64_t brkm = 0; // bonds that break in this pass
                if constexpr ( FRAC )
                {
                    // candidates: intact, neither end no-fail; FP32 decision
                    // except within the pair's band of s0, where the
                    // reference's FP64 test decides
                    const uint64_t cand = ww & __ballot( !nf_i && !nf_j );
                    const float s0p = MT ? tab_s0[ti4 + mj] : s0f;
                    const float bandp = MT ? tab_band[ti4 + mj] : bandK;
                    const float band = TH ? fmaf( A.bandf, fabsf( s_mech ) + s0p + fabsf( ath ), bandp ) : bandp;
                    const uint64_t inb = __ballot( fabsf( b.s - s0p ) <= band ) & cand;
                    brkm = __ballot( b.s > s0p ) & cand & ~inb;
                    if ( inb )
                    {
                        bool crit = false;
                        if ( __builtin_amdgcn_inverse_ballot_w64( inb ) )
                        {
                            // rare path: the reference positions are loaded
                            // here (the compiler barrier keeps the loads of
                            // x_i from being hoisted into registers held for
                            // the whole pass)
                            __asm__ volatile( "" ::: "memory" );
                            const int64_t j = HOLE ? static_cast<int64_t>( pos + ( pos < hw.y ? hw.x : hw.z ) ) : p + R.z + t;
                            Bond64 e;
                            getDistance64( x[p], x[n + p], x[2 * n + p], ui0, ui1, ui2, x[j], x[n + j], x[2 * n + j],
                                           uj0, uj1, uj2, e );
                            crit = criticalStretch64( e.r, e.xi,
                                                      TH ? thermalBcc( A, temp_avg ) : ( MT ? tab_bcc[ti4 + mj] : bcc ) );
                        }
                        brkm |= __ballot( crit ) & inb;
                    }
                }
                const bool ok = __builtin_amdgcn_inverse_ballot_w64( ww & ~brkm );
                float fr;
                if constexpr ( !kIsLps<MODEL> )
                {
                    // ElasticPerfectlyPlastic: the plastic stretch stays FP64
                    // and is updated on the bonds that carry force
                    float sd = b.s;
                    if constexpr ( EP )
                    {
                        if ( ok )
                            sd = static_cast<float>(
                                plasticStretchAt( spl + q * kSlice, spv, static_cast<double>( b.s ), A.sY ) );
                    }
                    const float cp = MT ? static_cast<float>( tab_c[ti4 + mj] ) : c32;
                    fr = ( fold ? sd : ( cp * static_cast<float>( wr[KV * kW] ) ) * sd ) * b.rinv;
                }
                else
                {
                    const float wl = infl1 ? 1.0f : xil; // infl |xi|
                    const float coeff = static_cast<float>( Ai + wr[( 3 + NX ) * kW] ) +
                                        b.s * static_cast<float>( Bi + wr[( 4 + NX ) * kW] );
                    fr = ( fold ? coeff * wl : ( coeff * wl ) * static_cast<float>( wr[KV * kW] ) ) * b.rinv;
                }
                fr = ok ? fr : 0.0f;
                if constexpr ( W > 1 )
                {
                    put( t, r0, r1, r2 );
                    putFactor( t, fr );
                }
                else
                {
                    const double frd = static_cast<double>( fr );
                    sx = fma( frd, r0, sx );
                    sy = fma( frd, r1, sy );
                    sz = fma( frd, r2, sz );
                }
                if constexpr ( FRAC )
                {
                    if ( __builtin_expect( brkm != 0, 0 ) )
                    {
                        if ( lane == 0 )
                            bits[q] = ww & ~brkm;
                    }
                }
            }
            moveOn( t );
        };
        // FP64 with shared reciprocals: the lanes the general code has to
        // evaluate (a plastic stretch is updated only where s is final, and
        // updating it again with the same s changes nothing)
        auto slotFast = [&]( const int t, const double lim ) __attribute__( ( always_inline ) ) {
            const int32_t q = R.x + t;
            const uint64_t ww = scalarLoad( mwords + q );
            const double* __restrict__ wr = window( t );
            double spv = 0.0;
            if constexpr ( EP )
                spv = spl[q * kSlice];
            bool brk = false, gen = false;
            double cx = -0.0, cy = -0.0, cz = -0.0;
            if ( __builtin_amdgcn_inverse_ballot_w64( ww ) )
            {
                int mj = 0;
                bool nf_j = false;
                if constexpr ( TAG )
                {
                    const int tag = static_cast<int>( wr[KT * kW] );
                    mj = tag >> 1;
                    nf_j = ( tag & 1 ) != 0;
                }
                if constexpr ( kIsLps<MODEL> )
                    nf_j = nf_i;
                const double vj = wr[KV * kW];
                Fast64 b;
                getDistanceFast( xi0, xi1, xi2, ui0, ui1, ui2, wr[3 * kW], wr[4 * kW], wr[5 * kW], wr[0], wr[kW],
                                 wr[2 * kW], b );
                double temp_avg = 0.0;
                if constexpr ( TH )
                {
                    temp_avg = thermalAvg( A, Ti, wr[KH * kW] );
                    b.s = b.s - ( A.alpha * temp_avg );
                }
                gen = !( fabs( b.s ) <= 0x1p600 ) || max( lowWord( b.r ), lowWord( b.xi ) ) == 0xffffffffu;
                if constexpr ( FRAC )
                {
                    const double bcc_ij = TH ? thermalBcc( A, temp_avg ) : ( MT ? tab_bcc[ti4 + mj] : bcc );
                    brk = !gen && criticalStretch64( b.r, b.xi, bcc_ij ) && !nf_i && !nf_j;
                }
                if ( !brk )
                {
                    double coeff;
                    if constexpr ( !kIsLps<MODEL> )
                    {
                        double sd = b.s;
                        if constexpr ( EP )
                        {
                            if ( !gen )
                                sd = plasticStretchAt( spl + q * kSlice, spv, b.s, A.sY );
                        }
                        coeff = ( MT ? tab_c[ti4 + mj] : c ) * sd * vj;
                    }
                    else
                    {
                        const double infl = infl1 ? 1.0 / b.xi : 1.0;
                        coeff = ( Ai + wr[( 3 + NX ) * kW] + b.s * ( Bi + wr[( 4 + NX ) * kW] ) ) * infl * b.xi * vj;
                    }
                    gen = gen || !( fabs( coeff ) <= lim );
                    cx = divBy( coeff * b.rx, b.r, b.yr );
                    cy = divBy( coeff * b.ry, b.r, b.yr );
                    cz = divBy( coeff * b.rz, b.r, b.yr );
                    if constexpr ( W == 1 )
                    {
                        fx += cx;
                        fy += cy;
                        fz += cz;
                    }
                }
            }
            if constexpr ( W > 1 )
                put( t, cx, cy, cz );
            moveOn( t );
            if constexpr ( FRAC )
            {
                const uint64_t brkm = __ballot( brk );
                if ( __builtin_expect( brkm != 0, 0 ) )
                {
                    if ( lane == 0 )
                        bits[q] = ww & ~brkm;
                }
            }
            return __ballot( gen );
        };
        // slotFast over NG slots at once, every lane evaluating (as kForceRows'
        // group): NG independent chains overlap in a split launch, which has
        // few waves per SIMD
        auto groupFast = [&]( auto ng, const int t0, const double lim ) __attribute__( ( always_inline ) ) {
            constexpr int NG = decltype( ng )::value;
            uint64_t ww[NG], brkm[NG], bad = 0;
            const double* wr[NG];
            double spv[NG];
            Fast64 b[NG];
            double temp_avg[NG];
            bool gen[NG];
#pragma unroll
            for ( int g = 0; g < NG; g++ )
            {
                ww[g] = scalarLoad( mwords + R.x + t0 + g );
                brkm[g] = 0;
                wr[g] = window( t0 + g );
                moveOn( t0 + g );
                spv[g] = 0.0;
                if constexpr ( EP )
                    spv[g] = spl[( R.x + t0 + g ) * kSlice];
            }
#pragma unroll
            for ( int g = 0; g < NG; g++ )
            {
                getDistanceFast( xi0, xi1, xi2, ui0, ui1, ui2, wr[g][3 * kW], wr[g][4 * kW], wr[g][5 * kW], wr[g][0],
                                 wr[g][kW], wr[g][2 * kW], b[g] );
                temp_avg[g] = 0.0;
                if constexpr ( TH )
                {
                    temp_avg[g] = thermalAvg( A, Ti, wr[g][KH * kW] );
                    b[g].s = b[g].s - ( A.alpha * temp_avg[g] );
                }
                gen[g] =
                    !( fabs( b[g].s ) <= 0x1p600 ) || max( lowWord( b[g].r ), lowWord( b[g].xi ) ) == 0xffffffffu;
            }
#pragma unroll
            for ( int g = 0; g < NG; g++ )
            {
                int mj = 0;
                bool nf_j = nf_i;
                if constexpr ( TAG )
                {
                    const int tag = static_cast<int>( wr[g][KT * kW] );
                    mj = tag >> 1;
                    if constexpr ( !kIsLps<MODEL> )
                        nf_j = ( tag & 1 ) != 0;
                }
                if constexpr ( FRAC )
                {
                    const double bcc_ij = TH ? thermalBcc( A, temp_avg[g] ) : ( MT ? tab_bcc[ti4 + mj] : bcc );
                    brkm[g] = __ballot( !gen[g] && criticalStretch64( b[g].r, b[g].xi, bcc_ij ) && !nf_i && !nf_j ) &
                              ww[g];
                }
                const bool live = __builtin_amdgcn_inverse_ballot_w64( ww[g] & ~brkm[g] );
                const double vj = wr[g][KV * kW];
                double coeff;
                if constexpr ( !kIsLps<MODEL> )
                {
                    double sd = b[g].s;
                    if constexpr ( EP )
                    {
                        if ( live && !gen[g] )
                            sd = plasticStretchAt( spl + ( R.x + t0 + g ) * kSlice, spv[g], b[g].s, A.sY );
                    }
                    coeff = ( MT ? tab_c[ti4 + mj] : c ) * sd * vj;
                }
                else
                {
                    const double infl = infl1 ? 1.0 / b[g].xi : 1.0;
                    coeff = ( Ai + wr[g][( 3 + NX ) * kW] + b[g].s * ( Bi + wr[g][( 4 + NX ) * kW] ) ) * infl * b[g].xi *
                            vj;
                }
                // (a bond that breaks needs no coefficient)
                bad |= __ballot( gen[g] || ( live && !( fabs( coeff ) <= lim ) ) ) & ww[g];
                const double cx = divBy( coeff * b[g].rx, b[g].r, b[g].yr );
                const double cy = divBy( coeff * b[g].ry, b[g].r, b[g].yr );
                const double cz = divBy( coeff * b[g].rz, b[g].r, b[g].yr );
                put( t0 + g, live ? cx : -0.0, live ? cy : -0.0, live ? cz : -0.0 );
            }
            if constexpr ( FRAC )
            {
#pragma unroll
                for ( int g = 0; g < NG; g++ )
                    if ( __builtin_expect( brkm[g] != 0, 0 ) )
                    {
                        if ( lane == 0 )
                            bits[R.x + t0 + g] = ww[g] & ~brkm[g];
                    }
            }
            return bad;
        };
        if constexpr ( PREC == kMixed )
        {
#pragma unroll
            for ( int t = 0; t < kRowMaxSlots; t++ )
                if ( t < R.y )
                    slot( t );
        }
        else
        {
            if constexpr ( FAST )
            {
                if ( plain )
                {
                    const double fx0 = fx, fy0 = fy, fz0 = fz;
                    uint64_t bad = 0;
                    if constexpr ( W > 1 )
                    {
                        int t = 0;
                        for ( ; t + 5 <= R.y; t += 5 )
                            bad |= groupFast( std::integral_constant<int, 5>{}, t, limit );
                        for ( ; t + 3 <= R.y; t += 3 )
                            bad |= groupFast( std::integral_constant<int, 3>{}, t, limit );
                        for ( ; t < R.y; t++ )
                            bad |= groupFast( std::integral_constant<int, 1>{}, t, limit );
                    }
                    else
                        for ( int t = 0; t < R.y; t++ )
                            bad |= slotFast( t, limit );
                    if ( __builtin_expect( bad == 0, 1 ) )
                        return;
                    fx = fx0;
                    fy = fy0;
                    fz = fz0;
                    pos = pos0;
                }
            }
            for ( int t = 0; t < R.y; t++ )
                slot( t );
        }
    };
    if constexpr ( W > 1 )
    {
        if ( wv < nrows )
            loadRow( wv );
        // component c is added by wave c mod W
        double sum[3] = { 0.0, 0.0, 0.0 };
#pragma unroll
        for ( int c = 0; c < 3; c++ )
            if ( PREC == kF64 && c % W == wv && accumulate && valid )
                sum[c] = A.f[c * n + p];
        for ( int rb = 0; rb < nrows; rb += W )
        {
            int filled = 0;
            if ( rb + wv < nrows )
            {
                evalRow( rb + wv );
                filled = scalarLoad( &rows[rb + wv].y );
            }
            for ( int t = filled; t < kSplitSlots; t++ )
            {
                put( t, -0.0, -0.0, -0.0 );
                putFactor( t, 1.0f ); // 1 x -0.0: nothing
            }
            __syncthreads();
#pragma unroll
            for ( int c = 0; c < 3; c++ )
                if ( c % W == wv )
                    sum[c] = addRound( T, lane, c, sum[c] );
            __syncthreads();
        }
        if ( !valid )
            return;
#pragma unroll
        for ( int c = 0; c < 3; c++ )
            if ( c % W == wv )
            {
                if constexpr ( PREC == kMixed )
                    sum[c] = fma( rscale, sum[c], accumulate ? A.f[c * n + p] : 0.0 );
                epilogueOf( A, p, w.epi, w.cur, c, sum[c] );
            }
        return;
    }
    loadRow( 0 );
    for ( int r = 0; r < nrows; r++ )
        evalRow( r );
    if constexpr ( PREC == kMixed )
    {
        fx = fma( rscale, sx, fx );
        fy = fma( rscale, sy, fy );
        fz = fma( rscale, sz, fz );
    }
    if ( !valid )
        return;
    epilogue( A, p, w.epi, w.cur, fx, fy, fz );
}

// ---------------------------------------------------------------------------
// The LPS state pass with neighbor data staged in LDS row windows (stencil-slot
// form on lattice rows), as kForceRows does for the force pass.  Same bonds,
// order and expressions as kLpsState, so the results are identical; the FP64
// form walks the rows twice (m_i must be complete before each bond's share of
// theta_i is divided by it), the mixed form once.
// ---------------------------------------------------------------------------
// (W, HOLE: as kForceRows; a split slice's waves 0 and 1 add the two sums)
template <bool FRAC, int PREC, bool GEN, int W = 1, bool HOLE = false>
__global__ __launch_bounds__( W == 1 ? kBlock : W * kSlice ) void kLpsStateRows( const PDArgs* __restrict__ specs,
                                                           const int32_t* __restrict__ tile_spec,
                                                           const int64_t* __restrict__ tile_slice,
                                                           int32_t parity, int64_t launch,
                                                           int32_t do_m, int32_t do_theta )
{
#pragma clang fp contract( off )
    constexpr int kW = HOLE ? 2 * kSlice : kSlice + kRowMaxSlots - 1;
    constexpr int NX = ( PREC == kF64 ) ? 3 : 0; // staged x components
    constexpr int KV = 3 + NX;                   // staged vol (GEN)
    // mixed form: the bond vector r = xi + (u_j - u_i) in FP64 from the slot's
    // FP64 stencil offset xi; the windows hold u only
    constexpr int NC = KV + ( GEN ? 1 : 0 );
    constexpr int NBUF = ( W == 1 && !HOLE ) ? 2 : 1;
    __shared__ double win[W == 1 ? kSlicesPerBlock : W][NBUF][NC][kW];
    __shared__ double msum[W == 1 ? 1 : kSlice];
    WaveCtx w;
    if ( !waveSetup<( W > 1 )>( specs, tile_spec, tile_slice, 0, parity, launch, w ) )
        return; // one wave per slice: waves are independent; split: the whole block leaves
    const PDArgs& A = *w.A;
    const int wv = __builtin_amdgcn_readfirstlane( static_cast<int>( threadIdx.x / kSlice ) );
    const int lane = threadIdx.x & ( kSlice - 1 );
    const int64_t n = scalarLoad( &A.n );
    const int64_t p0 = w.slice * kSlice;
    const int64_t p = p0 + lane;
    const bool valid = p < n;
    const int64_t pc = valid ? p : p0;
    const double* __restrict__ x = scalarLoad( &A.x );
    const double* __restrict__ u = scalarLoad( &A.U[w.cur] );
    const int4* __restrict__ rows = scalarLoad( &A.rows );
    const double xi0 = x[pc], xi1 = x[n + pc], xi2 = x[2 * n + pc];
    const double ui0 = u[pc], ui1 = u[n + pc], ui2 = u[2 * n + pc];
    // per-slot lane masks (intact words, a subset of the existence words,
    // or the existence words without fracture) and the stencil tables, all
    // wave-uniform: scalar loads
    const int64_t row0 = scalarLoad( scalarLoad( &A.slice_ptr ) + w.slice );
    const uint64_t* __restrict__ mwords = scalarLoad( FRAC ? &A.intact : &A.exist ) + row0;
    const double* __restrict__ srec = scalarLoad( &A.stencil_rec );
    const int infl1 = A.influence;
    const double volu = A.vol_value;
    const float vol32 = static_cast<float>( A.vol_value );

    const double* src[KV];
    src[0] = u;
    src[1] = u + n;
    src[2] = u + 2 * n;
    if constexpr ( NX )
    {
        src[3] = x;
        src[4] = x + n;
        src[5] = x + 2 * n;
    }
    const double* __restrict__ volp = scalarLoad( &A.vol );
    const int32_t p032 = static_cast<int32_t>( p0 );
    double v0[NC], v1[NC];
#pragma unroll
    for ( int k = 0; k < NC; k++ )
        v1[k] = 0.0;
    // Row windows through raw buffer loads, as in kForceRows (n < 2^28).
    const uint32_t nbytes = static_cast<uint32_t>( n ) * 8u;
    __amdgpu_buffer_rsrc_t rs[NC];
#pragma unroll
    for ( int k = 0; k < KV; k++ )
        rs[k] = bufferOf( src[k], nbytes );
    if constexpr ( GEN )
        rs[KV] = bufferOf( volp, nbytes );
    const uint32_t lane8 = static_cast<uint32_t>( lane ) * 8u;
    auto loadAt = [&]( double* dst, uint32_t vo, uint32_t so ) {
#pragma unroll
        for ( int k = 0; k < NC; k++ )
            dst[k] = bufferLoad64( rs[k], vo, so );
    };
    auto loadHalf = [&]( double* dst, int32_t g ) {
        loadAt( dst, g >= 0 ? lane8 : static_cast<uint32_t>( g + lane ) * 8u,
                g >= 0 ? static_cast<uint32_t>( g ) * 8u : 0u );
    };
    auto loadIds = [&]( double* dst, int32_t id ) { loadAt( dst, static_cast<uint32_t>( id ) * 8u, 0u ); };
    const int nrows = scalarLoad( &A.nrows );
    const int64_t hole0 = HOLE ? w.slice * nrows : 0;
    const int4* __restrict__ hwin = HOLE ? scalarLoad( &A.hole_win ) + hole0 : nullptr;
    const uint8_t* __restrict__ hpos = HOLE ? scalarLoad( &A.hole_pos ) + hole0 * kSlice + lane : nullptr;
    const uint64_t* __restrict__ exw = HOLE ? scalarLoad( &A.exist ) + row0 : nullptr;
    int32_t pnext = 0; // place in the window of the row being loaded
    auto loadRow = [&]( int r ) {
        const int4 R = scalarLoad4( rows + r );
        if constexpr ( HOLE )
        {
            const int4 wnext = scalarLoad4( hwin + r );
            pnext = hpos[r * kSlice];
            loadIds( v0, lane + ( lane < wnext.y ? wnext.x : wnext.z ) );
            if ( lane + kSlice < wnext.w )
                loadIds( v1, lane + kSlice + ( lane + kSlice < wnext.y ? wnext.x : wnext.z ) );
            return;
        }
        const int32_t g = p032 + R.z; // uniform
        loadHalf( v0, g );
        if ( lane < R.y - 1 )
            loadHalf( v1, g + kSlice );
    };
    // split: a bond's terms -- FP64: the one of the sum being formed; mixed:
    // of m and of theta, as FP64 values of their FP32 terms
    constexpr int ND = PREC == kF64 ? 1 : 2;
    __shared__ SplitTerms<W == 1 ? 1 : W, W == 1 ? 0 : ND, 0> T;
    auto put = [&]( int t, int k, double c ) {
        if constexpr ( W > 1 )
            T.d[wv][t][k][lane] = c;
    };
    // Walk every bond slot in slot order; bond(live, wr, q, ...) gets the
    // window position of the neighbor's staged values and returns the bond's
    // term (FP64), added to sum, or its two (mixed, float2), added to sum and
    // sum2.  FP64: where plain, a row goes through fast first, whose gen marks
    // the lanes that need the general code; then the row is evaluated again
    // by bond, from the sum as it was.  Terms of absent bonds are -0.0, which
    // leave every sum as it is.
    const bool plain = PREC == kF64 && scalarLoad( &A.plain_low ) != 0;
    auto walk = [&]( auto&& bond, auto&& fast, double& sum, double& sum2 ) {
        auto evalRow = [&]( const int r ) __attribute__( ( always_inline ) ) {
            const int4 R = scalarLoad4( rows + r );
            double* __restrict__ wb = &win[wv][NBUF == 2 ? r & 1 : 0][0][0];
            const int32_t pos0 = pnext;
            if constexpr ( NBUF == 1 )
            {
                // the previous row's window reads stay above this row's stores
                __builtin_amdgcn_fence( __ATOMIC_RELEASE, "wavefront" );
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "wavefront" );
            }
#pragma unroll
            for ( int k = 0; k < NC; k++ )
            {
                wb[k * kW + lane] = v0[k];
                if ( HOLE || lane < R.y - 1 )
                    wb[k * kW + kSlice + lane] = v1[k];
            }
            __builtin_amdgcn_fence( __ATOMIC_RELEASE, "wavefront" );
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "wavefront" );
            if ( r + W < nrows )
                loadRow( r + W );
            int32_t pos = pos0; // the lane's place in the window (HOLE)
            auto window = [&]( int t ) { return HOLE ? wb + pos : wb + lane + t; };
            auto moveOn = [&]( int t ) {
                if constexpr ( HOLE )
                    pos += __builtin_amdgcn_inverse_ballot_w64( scalarLoad( exw + R.x + t ) ) ? 1 : 0;
            };
            // mixed form: the row's slots unrolled (immediate window offsets);
            // xi_y - u_i,y and xi_z - u_i,z once per row (the slots of a
            // lattice row differ in xi_x only)
            if constexpr ( PREC == kMixed )
            {
                const double* rec_r = srec + kRecStride * R.x;
                const double ay = scalarLoad( rec_r + kRecXiY ) - ui1;
                const double az = scalarLoad( rec_r + kRecXiZ ) - ui2;
#pragma unroll
                for ( int t = 0; t < kRowMaxSlots; t++ )
                    if ( t < R.y )
                    {
                        const int32_t q = R.x + t;
                        float2 c = make_float2( -0.0f, -0.0f );
                        if ( __builtin_amdgcn_inverse_ballot_w64( scalarLoad( mwords + q ) ) )
                            c = bond( window( t ), q, ay, az );
                        moveOn( t );
                        if constexpr ( W > 1 )
                        {
                            put( t, 0, static_cast<double>( c.x ) );
                            put( t, 1, static_cast<double>( c.y ) );
                        }
                        else
                        {
                            sum += static_cast<double>( c.x );
                            sum2 += static_cast<double>( c.y );
                        }
                    }
            }
            else
            {
                if ( plain )
                {
                    const double sum0 = sum;
                    uint64_t bad = 0;
                    for ( int t = 0; t < R.y; t++ )
                    {
                        bool gen = false;
                        double c = -0.0;
                        if ( __builtin_amdgcn_inverse_ballot_w64( scalarLoad( mwords + R.x + t ) ) )
                            c = fast( window( t ), gen );
                        moveOn( t );
                        if constexpr ( W > 1 )
                            put( t, 0, c );
                        else
                            sum += c;
                        bad |= __ballot( gen );
                    }
                    if ( __builtin_expect( bad == 0, 1 ) )
                        return;
                    sum = sum0;
                    pos = pos0;
                }
                for ( int t = 0; t < R.y; t++ )
                {
                    const int32_t q = R.x + t;
                    double c = -0.0;
                    if ( __builtin_amdgcn_inverse_ballot_w64( scalarLoad( mwords + q ) ) )
                        c = bond( window( t ), q, 0.0, 0.0 );
                    moveOn( t );
                    if constexpr ( W > 1 )
                        put( t, 0, c );
                    else
                        sum += c;
                }
            }
        };
        if constexpr ( W > 1 )
        {
            if ( wv < nrows )
                loadRow( wv );
            for ( int rb = 0; rb < nrows; rb += W )
            {
                int filled = 0;
                if ( rb + wv < nrows )
                {
                    evalRow( rb + wv );
                    filled = scalarLoad( &rows[rb + wv].y );
                }
                for ( int t = filled; t < kSplitSlots; t++ )
                    for ( int k = 0; k < ND; k++ )
                        put( t, k, -0.0 );
                __syncthreads();
                if ( wv == 0 )
                    sum = addRound( T, lane, 0, sum );
                else if ( ND > 1 && wv == 1 )
                    sum2 = addRound( T, lane, ND - 1, sum2 );
                __syncthreads();
            }
        }
        else
        {
            loadRow( 0 );
            for ( int r = 0; r < nrows; r++ )
                evalRow( r );
        }
    };
    // split: wave 0's m_i to every wave
    auto shareM = [&]( double& m ) {
        if constexpr ( W > 1 )
        {
            if ( wv == 0 )
                msum[lane] = m;
            __syncthreads();
            m = msum[lane];
        }
    };

    double m_i = 0.0;
    double th = 0.0;
    double none = 0.0;
    if constexpr ( PREC == kF64 )
    {
        if ( do_m )
        {
            walk(
                [&]( const double* wr, int32_t, double, double ) {
                    Bond64 b;
                    getDistance64( xi0, xi1, xi2, ui0, ui1, ui2, wr[3 * kW], wr[4 * kW], wr[5 * kW], wr[0], wr[kW],
                                   wr[2 * kW], b );
                    const double infl = infl1 ? 1.0 / b.xi : 1.0;
                    return infl * b.xi * b.xi * ( GEN ? wr[KV * kW] : volu );
                },
                [&]( const double* wr, bool& ) {
                    // |xi| alone: its range is the lattice's
                    const double xi_x = wr[3 * kW] - xi0, xi_y = wr[4 * kW] - xi1, xi_z = wr[5 * kW] - xi2;
                    const double xi = rootRecip( xi_x * xi_x + xi_y * xi_y + xi_z * xi_z ).r;
                    const double infl = infl1 ? 1.0 / xi : 1.0;
                    return infl * xi * xi * ( GEN ? wr[KV * kW] : volu );
                },
                m_i, none );
            shareM( m_i );
        }
        else if ( valid )
            m_i = A.m[p];
        const bool mpos = FRAC ? ( m_i > 0 ) : true;
        if ( do_theta )
        {
            // one reciprocal of m_i for all its bonds
            const double ym = recip64( m_i );
            const bool gen_m = !( m_i >= 0x1p-300 && m_i <= 0x1p300 ) || lowWord( m_i ) == 0xffffffffu;
            walk(
                [&]( const double* wr, int32_t, double, double ) {
                    if ( !mpos )
                        return -0.0;
                    Bond64 b;
                    getDistance64( xi0, xi1, xi2, ui0, ui1, ui2, wr[3 * kW], wr[4 * kW], wr[5 * kW], wr[0], wr[kW],
                                   wr[2 * kW], b );
                    const double infl = infl1 ? 1.0 / b.xi : 1.0;
                    const double theta_b = infl * b.s * b.xi * b.xi * ( GEN ? wr[KV * kW] : volu );
                    return 3.0 * theta_b / m_i;
                },
                [&]( const double* wr, bool& gen ) {
                    if ( !mpos )
                        return -0.0;
                    Fast64 b;
                    getDistanceFast( xi0, xi1, xi2, ui0, ui1, ui2, wr[3 * kW], wr[4 * kW], wr[5 * kW], wr[0], wr[kW],
                                     wr[2 * kW], b );
                    const double infl = infl1 ? 1.0 / b.xi : 1.0;
                    const double theta_b = infl * b.s * b.xi * b.xi * ( GEN ? wr[KV * kW] : volu );
                    gen = gen_m || !( fabs( theta_b ) <= 0x1p300 ) || lowWord( b.xi ) == 0xffffffffu;
                    return divBy( 3.0 * theta_b, m_i, ym );
                },
                th, none );
        }
    }
    else
    {
        if ( !do_m && valid )
            m_i = A.m[p];
        // m_i for the theta condition is only known after the walk: sum both,
        // apply the condition at the end (the sums are the same per-bond terms)
        walk(
            [&]( const double* wr, int32_t q, double ay, double az ) {
                // the slot's record: xi_x, |xi|^2, |xi|, infl |xi|^2
                const double* rr = srec + kRecStride * q;
                const float* rf = reinterpret_cast<const float*>( rr + kRecF );
                const float w2 = scalarLoad( rf + 2 ); // infl |xi|^2
                const float vj32 = GEN ? static_cast<float>( wr[KV * kW] ) : vol32;
                float2 c = make_float2( -0.0f, -0.0f );
                if ( do_m )
                    c.x = w2 * vj32;
                if ( do_theta )
                {
                    Bond32 b;
                    mixedBond( ( wr[0] - ui0 ) + scalarLoad( rr + kRecXiX ), wr[kW] + ay, wr[2 * kW] + az,
                               scalarLoad( rr + kRecXi2 ), scalarLoad( rf ), b );
                    c.y = w2 * b.s * vj32;
                }
                return c;
            },
            [&]( const double*, bool& ) { return 0.0; }, m_i, th );
        if constexpr ( W > 1 )
        {
            // wave 1's theta to wave 0, which holds m
            if ( wv == 1 )
                msum[lane] = th;
            __syncthreads();
            th = msum[lane];
        }
        if ( do_theta )
        {
            const bool mpos = FRAC ? ( m_i > 0 ) : true;
            if ( !mpos )
                th = 0.0;
            else if ( valid && A.cnt[p] > 0 )
                th = 3.0 * th / m_i;
        }
    }
    if ( ( W > 1 && wv != 0 ) || !valid )
        return;
    if ( do_m )
        A.m[p] = m_i;
    if ( !do_theta )
        return;
    A.theta[p] = th;
    // ForceCoeffTag per-particle subexpressions (force_models/CabanaPD_LPS.hpp:131-132),
    // with the particle's own material coefficients in a multi-material specimen
    const double tc = A.mtype ? A.mat_tc[A.mtype[p]] : A.theta_coeff;
    const double sc = A.mtype ? A.mat_sc[A.mtype[p]] : A.s_coeff;
    A.lpsA[p] = tc * th / m_i;
    A.lpsB[p] = sc / m_i;
}

} // namespace

using ForceFn = void ( * )( const PDArgs*, const int32_t*, const int64_t*, int32_t, int32_t, int64_t, int32_t );
using LpsFn = void ( * )( const PDArgs*, const int32_t*, const int64_t*, int32_t, int64_t, int32_t, int32_t );

// The split and missing-site instances (waves: 1, 4 or 8 per slice; 1 with
// hole only), from the other translation units.
ForceFn splitForceRows( const PDArgs& a, int waves, bool hole );
ForceFn splitForceRowsFeat( const PDArgs& a, int waves, bool hole );
LpsFn splitLpsRows( const PDArgs& a, int waves, bool hole );

// Per-particle features of the force pass (kFeat* bits): several materials,
// temperature, plastic stretch (the LPS model has the first only).
inline int rowFeatures( const PDArgs& a )
{
    const bool lps = a.model == kLPS || a.model == kLinLPS;
    return ( a.mtype ? kFeatMT : 0 ) | ( !lps && a.temp ? kFeatTH : 0 ) | ( !lps && a.splas ? kFeatEP : 0 );
}

} // namespace pdk

#endif

// Device-side building blocks of the MHM/MHM_RP patch-group solver: ideal-gas conversions, the HLLC / HLLE /
// Roe interface solvers and the PLM slope limiters.  Written for gfx950 wave64 VALU; templated on the bulk
// arithmetic type R (float or double).  Pressure recovery E - |m|^2/(2 rho) goes through type A (double).
//
// Operation order follows the reference where it matters for parity:
//   Riemann solvers   src/Model_Hydro/CPU_Hydro/CPU_Shared_RiemannSolver_{HLLC:391-655, HLLE:301-698, Roe:87-711}.cpp
//   limiter + clamp   src/Model_Hydro/CPU_Hydro/CPU_Shared_DataReconstruction.cpp:403-430, 1917-2032
//   conversions       src/Model_Hydro/CPU_Hydro/CPU_Shared_FluUtility.cpp:209-551, 681-805
// Interface states arrive already rotated to the face normal with their pressure, 1/rho and sound speed
// evaluated once (per cell for the half step, per face for the full step) instead of inside every solve.
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>

namespace gamer_amd {

constexpr int NV = 5;

// ---------------- scalar helpers ----------------
__device__ __forceinline__ float  rcp( float x )  { return __builtin_amdgcn_rcpf( x ); }
__device__ __forceinline__ double rcp( double x )
{
   // hardware estimate r = (1 - e)/x and one third-order step r (1 + e + e^2): the estimate's relative error (about
   // 1e-7) enters cubed, so the result is within 1 ulp of 1/x for normal x, as two Newton steps gave with one
   // instruction and one link of the dependent chain more
   const double r = __builtin_amdgcn_rcp( x );
   const double e = __builtin_fma( -x, r, 1.0 );
   return __builtin_fma( r, __builtin_fma( e, e, e ), r );
}
__device__ __forceinline__ float  vsqrt( float x )  { return __builtin_amdgcn_sqrtf( x ); }
__device__ __forceinline__ double vsqrt( double x ) { return __builtin_sqrt( x ); }
// fused multiply-add written out where the rounding of an expression must not depend on how the compiler
// contracts it (the same face state is built by different code paths)
__device__ __forceinline__ float  fmad( float a, float b, float c )    { return __builtin_fmaf( a, b, c ); }
__device__ __forceinline__ double fmad( double a, double b, double c ) { return __builtin_fma( a, b, c ); }
template <typename R> __device__ __forceinline__ R vmax( R a, R b ) { return __builtin_fmax( a, b ); }
template <typename R> __device__ __forceinline__ R vmin( R a, R b ) { return __builtin_fmin( a, b ); }
template <typename R> __device__ __forceinline__ R vabs( R a )      { return __builtin_fabs( a ); }
template <typename R> __device__ __forceinline__ R vcopysign( R m, R s ) { return __builtin_copysign( m, s ); }

// reciprocal for the FP64 pressure recovery of the FP32-bulk kernels: hardware estimate + one Newton step, a
// relative error near 1e-14, far below what the float result keeps (two steps, as in rcp(double), for FP64)
__device__ __forceinline__ double rcp_recover( double x )
{
   const double r = __builtin_amdgcn_rcp( x );
   return __builtin_fma( r, __builtin_fma( -x, r, 1.0 ), r );
}

template <typename R> __device__ __forceinline__ double rcp_pres( double x ) { return sizeof( R ) == 4 ? rcp_recover( x ) : rcp( x ); }

// s = x^1/2 and y = x^-1/2 of a positive x, each within 1 ulp.  FP64: from the hardware reciprocal square root y and
// its third-order correction 1 + e/2 + 3/8 e^2, e = 1 - x y^2 (the estimate's error enters cubed); FP32: the
// hardware square root and reciprocal
__device__ __forceinline__ void sqrt_rsq( double x, double &s, double &y )
{
   const double y0 = __builtin_amdgcn_rsq( x ), s0 = x*y0;
   const double e = __builtin_fma( -s0, y0, 1.0 ), t = __builtin_fma( e, 0.375, 0.5 );
   s = __builtin_fma( s0*e, t, s0 );
   y = __builtin_fma( y0*e, t, y0 );
}
__device__ __forceinline__ void sqrt_rsq( float x, float &s, float &y ) { s = vsqrt( x );  y = rcp( s ); }

// sound speed (gamma P / rho)^1/2 from gp = gamma P, rho and ir = 1/rho.  Generic form sqrt(gp ir).  FP64:
// gp (gp rho)^-1/2 from the hardware reciprocal square root and two Newton steps, about 2 ulp, one transcendental
// and 9 instructions where the reciprocal's Newton steps and the IEEE square root take about 20; gp == 0 gives 0
// and NaN passes.  One third-order step on gp y instead has 4% more error in the HLLC fluxes of gas near rest (10% in
// MHM's) and is not faster (1331 patch groups with dt 446 us, this 438).  FP32 keeps the generic form: gp rho leaves its
// range for gases (1e-24 g/cm^3) whose gp/rho does not.  The derivative kernels define HYDRO_IEEE_SOUND_SPEED before
// including this header and keep the generic form, which their dual-number twins evaluate bit for bit.
template <typename R> __device__ __forceinline__ R sound_speed( R gp, R rho, R ir ) { (void)rho; return vsqrt( gp*ir ); }
#ifndef HYDRO_IEEE_SOUND_SPEED
template <> __device__ __forceinline__ double sound_speed<double>( double gp, double rho, double ir )
{
   (void)ir;
   const double a = gp*rho, h = 0.5*a;
   double y = __builtin_amdgcn_rsq( a );
   double r = __builtin_fma( -h*y, y, 0.5 );        // y (1.5 - a y^2 / 2) = y + y (0.5 - h y^2)
   y = __builtin_fma( y, r, y );
   r = __builtin_fma( -h*y, y, 0.5 );
   y = __builtin_fma( y, r, y );
   return ( gp == 0.0 ) ? 0.0 : gp*y;
}
#endif

// pressure floor that lets NaN through (FluUtility.cpp:681-690): a NaN compares false and is returned as is.
// One compare + select; max() would first have to quiet operands read from memory (IEEE mode).
template <typename R> __device__ __forceinline__ R floor_pres( R p, R pmin ) { return ( p < pmin ) ? pmin : p; }

// ---------------- raw buffer access ----------------
// Global loads and stores of the z-marching kernels go through a buffer descriptor per patch group: the 64-bit
// base stays in SGPRs and every access takes a lane-constant 32-bit byte offset plus a wave-uniform byte offset,
// so the march does no 64-bit address arithmetic per access.  The hardware range-checks each access against
// `bytes`: a read past it returns 0 and a write past it is dropped.  Word 3 = 0x00020000 is the gfx9-family
// raw-buffer format (32-bit data format, no swizzle).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_buf( const void *base, unsigned bytes )
{
   return __builtin_amdgcn_make_buffer_rsrc( const_cast<void *>( base ), (short)0, (int)bytes, 0x00020000 );
}
__device__ __forceinline__ void buf_load( __amdgpu_buffer_rsrc_t r, int voff, int soff, float &x )
{
   x = __builtin_bit_cast( float, __builtin_amdgcn_raw_buffer_load_b32( r, voff, soff, 0 ) );
}
__device__ __forceinline__ void buf_load( __amdgpu_buffer_rsrc_t r, int voff, int soff, double &x )
{
   x = __builtin_bit_cast( double, __builtin_amdgcn_raw_buffer_load_b64( r, voff, soff, 0 ) );
}
__device__ __forceinline__ void buf_store( float x, __amdgpu_buffer_rsrc_t r, int voff, int soff )
{
   __builtin_amdgcn_raw_buffer_store_b32( __builtin_bit_cast( unsigned, x ), r, voff, soff, 0 );
}
__device__ __forceinline__ void buf_store( double x, __amdgpu_buffer_rsrc_t r, int voff, int soff )
{
   using U2 = decltype( __builtin_amdgcn_raw_buffer_load_b64( __amdgpu_buffer_rsrc_t(), 0, 0, 0 ) );
   __builtin_amdgcn_raw_buffer_store_b64( __builtin_bit_cast( U2, x ), r, voff, soff, 0 );
}

// ---------------- solver constants ----------------
template <typename R>
struct Prm {
   R gamma, gm1, inv_gm1, min_dens, min_pres, min_eint, coeff;
   double dt_dh2, dt_dh, gm1_d, min_dens_d, min_pres_d, min_eint_d;
   int limiter;
};

// Multi-level batch description: optional per-PG (dt, dh) pairs in device memory (uneven AMR batches, local
// time steps) and an optional global work-queue counter for the persistent mode (each workgroup pulls tickets of
// `claim` consecutive patch groups until the queue is exhausted).  pg_dt_dh == nullptr: every PG uses Prm's dt/dh;
// counter == nullptr: the patch groups from `whole` on are split into `slabs` z slabs, one workgroup each, the others
// run one per workgroup (slab_split() in hydro_kernels.hpp).
struct Batch {
   const double *pg_dt_dh;
   unsigned     *counter;
   double        safety;
   int           claim;
   int           whole, slabs;
};

// c ? a : b as a select of values; of dual numbers, part by part (hydro_dual.hpp)
template <typename R> __device__ __forceinline__ R sel( bool c, R a, R b ) { return c ? a : b; }

// vector components of the axes (x, y, z) <-> those of a d-normal face (normal, two tangential ones).  d is a run-time
// value: one solve serves all three directions.  With a copy of the solve per direction, lanes of different directions
// ran them one after the other, and the compiler merged the copies' ends through scratch memory.
// FP64 derivative kernels, with the reverse sweeps and dual numbers in selects of values, copies -> run time: half-step
// reverse faces of 512 patch groups 674 -> 528 us, half-step fluxes 316 -> 264; dual numbers on 125: 157 -> 129 and full-step
// faces 124 -> 103.  Same bits.
template <typename R>
__device__ __forceinline__ void to_face( int d, R x, R y, R z, R &n, R &a, R &b )
{
   n = sel( d == 0, x, sel( d == 1, y, z ) );
   a = sel( d == 0, y, sel( d == 1, z, x ) );
   b = sel( d == 0, z, sel( d == 1, x, y ) );
}
template <typename R>
__device__ __forceinline__ void from_face( int d, R n, R a, R b, R &x, R &y, R &z )
{
   x = sel( d == 0, n, sel( d == 1, b, a ) );
   y = sel( d == 0, a, sel( d == 1, n, b ) );
   z = sel( d == 0, b, sel( d == 1, a, n ) );
}

// an interface state rotated to the face normal: conserved fields + derived quantities
template <typename R>
struct St { R d, mn, m1, m2, e, p, ir, cs, u; };

// ---------------- Riemann solvers (Davis wave speeds), flux returned in the rotated frame ----------------
template <typename R>
__device__ __forceinline__ void xflux_minus( const St<R> &s, R sp, R f[NV] )
{
   // physical x-flux minus sp*U (HLLC.cpp:600-612, HLLE.cpp:640-651), with (u - sp) factored out: one
   // instruction per transverse component instead of two
   const R us = s.u - sp;
   f[0] = s.mn - sp*s.d;
   f[1] = us*s.mn + s.p;
   f[2] = us*s.m1;
   f[3] = us*s.m2;
   f[4] = us*s.e + s.u*s.p;
}

template <typename R>
__device__ __forceinline__ void xflux( const St<R> &s, R f[NV] )
{
   f[0] = s.mn;
   f[1] = s.u*s.mn + s.p;
   f[2] = s.u*s.m1;
   f[3] = s.u*s.m2;
   f[4] = s.u*( s.e + s.p );
}

template <typename R>
__device__ __forceinline__ void rs_hlle( const St<R> &L, const St<R> &Q, R f[NV] )
{
   const R Z = (R)0;
   R sl = vmin( L.u - L.cs, Q.u - Q.cs );
   R sr = vmax( L.u + L.cs, Q.u + Q.cs );
   sl = vmin( sl, Z );
   sr = vmax( sr, Z );
   R fl[NV], fr[NV];
   xflux_minus( L, sl, fl );
   xflux_minus( Q, sr, fr );
   const bool both0 = ( sl == Z ) && ( sr == Z );
   const R inv = rcp( sr - sl );
#  pragma unroll
   for (int v=0; v<NV; v++) f[v] = sel( both0, fl[v], inv*( sr*fl[v] - sl*fr[v] ) );
}

template <typename R>
__device__ __forceinline__ void rs_hllc( const St<R> &L, const St<R> &Q, R pmin, R f[NV] )
{
   const R Z = (R)0, ONE = (R)1;
   const R wl1 = L.u - L.cs, wl2 = Q.u - Q.cs, wr1 = L.u + L.cs, wr2 = Q.u + Q.cs;
   const R wl = vmin( wl1, wl2 ), wr = vmax( wr1, wr2 );
   const R du = L.u - Q.u;
   const R tl =  L.d*sel( wl1 < wl2, L.cs, du + Q.cs );
   const R tr = -Q.d*sel( wr2 > wr1, Q.cs, du + L.cs );
   const R t2 = rcp( tl - tr );
   const R vs = t2*( L.p - Q.p + tl*L.u - tr*Q.u );
   R ps = t2*( tl*( Q.p + tr*Q.u ) - tr*( L.p + tl*L.u ) );
   ps = floor_pres( ps, pmin );

   const bool left = ( vs >= Z );
   St<R> s;
   s.d  = sel( left, L.d,  Q.d );   s.mn = sel( left, L.mn, Q.mn );  s.m1 = sel( left, L.m1, Q.m1 );
   s.m2 = sel( left, L.m2, Q.m2 );  s.e  = sel( left, L.e,  Q.e );   s.p  = sel( left, L.p,  Q.p );
   s.u  = sel( left, L.u,  Q.u );
   const R sp = sel( left, vmin( wl, Z ), vmax( wr, Z ) );
   R F[NV];
   xflux_minus( s, sp, F );
   const bool deg = left && ( vs == Z ) && ( sp == Z );
   const R t4 = rcp( vs - sp );
   const R cf = sel( deg, ONE, t4*vs );
   const R cs = sel( deg, Z, -t4*sp*ps );
   f[0] = cf*F[0];
   f[1] = cf*F[1] + cs;
   f[2] = cf*F[2];
   f[3] = cf*F[3];
   f[4] = cf*F[4] + cs*vs;
}

// Roe solver with the intermediate-state positivity check falling back to HLLE (Roe.cpp:87-711).  GAMER compiles
// that check only into builds whose RSOLVER is ROE (include/CUFLU.h:178-186, CHECK_INTERMEDIATE); CHECK = false is
// the Roe solve of the other builds, which CorrectUnphysical's first-order correction can still select.
template <typename R, bool CHECK = true>
__device__ __forceinline__ void rs_roe( const St<R> &L, const St<R> &Q, const Prm<R> &P, R f[NV] )
{
   const R Z = (R)0, HALF = (R)0.5;
   const R hl = L.ir*( L.e + L.p ), hr = Q.ir*( Q.e + Q.p );
   const R sql = vsqrt( L.d ), sqr = vsqrt( Q.d );
   const R rho = sql*sqr, irho = rcp( rho );
   const R isql = rcp( sql ), isqr = rcp( sqr ), isum = rcp( sql + sqr );
   const R u = isum*( isql*L.mn + isqr*Q.mn );
   const R v = isum*( isql*L.m1 + isqr*Q.m1 );
   const R w = isum*( isql*L.m2 + isqr*Q.m2 );
   const R V2 = u*u + v*v + w*w;
   const R H  = isum*( sql*hl + sqr*hr );
   R gpr = P.gm1*( H - HALF*V2 );
   gpr = P.gamma*irho*floor_pres( gpr*rho*rcp( P.gamma ), P.min_pres );
   const R a2 = gpr, a = vsqrt( a2 );
   const R e0 = u - a, e4 = u + a;

   R fl[NV], fr[NV];
   xflux( L, fl );
   xflux( Q, fr );
   if ( e0 >= Z ) { for (int k=0; k<NV; k++) f[k] = fl[k];  return; }
   if ( e4 <= Z ) { for (int k=0; k<NV; k++) f[k] = fr[k];  return; }

   const R j0 = Q.d - L.d, j1 = Q.mn - L.mn, j2 = Q.m1 - L.m1, j3 = Q.m2 - L.m2, j4 = Q.e - L.e;
   const R a2_ = j2 - v*j0;
   const R a3_ = j3 - w*j0;
   const R a1_ = P.gm1*rcp( a2 )*( j0*( H - u*u ) + u*j1 - j4 + v*a2_ + w*a3_ );
   const R a0_ = HALF*rcp( a )*( j0*( u + a ) - j1 - a*a1_ );
   const R a4_ = j0 - a0_ - a1_;

   // intermediate states after the 1st and 4th waves (the degenerate middle waves are skipped)
   if constexpr ( CHECK )
   {
      const R d1 = L.d + a0_, m1 = L.mn + a0_*e0, t1 = L.m1 + a0_*v, t2 = L.m2 + a0_*w, en1 = L.e + a0_*( H - u*a );
      const R ie1 = en1 - HALF*( m1*m1 + t1*t1 + t2*t2 )*rcp( d1 );
      bool bad = ( u > e0 ) && ( d1 <= Z || ie1*P.gm1 <= Z );
      const R d4 = d1 + a1_, m4 = m1 + a1_*u, s4 = t1 + a1_*v + a2_, r4 = t2 + a1_*w + a3_,
              en4 = en1 + a1_*( HALF*V2 ) + a2_*v + a3_*w;
      const R ie4 = en4 - HALF*( m4*m4 + s4*s4 + r4*r4 )*rcp( d4 );
      bad = bad || ( ( e4 > u ) && ( d4 <= Z || ie4*P.gm1 <= Z ) );
      if ( bad ) { rs_hlle( L, Q, f );  return; }
   }

   const R A0 = a0_*vabs( e0 ), A1 = a1_*vabs( u ), A2 = a2_*vabs( u ), A3 = a3_*vabs( u ), A4 = a4_*vabs( e4 );
   f[0] = HALF*( fl[0] + fr[0] - A0 - A1 - A4 );
   f[1] = HALF*( fl[1] + fr[1] - A0*e0 - A1*u - A4*e4 );
   f[2] = HALF*( fl[2] + fr[2] - A0*v - A1*v - A2 - A4*v );
   f[3] = HALF*( fl[3] + fr[3] - A0*w - A1*w - A3 - A4*w );
   f[4] = HALF*( fl[4] + fr[4] - A0*( H - u*a ) - A1*( HALF*V2 ) - A2*v - A3*w - A4*( H + u*a ) );
}

// ---------------- PLM reconstruction of one cell along one direction ----------------
// Limited slope (DataReconstruction.cpp:1917-2032), faces C -/+ slope/2, then clamp each face between the
// cell and its neighbour and mirror the other face about the cell value (:415-430).  LIM is the limiter id
// (include/Typedef.h:188-193) when known at compile time, or 0 to dispatch on `lim` at run time.
template <int LIM, typename R>
__device__ __forceinline__ R plm_slope( R sl, R sr, R lim_rt, int lim, R coeff )
{
   const R Z = (R)0;
   const R sc = (R)0.5*( sl + sr ), lr = sl*sr;
   const int L = ( LIM != 0 ) ? LIM : lim;
   R s;
   if ( L == 6 )      s = sc;                                                   // central
   else if ( L == 1 ) s = (R)2.0*lr*rcp( sl + sr );                             // van Leer
   else if ( L == 3 ) s = lr*( sl + sr )*rcp( sl*sl + sr*sr );                  // van Albada
   else
   {
      R m = vmin( vabs( sc ), vmin( vabs( sl*coeff ), vabs( sr*coeff ) ) );     // generalised MinMod
      if ( L == 4 ) m = vmin( vabs( (R)2.0*sl*sr*rcp( sl + sr ) ), m );          // + van Leer
      s = ( sc < Z ) ? -m : m;
   }
   (void)lim_rt;
   return ( lr > Z ) ? s : Z;
}

// clamp x into [min(a,b), max(a,b)] = median of (x, a, b)
__device__ __forceinline__ float  clamp_between( float x, float a, float b )   { return __builtin_amdgcn_fmed3f( x, a, b ); }
__device__ __forceinline__ double clamp_between( double x, double a, double b ) { return vmin( vmax( x, vmin( a, b ) ), vmax( a, b ) ); }

// van Leer + generalised MinMod slope without branches:
//   sign(sc) * min( theta|sl|, theta|sr|, |sc|, |2 sl sr/(sl+sr)| )  if sl*sr > 0, else 0.
// h = 2 sl sr / |sl+sr| equals the harmonic-mean magnitude when sl*sr > 0 and is <= 0 otherwise, or NaN when
// sl*sr underflows to zero while 1/|sl+sr| overflows (both slopes below about 1e-38 in FP32); max(h, 0) maps
// both cases to 0, which realises the sign test.  |sc| >= |harmonic mean| is implied and dropped.
template <typename R>
__device__ __forceinline__ R gminmod_mag( R h, R x ) { return vmin( x, vmax( h, (R)0 ) ); }
// FP32, x >= 0: med3(h, 0, x) is 0, h or x for h < 0, 0 <= h <= x or h > x, and 0 for a NaN h (with a NaN
// operand v_med3_f32 returns the minimum of the other two)
__device__ __forceinline__ float gminmod_mag( float h, float x ) { return __builtin_amdgcn_fmed3f( h, 0.0f, x ); }

template <typename R>
__device__ __forceinline__ R slope_vl_gminmod( R sl, R sr, R coeff )
{
   const R t = sl + sr;
   const R h = (R)2.0*( sl*sr )*rcp( vabs( t ) );
   return vcopysign( gminmod_mag( h, vmin( vabs( sl )*coeff, vabs( sr )*coeff ) ), t );
}

// Coefficients up to this value leave the PLM face clamps inactive under VL_GMINMOD (plm_face).
constexpr double VLGM_NOCLAMP_COEFF = 1.9999;

// Limiter id to instantiate a kernel with: 4 (VL_GMINMOD, resolved at compile time, face clamps left out) only
// for a MinMod coefficient <= VLGM_NOCLAMP_COEFF; otherwise 0, the run-time dispatch that keeps the clamps.
// The MinMod retries only lower the coefficient.
inline int kernel_limiter( int limiter, double minmod_coeff )
{
   return ( limiter == 4 && minmod_coeff <= VLGM_NOCLAMP_COEFF ) ? 4 : 0;
}

// Faces C -/+ s/2, the left one clamped between C and L, the right one 2C - (left face) clamped between C and R
// (DataReconstruction.cpp:415-430).  With LIM == 4 and plain FP32/FP64 arithmetic the clamps never act, and are
// left out: the slope is at most theta*|C-L|*(1+u)^2 <= 2|C-L| for theta <= 1.9999, so the exact C - s/2 lies
// in [min(C,L), max(C,L)], whose ends are representable, and rounding keeps it there; likewise s/2 <= |R-C|
// puts 2C - (left face) between C and R before its rounding.  Same bits as the clamped form; dual numbers keep
// the clamps for their derivative tie rules.
template <int LIM, typename R>
__device__ __forceinline__ void plm_face( R L, R C, R Rr, int lim, R coeff, R &fL, R &fR )
{
   const R s = ( LIM == 4 ) ? slope_vl_gminmod( C - L, Rr - C, coeff ) : plm_slope<LIM>( C - L, Rr - C, (R)0, lim, coeff );
   R fl, fr;
   if constexpr ( LIM == 4 && std::is_floating_point<R>::value )
   {
      fl = C - (R)0.5*s;
      fr = (R)2.0*C - fl;
   }
   else
   {
      fl = clamp_between( C - (R)0.5*s, C, L );
      fr = clamp_between( (R)2.0*C - fl, C, Rr );
   }
   fL = (R)2.0*C - fr;
   fR = fr;
}

// primitive face state (rho, vx, vy, vz, P) -> interface state rotated to direction d
// (Pri2Con, FluUtility.cpp:343-420; the solver takes the face pressure and velocity directly instead of
// recovering them from the conserved face state)
template <typename R>
__device__ __forceinline__ St<R> face_state( int d, const R w[NV], const Prm<R> &P )
{
   St<R> s;
   R vn, v1, v2;
   to_face( d, w[1], w[2], w[3], vn, v1, v2 );
   s.d  = w[0];
   s.mn = w[0]*vn;
   s.m1 = w[0]*v1;
   s.m2 = w[0]*v2;
   s.u  = vn;
   s.ir = rcp( w[0] );
   s.p  = floor_pres( w[4], P.min_pres );
   s.e  = fmad( (R)0.5*w[0], fmad( w[3], w[3], fmad( w[2], w[2], w[1]*w[1] ) ), w[4]*P.inv_gm1 );
   s.cs = sound_speed( P.gamma*s.p, s.d, s.ir );
   return s;
}

// conserved cell (with its pressure, 1/rho and sound speed) -> interface state rotated to direction d
template <typename R>
__device__ __forceinline__ St<R> cell_state( int d, const R c[NV], R p, R ir, R cs )
{
   St<R> s;
   s.d  = c[0];
   to_face( d, c[1], c[2], c[3], s.mn, s.m1, s.m2 );
   s.e  = c[4];
   s.p  = p;  s.ir = ir;  s.cs = cs;
   s.u  = ir*s.mn;
   return s;
}

// whether a flux component is NaN (an infinite component is not)
template <typename R>
__device__ __forceinline__ bool any_nan5( const R f[NV] )
{
   return f[0] != f[0] || f[1] != f[1] || f[2] != f[2] || f[3] != f[3] || f[4] != f[4];
}
// float: gfx950's v_maximum3_f32 propagates NaN, so two of them and one unordered compare test all five components
__device__ __forceinline__ bool any_nan5( const float f[NV] )
{
   const float m = __builtin_elementwise_maximum( __builtin_elementwise_maximum( f[0], f[1] ),
                                                  __builtin_elementwise_maximum( f[2], __builtin_elementwise_maximum( f[3], f[4] ) ) );
   return m != m;
}

// Riemann solve across a d-normal face; flux returned in the lab frame.  HLLC falls back to HLLE when a flux
// component is NaN (RSOLVER_RESCUE, CPU_FluidSolver_MHM.cpp:737-786, ComputeFlux.cpp:313-362).
template <int RS, typename R>
__device__ __forceinline__ void riemann( int d, const St<R> &L, const St<R> &Q, const Prm<R> &P, R out[NV] )
{
   R f[NV];
   if ( RS == 4 )
   {
      rs_hllc( L, Q, P.min_pres, f );
      if ( any_nan5( f ) ) rs_hlle( L, Q, f );
   }
   else if ( RS == 3 ) rs_hlle( L, Q, f );
   else                rs_roe( L, Q, P, f );
   out[0] = f[0];
   out[4] = f[4];
   from_face( d, f[1], f[2], f[3], out[1], out[2], out[3] );
}

// conserved face state -> interface state rotated to direction D, pressure recovered in FP64
template <int D, typename R>
__device__ __forceinline__ St<R> cons_state( const R c[NV], const Prm<R> &P )
{
   St<R> s;
   const double eint = (double)c[4] - 0.5*( (double)c[1]*c[1] + (double)c[2]*c[2] + (double)c[3]*c[3] )
                                      *rcp_pres<R>( (double)c[0] );
   s.d  = c[0];
   s.mn = c[1 + D];
   s.m1 = c[1 + ( D + 1 ) % 3];
   s.m2 = c[1 + ( D + 2 ) % 3];
   s.e  = c[4];
   s.p  = floor_pres( (R)( eint*P.gm1_d ), P.min_pres );
   s.ir = rcp( c[0] );
   s.u  = s.ir*s.mn;
   s.cs = sound_speed( P.gamma*s.p, s.d, s.ir );
   return s;
}

// ---------------- interface solves of the marching kernels ----------------
// One side of an interface: density, normal velocity u, pressure, sound speed, and by kind
//   KIND 0  an input cell (half step): a, b transverse momenta, e the energy
//   KIND 1  a primitive face (MHM_RP's full step): a, b transverse velocities, e the internal energy
//   KIND 2  a conserved face (MHM): mn the normal and a, b the transverse momenta, e the energy
// The marching kernels solve 35,712 interfaces per patch group, half of their instructions.  Measured per wave64
// instruction and SIMD, FP32 add, mul and fma issue in 2.2 cycles, min, max, compare and select in 4.8, reciprocals in
// 9.2 (FP64: 4.8 and 18.5), with two wait states between a compare and its select.  Against rs_hllc() of the
// derivative and correction kernels (the same HLLC fluxes, CPU_Shared_RiemannSolver_HLLC.cpp:391-655) this form
//   * takes tl = rho_L (u_L - w_L), tr = rho_R (w_R - u_R) from the wave speeds instead of by selects,
//   * takes the contact's speed and pressure as means of both sides with the weights tl and tr, the pressure's velocity
//     term from the difference: (tl (p_R + tr (u_L - u_R)) + tr p_L)/(tl + tr).  Where one side is much denser, neither
//     may be formed from a value of one side and a step: the step cancels the heavy side's pressure or the fast side's
//     velocity, and its rounding stays (p_L - tl x, x = (p_L - p_R - tr (u_L - u_R))/(tl + tr), was off by 6e-3 in the
//     light gas at a density contrast of 1e6 in FP32).  tl tr alone leaves the FP32 range for gases of 1e-24 g/cm^3,
//   * forms the flux as mass flux times (1, u, a, b, e) plus pressure terms, and, on faces, the energy only of the
//     side that the contact selects,
//   * leaves the vs == sp == 0 case to the NaN rescue: HLLE's flux there is the physical flux of the left state.
// Contraction is off and fused multiply-adds are written out, so that every code path that solves a face gets the
// same bits.  Roe and HLLE follow the same layout.  With the PLM below and the third-order reciprocals, on 4096 patch
// groups FP32 HLLC went from 0.696 to 0.654 ms, on 1331 FP64 HLLC from 0.594 to 0.516 ms, on 300 FP64 Roe from 0.445
// to 0.325 ms, on 1000 FP32 MHM HLLE from 0.264 to 0.257 ms (the kernels as they were then; the weighted means of HLLC's
// contact and the Newton steps of the FP64 sound speed cost 1.2% and gain 1.8% of that).  Against 80-bit arithmetic (L1 of
// five kinds of data) the outputs of a step are as far off as with rs_*(): FP64 Roe 0.993, FP32 HLLE 0.99 of it.  HLLE's
// FP32 mass flux has 1.08 times the error in a flow and half of it in static gas, where the sides cancel exactly.
template <typename R>
struct Side { R d, u, a, b, p, cs, e, mn; };

template <int D, typename R>
__device__ __forceinline__ Side<R> cell_side( const R q[8] )          // (rho, m, E, P, 1/rho, c_s); a, b: momenta
{
   Side<R> s;
   s.d = q[0];  s.u = q[6]*q[1 + D];  s.a = q[1 + ( D + 1 ) % 3];  s.b = q[1 + ( D + 2 ) % 3];
   s.e = q[4];  s.p = q[5];  s.cs = q[7];
   return s;
}
template <typename R>
__device__ __forceinline__ Side<R> cell_side_xy( const R q[8], bool dy )
{
   Side<R> s;
   s.d = q[0];  s.u = q[6]*( dy ? q[2] : q[1] );  s.a = dy ? q[3] : q[2];  s.b = dy ? q[1] : q[3];
   s.e = q[4];  s.p = q[5];  s.cs = q[7];
   return s;
}

// pressure floor that lets NaN through, as floor_pres; FP32 in one instruction (gfx950's v_maximum3_f32)
__device__ __forceinline__ double floor_nan( double p, double pmin ) { return floor_pres( p, pmin ); }
__device__ __forceinline__ float  floor_nan( float p, float pmin )   { return __builtin_elementwise_maximum( p, pmin ); }

template <typename R>
__device__ __forceinline__ void face_cs( Side<R> &s, R p, const Prm<R> &P )
{
   s.p  = floor_nan( p, P.min_pres );
   s.cs = sound_speed( P.gamma*s.p, s.d, rcp( s.d ) );
   s.e  = p*P.inv_gm1;                                                // internal energy of the unfloored pressure
}
// conserved face state (MHM's Hancock faces), its pressure recovered in FP64; a, b: momenta
template <int D, typename R>
__device__ __forceinline__ Side<R> cons_side( const R c[NV], const Prm<R> &P )
{
   const St<R> t = cons_state<D>( c, P );
   Side<R> s;
   s.d = t.d;  s.u = t.u;  s.a = t.m1;  s.b = t.m2;  s.p = t.p;  s.cs = t.cs;  s.e = t.e;  s.mn = t.mn;
   return s;
}
template <int D, typename R>
__device__ __forceinline__ Side<R> face_side( const R w[NV], const Prm<R> &P )   // primitive; a, b: velocities
{
   Side<R> s;
   s.d = w[0];  s.u = w[1 + D];  s.a = w[1 + ( D + 1 ) % 3];  s.b = w[1 + ( D + 2 ) % 3];
   face_cs( s, w[4], P );
   return s;
}
template <typename R>
__device__ __forceinline__ Side<R> face_side_xy( const R w[NV], bool dy, const Prm<R> &P )
{
   Side<R> s;
   s.d = w[0];  s.u = dy ? w[2] : w[1];  s.a = dy ? w[3] : w[2];  s.b = dy ? w[1] : w[3];
   face_cs( s, w[4], P );
   return s;
}
// energy density of a face side (Pri2Con)
template <typename R>
__device__ __forceinline__ R face_energy( R d, R u, R a, R b, R eint )
{
   return fmad( (R)0.5*d, fmad( b, b, fmad( a, a, u*u ) ), eint );
}

// N interfaces at a time, one operation of all of them after the other: a solve is a chain of about 25 dependent
// operations of 8 cycles each, and a wave that issues it alone fills half of its issue slots
template <int KIND, int N, typename R>
__device__ __forceinline__ void hllc_flux( const Side<R> L[N], const Side<R> Q[N], R pmin, R f[N][NV] )
{
   #pragma clang fp contract(off)
   const R Z = (R)0;
   R wl[N], wr[N], tl[N], tr[N], r[N], vs[N], ps[N], sp[N], t[N], m[N], cp[N], cs[N];
   bool left[N];
#  define GA_N _Pragma( "unroll" ) for (int n=0; n<N; n++)
   GA_N { wl[n] = vmin( L[n].u - L[n].cs, Q[n].u - Q[n].cs );  wr[n] = vmax( L[n].u + L[n].cs, Q[n].u + Q[n].cs ); }
   GA_N { tl[n] = L[n].d*( L[n].u - wl[n] );  tr[n] = Q[n].d*( wr[n] - Q[n].u ); }
   GA_N r[n]  = rcp( tl[n] + tr[n] );
   GA_N vs[n] = r[n]*fmad( tl[n], L[n].u, fmad( tr[n], Q[n].u, L[n].p - Q[n].p ) );
   GA_N ps[n] = floor_nan( r[n]*fmad( tl[n], fmad( tr[n], L[n].u - Q[n].u, Q[n].p ), tr[n]*L[n].p ), pmin );
   GA_N left[n] = ( vs[n] >= Z );
   GA_N sp[n] = left[n] ? vmin( wl[n], Z ) : vmax( wr[n], Z );
   GA_N t[n]  = rcp( vs[n] - sp[n] );
   R d[N], u[N], a[N], b[N], p[N], e[N], mn[N];
   GA_N
   {
      d[n] = left[n] ? L[n].d : Q[n].d;  u[n] = left[n] ? L[n].u : Q[n].u;  a[n] = left[n] ? L[n].a : Q[n].a;
      b[n] = left[n] ? L[n].b : Q[n].b;  p[n] = left[n] ? L[n].p : Q[n].p;  e[n] = left[n] ? L[n].e : Q[n].e;
      mn[n] = left[n] ? L[n].mn : Q[n].mn;
   }
   GA_N if ( KIND == 1 ) e[n] = face_energy( d[n], u[n], a[n], b[n], e[n] );
   GA_N { const R cf = t[n]*vs[n];  m[n] = cf*( u[n] - sp[n] );  cp[n] = cf*p[n];  cs[n] = -( t[n]*sp[n] )*ps[n];
          f[n][0] = KIND == 2 ? cf*fmad( -sp[n], d[n], mn[n] ) : m[n]*d[n]; }
   GA_N
   {
      const R pp = cp[n] + cs[n];
      f[n][1] = KIND == 2 ? fmad( m[n], mn[n], pp ) : fmad( f[n][0], u[n], pp );
      f[n][2] = ( KIND == 1 ? f[n][0] : m[n] )*a[n];
      f[n][3] = ( KIND == 1 ? f[n][0] : m[n] )*b[n];
      f[n][4] = fmad( m[n], e[n], fmad( cp[n], u[n], cs[n]*vs[n] ) );
   }
#  undef GA_N
}

template <int KIND, typename R>
__device__ __forceinline__ void hlle_flux( const Side<R> &L, const Side<R> &Q, R f[NV] )
{
   #pragma clang fp contract(off)
   const R Z = (R)0;
   const R sl = vmin( vmin( L.u - L.cs, Q.u - Q.cs ), Z ), sr = vmax( vmax( L.u + L.cs, Q.u + Q.cs ), Z );
   const bool both0 = ( sl == Z ) && ( sr == Z );
   const R inv = rcp( sr - sl );
   const R cl = both0 ? (R)1 : inv*sr, cr = both0 ? Z : -( inv*sl );
   const R ml = cl*( L.u - sl ), mr = cr*( Q.u - sr );                // mass flux per density of each side
   const R fl = KIND == 2 ? cl*fmad( -sl, L.d, L.mn ) : ml*L.d, fr = KIND == 2 ? cr*fmad( -sr, Q.d, Q.mn ) : mr*Q.d;
   const R pl = cl*L.p, pr = cr*Q.p;
   const R el = KIND == 1 ? face_energy( L.d, L.u, L.a, L.b, L.e ) : L.e, er = KIND == 1 ? face_energy( Q.d, Q.u, Q.a, Q.b, Q.e ) : Q.e;
   const R al = KIND == 1 ? fl : ml, ar = KIND == 1 ? fr : mr;
   f[0] = fl + fr;
   f[1] = KIND == 2 ? fmad( ml, L.mn, fmad( mr, Q.mn, pl + pr ) ) : fmad( fl, L.u, fmad( fr, Q.u, pl + pr ) );
   f[2] = fmad( al, L.a, ar*Q.a );
   f[3] = fmad( al, L.b, ar*Q.b );
   f[4] = fmad( ml, el, fmad( mr, er, fmad( pl, L.u, pr*Q.u ) ) );
}

// Roe with the intermediate-state check (Roe.cpp:87-711).  Square roots and reciprocals of the densities and of the
// sound speed come in pairs from one reciprocal square root each; rs_roe() of the derivative kernels takes 3 IEEE
// square roots and 8 reciprocals.
template <int KIND, typename R>
__device__ __forceinline__ void roe_flux( const Side<R> &L, const Side<R> &Q, const Prm<R> &P, R f[NV] )
{
   #pragma clang fp contract(off)
   const R Z = (R)0, HALF = (R)0.5;
   R sql, sqr, isl, isr;
   sqrt_rsq( L.d, sql, isl );
   sqrt_rsq( Q.d, sqr, isr );
   const R isum = rcp( sql + sqr );
   const R el = KIND == 1 ? face_energy( L.d, L.u, L.a, L.b, L.e ) : L.e, er = KIND == 1 ? face_energy( Q.d, Q.u, Q.a, Q.b, Q.e ) : Q.e;
   const R l1 = KIND == 1 ? L.d*L.a : L.a, l2 = KIND == 1 ? L.d*L.b : L.b, r1 = KIND == 1 ? Q.d*Q.a : Q.a, r2 = KIND == 1 ? Q.d*Q.b : Q.b;
   const R ln = KIND == 2 ? L.mn : L.d*L.u, rn = KIND == 2 ? Q.mn : Q.d*Q.u;
   const R u = isum*( KIND == 2 ? fmad( isl, ln, isr*rn ) : fmad( sql, L.u, sqr*Q.u ) );
   const R v = isum*( KIND == 1 ? fmad( sql, L.a, sqr*Q.a ) : fmad( isl, L.a, isr*Q.a ) );
   const R w = isum*( KIND == 1 ? fmad( sql, L.b, sqr*Q.b ) : fmad( isl, L.b, isr*Q.b ) );
   const R V2h = HALF*fmad( w, w, fmad( v, v, u*u ) );
   const R H  = isum*fmad( isl, el + L.p, isr*( er + Q.p ) );
   // a^2 = (gamma-1)(H - V^2/2), its pressure a^2 rho/gamma floored as the reference does
   const R g0 = P.gm1*( H - V2h ), irho = isl*isr, gmin = P.gamma*P.min_pres*irho;
   const R a2 = floor_nan( g0, gmin );
   R a, ia;
   sqrt_rsq( a2, a, ia );
   a = ( a2 == Z ) ? Z : a;
   const R e0 = u - a, e4 = u + a;
   if ( e0 >= Z || e4 <= Z )                                          // supersonic: the upwind side's flux
   {
      const bool left = ( e0 >= Z );
      const R un = left ? L.u : Q.u, p = left ? L.p : Q.p;
      f[0] = left ? ln : rn;
      f[1] = fmad( f[0], un, p );
      f[2] = un*( left ? l1 : r1 );
      f[3] = un*( left ? l2 : r2 );
      f[4] = un*( ( left ? el : er ) + p );
      return;
   }
   const R j0 = Q.d - L.d, j1 = rn - ln, j2 = r1 - l1, j3 = r2 - l2, j4 = er - el;
   const R a2_ = fmad( -v, j0, j2 ), a3_ = fmad( -w, j0, j3 );
   const R a1_ = ( P.gm1*( ia*ia ) )*( fmad( j0, fmad( -u, u, H ), fmad( u, j1, -j4 ) ) + fmad( v, a2_, w*a3_ ) );
   const R a0_ = ( HALF*ia )*( fmad( j0, e4, -j1 ) - a*a1_ );
   const R a4_ = j0 - a0_ - a1_;
   const R ua = u*a, hm = H - ua, hp = H + ua;
   // intermediate states after the 1st and 4th waves (the degenerate middle waves are skipped)
   const R d1 = L.d + a0_, m1 = fmad( a0_, e0, ln ), t1 = fmad( a0_, v, l1 ), t2 = fmad( a0_, w, l2 ), n1 = fmad( a0_, hm, el );
   const R i1 = n1 - HALF*fmad( t2, t2, fmad( t1, t1, m1*m1 ) )*rcp( d1 );
   const R d4 = d1 + a1_, m4 = fmad( a1_, u, m1 ), s4 = fmad( a1_, v, t1 ) + a2_, r4 = fmad( a1_, w, t2 ) + a3_,
           n4 = fmad( a1_, V2h, n1 ) + fmad( a2_, v, a3_*w );
   const R i4 = n4 - HALF*fmad( r4, r4, fmad( s4, s4, m4*m4 ) )*rcp( d4 );
   if ( ( ( u > e0 ) && ( d1 <= Z || i1*P.gm1 <= Z ) ) || ( ( e4 > u ) && ( d4 <= Z || i4*P.gm1 <= Z ) ) )
   {
      hlle_flux<KIND>( L, Q, f );
      return;
   }
   const R A0 = a0_*vabs( e0 ), A1 = a1_*vabs( u ), A2 = a2_*vabs( u ), A3 = a3_*vabs( u ), A4 = a4_*vabs( e4 ), S = A0 + A1 + A4;
   f[0] = HALF*( ( ln + rn ) - S );
   f[1] = HALF*( ( fmad( ln, L.u, L.p ) + fmad( rn, Q.u, Q.p ) ) - fmad( A0, e0, fmad( A1, u, A4*e4 ) ) );
   f[2] = HALF*( fmad( L.u, l1, Q.u*r1 ) - fmad( S, v, A2 ) );
   f[3] = HALF*( fmad( L.u, l2, Q.u*r2 ) - fmad( S, w, A3 ) );
   f[4] = HALF*( fmad( L.u, el + L.p, Q.u*( er + Q.p ) ) - fmad( A0, hm, fmad( A1, V2h, fmad( A2, v, fmad( A3, w, A4*hp ) ) ) ) );
}

// N solves in the rotated frames; they share one branch to the HLLE rescue of NaN fluxes (RSOLVER_RESCUE), so that
// nothing separates them for the scheduler
template <int RS, int KIND, int N, typename R>
__device__ __forceinline__ void solve_n( const Side<R> L[N], const Side<R> Q[N], const Prm<R> &P, R f[N][NV] )
{
   if ( RS == 4 )
   {
      hllc_flux<KIND, N>( L, Q, P.min_pres, f );
      bool nan[N], any = false;
#     pragma unroll
      for (int n=0; n<N; n++) { nan[n] = any_nan5( f[n] );  any = any || nan[n]; }
      if ( any )
#        pragma unroll
         for (int n=0; n<N; n++) if ( nan[n] ) hlle_flux<KIND>( L[n], Q[n], f[n] );
   }
   else
#     pragma unroll
      for (int n=0; n<N; n++)
         if ( RS == 3 ) hlle_flux<KIND>( L[n], Q[n], f[n] );
         else           roe_flux<KIND>( L[n], Q[n], P, f[n] );
}
// rotated flux -> lab frame, of a D-normal face and of an x- or y-normal one chosen per lane
template <int D, typename R>
__device__ __forceinline__ void to_lab( const R f[NV], R out[NV] )
{
   out[0] = f[0];  out[1 + D] = f[1];  out[1 + ( D + 1 ) % 3] = f[2];  out[1 + ( D + 2 ) % 3] = f[3];  out[4] = f[4];
}
template <typename R>
__device__ __forceinline__ void to_lab_xy( const R f[NV], bool dy, R out[NV] )
{
   out[0] = f[0];  out[1] = dy ? f[3] : f[1];  out[2] = dy ? f[1] : f[2];  out[3] = dy ? f[2] : f[3];  out[4] = f[4];
}
// flux across a D-normal interface in the lab frame
template <int RS, int D, int KIND, typename R>
__device__ __forceinline__ void solve( const Side<R> &L, const Side<R> &Q, const Prm<R> &P, R out[NV] )
{
   const Side<R> l[1] = { L }, q[1] = { Q };
   R f[1][NV];
   solve_n<RS, KIND, 1>( l, q, P, f );
   to_lab<D>( f[0], out );
}
template <int RS, int KIND, typename R>
__device__ __forceinline__ void solve_xy( const Side<R> &L, const Side<R> &Q, const Prm<R> &P, bool dy, R out[NV] )
{
   const Side<R> l[1] = { L }, q[1] = { Q };
   R f[1][NV];
   solve_n<RS, KIND, 1>( l, q, P, f );
   to_lab_xy( f[0], dy, out );
}

// ---------------- PLM of the marching kernels ----------------
// plm_face for all five fields of a cell.  VL_GMINMOD (LIM == 4) takes half slopes: h = sl sr / |sl + sr|, the limit
// theta/2 min(|sl|, |sr|) from one min and one mul, and mirrors the left face C - h once, where the reference mirrors
// it back too (the same up to one rounding); no clamp can act (see plm_face).  12 instructions a pair instead of 17.  The
// run-time limiter is dispatched once per cell and direction, not per field.
template <typename R>
__device__ __forceinline__ void plm_pair4( R L, R C, R Rr, R coeff, R &fL, R &fR )
{
   #pragma clang fp contract(off)
   const R sl = C - L, sr = Rr - C, t = sl + sr;
   const R h = ( sl*sr )*rcp( vabs( t ) );
   const R s = vcopysign( gminmod_mag( h, ( (R)0.5*coeff )*vmin( vabs( sl ), vabs( sr ) ) ), t );
   fL = C - s;
   fR = fmad( (R)2, C, -fL );
}
template <int L_, typename R>
__device__ __forceinline__ void plm_cell_as( const R L[NV], const R C[NV], const R Rr[NV], R coeff, R fL[NV], R fR[NV] )
{
#  pragma unroll
   for (int v=0; v<NV; v++)
   {
      const R s = plm_slope<L_>( C[v] - L[v], Rr[v] - C[v], (R)0, L_, coeff );
      const R fl = clamp_between( C[v] - (R)0.5*s, C[v], L[v] );
      fR[v] = clamp_between( (R)2.0*C[v] - fl, C[v], Rr[v] );
      fL[v] = (R)2.0*C[v] - fR[v];
   }
}
template <int LIM, typename R>
__device__ __forceinline__ void plm_cell( const R L[NV], const R C[NV], const R Rr[NV], const Prm<R> &P, R fL[NV], R fR[NV] )
{
   if constexpr ( LIM == 4 )
   {
#     pragma unroll
      for (int v=0; v<NV; v++) plm_pair4( L[v], C[v], Rr[v], P.coeff, fL[v], fR[v] );
   }
   else switch ( P.limiter )
   {
      case 1:  plm_cell_as<1>( L, C, Rr, P.coeff, fL, fR );  break;
      case 2:  plm_cell_as<2>( L, C, Rr, P.coeff, fL, fR );  break;
      case 3:  plm_cell_as<3>( L, C, Rr, P.coeff, fL, fR );  break;
      case 4:  plm_cell_as<4>( L, C, Rr, P.coeff, fL, fR );  break;
      default: plm_cell_as<6>( L, C, Rr, P.coeff, fL, fR );  break;
   }
}

template <typename IO> struct IOLim;
template <> struct IOLim<double> { static constexpr double huge = 1.7976931348623157e308; static constexpr double eps = 2.2204460492503131e-16; };
template <> struct IOLim<float>  { static constexpr float  huge = 3.40282346638528859812e+38f; static constexpr float eps = 1.1920928955078125e-07f; };

// full-step update of one output cell, accumulated in FP64, + the CONS-mode unphysical check on the stored
// values (FullStepUpdate.cpp:106-235, FluUtility.cpp:843-940)
template <typename R, typename IO>
__device__ __forceinline__ bool full_cell( const IO u[NV], const R dfxy[NV], const R fzl[NV], const R fzu[NV],
                                           const Prm<R> &P, IO o[NV] )
{
   #pragma clang fp contract(off)      // fused where written: every launch mode rounds alike
#  pragma unroll
   for (int v=0; v<NV; v++)
      o[v] = (IO)fmad( -P.dt_dh, (double)dfxy[v] + ( (double)fzu[v] - (double)fzl[v] ), (double)u[v] );
   // each test is one ordered compare, false for NaN: "not finite-and-in-range" covers the NaN test too
   const IO huge = IOLim<IO>::huge, Z = (IO)0;
   bool ok = ( vabs( o[1] ) <= huge ) && ( vabs( o[2] ) <= huge ) && ( vabs( o[3] ) <= huge );
   ok = ok && ( o[0] > Z && o[0] <= huge ) && ( o[4] > Z && o[4] <= huge );
   const IO ei = fmad( (IO)-0.5*fmad( o[3], o[3], fmad( o[2], o[2], o[1]*o[1] ) ), rcp( o[0] ), o[4] );
   ok = ok && ( ei >= (IO)-3.0*o[4]*IOLim<IO>::eps && ei <= huge );
   return !ok;
}

// Hancock half-step advance of the six face states of one cell (MHM only;
// DataReconstruction.cpp:2063-2160): fluxes of the conserved face states (pressure recovered in FP64),
// U_f -= dt/(2dh) * sum_d (F_{d,R} - F_{d,L}), then either a reset of all six faces to the cell value if
// any face density/energy or input face pressure is invalid, or density and internal-energy floors.
template <typename R, typename IO>
__device__ __forceinline__ void hancock( R fc[6][NV], const R fcp[6][NV], const R ucell[NV], const Prm<R> &P )
{
   R F[6][NV];
#  pragma unroll
   for (int f=0; f<6; f++)
   {
      const int d = f/2;
      const R mn = fc[f][1 + d];
      const double eint = (double)fc[f][4] - 0.5*( (double)fc[f][1]*fc[f][1] + (double)fc[f][2]*fc[f][2]
                                                    + (double)fc[f][3]*fc[f][3] )*rcp_pres<R>( (double)fc[f][0] );
      const R p  = floor_pres( (R)( eint*P.gm1_d ), P.min_pres );
      const R vn = rcp( fc[f][0] )*mn;
      F[f][0] = mn;
      F[f][1] = vn*fc[f][1];
      F[f][2] = vn*fc[f][2];
      F[f][3] = vn*fc[f][3];
      F[f][1 + d] += p;
      F[f][4] = vn*( fc[f][4] + p );
   }
   const R dt_dh2 = (R)P.dt_dh2;
#  pragma unroll
   for (int v=0; v<NV; v++)
   {
      const R dF = dt_dh2*( F[1][v] - F[0][v] + F[3][v] - F[2][v] + F[5][v] - F[4][v] );
#     pragma unroll
      for (int f=0; f<6; f++) fc[f][v] -= dF;
   }
   const R tiny = ( sizeof(R) == 8 ) ? (R)2.2250738585072014e-308 : (R)1.17549435e-38f;
   const R huge = (R)IOLim<IO>::huge;
   bool reset = false;
#  pragma unroll
   for (int f=0; f<6; f++)
   {
      const R d = fc[f][0], e = fc[f][4], pr = fcp[f][4];
      reset |= ( d < tiny || d > huge || d != d ) || ( e < tiny || e > huge || e != e ) ||
               ( pr < (R)0 || pr > huge || pr != pr );
   }
   if ( reset )
   {
#     pragma unroll
      for (int f=0; f<6; f++)
#        pragma unroll
         for (int v=0; v<NV; v++) fc[f][v] = ucell[v];
   }
   else
   {
#     pragma unroll
      for (int f=0; f<6; f++)
      {
         fc[f][0] = vmax( fc[f][0], P.min_dens );
         const double ke  = 0.5*( (double)fc[f][1]*fc[f][1] + (double)fc[f][2]*fc[f][2] + (double)fc[f][3]*fc[f][3] )
                            *rcp_pres<R>( (double)fc[f][0] );
         const double ein = (double)fc[f][4] - ke;
         const double eo  = ( ein == ein ) ? __builtin_fmax( ein, P.min_eint_d ) : ein;
         if ( ein != eo ) fc[f][4] = (R)( (double)fc[f][4] - ein + eo );
      }
   }
}

// primitive -> conserved (Pri2Con, FluUtility.cpp:343-420)
template <typename R>
__device__ __forceinline__ void pri2con( const R w[NV], R c[NV], const Prm<R> &P )
{
   c[0] = w[0];
   c[1] = w[0]*w[1];  c[2] = w[0]*w[2];  c[3] = w[0]*w[3];
   c[4] = (R)0.5*( c[1]*c[1] + c[2]*c[2] + c[3]*c[3] )*rcp( w[0] ) + w[4]*P.inv_gm1;
}

// max_d(|v_d| + c_s) of one cell, pressure recovered in FP64 (CPU_dtSolver_HydroCFL.cpp:104-190)
template <typename IO>
__device__ __forceinline__ IO cell_cfl( const IO u[NV], double gamma, double gm1, double min_pres )
{
   const double d = (double)u[0], ir = 1.0/d;
   double p = ( (double)u[4] - 0.5*( (double)u[1]*u[1] + (double)u[2]*u[2] + (double)u[3]*u[3] )*ir )*gm1;
   p = ( p == p ) ? __builtin_fmax( p, min_pres ) : p;
   const IO cs = (IO)__builtin_sqrt( gamma*p*ir );
   const IO ri = (IO)ir;
   const IO vx = vabs( u[1] )*ri, vy = vabs( u[2] )*ri, vz = vabs( u[3] )*ri;
   return vmax( vmax( cs + vx, cs + vy ), cs + vz );
}

// Fused CFL of one patch group: each lane holds the maxima of its output column in the two z-halves; the 8
// patches (px + 2 py + 4 pz, x fastest) are reduced with wave64 butterflies and LDS across the 4 waves, in the
// I/O type (the reference computes dt in `real`, CPU_dtSolver_HydroCFL.cpp:62-209).
// Called by every lane of the workgroup (waves 0-3 hold the output columns); writes dt[8] = dh_safety / max, or only
// the four patches of z half `half` if that is 0 or 1.
template <typename IO>
__device__ __forceinline__ void fused_dt( const IO cfl[2], int pxy, IO (*red)[4], IO *dt, double dh_safety, int half )
{
   const int tid = threadIdx.x, w = tid >> 6;
   if ( w < 4 )                      // the output columns live on waves 0-3; further waves hold ghost columns
#  pragma unroll
   for (int pz=0; pz<2; pz++)
#     pragma unroll
      for (int q=0; q<4; q++)
      {
         IO m = ( pxy == q ) ? cfl[pz] : (IO)0;
#        pragma unroll
         for (int o = 32; o > 0; o >>= 1) m = vmax( m, __shfl_xor( m, o, 64 ) );
         if ( ( tid & 63 ) == 0 ) red[q + 4*pz][w] = m;
      }
   __syncthreads();
   if ( tid < 8 && ( half < 0 || ( tid >> 2 ) == half ) )
   {
      const IO m = vmax( vmax( red[tid][0], red[tid][1] ), vmax( red[tid][2], red[tid][3] ) );
      dt[tid] = (IO)( dh_safety / (double)m );
   }
}

} // namespace gamer_amd

// MHM_RP (MUSCL-Hancock with Riemann-solver prediction) patch-group kernel for gfx950.
//
// One 512-lane workgroup updates one patch group: 22^3 input cells (16^3 interior + 3 ghost zones) ->
// 16^3 output cells + 9 coarse-fine flux planes.  The reference runs the same update as eight global-memory
// phases over the whole 22^3 block (src/Model_Hydro/CPU_Hydro/CPU_FluidSolver_MHM.cpp:263-589, ~2.9 MB of
// scratch per patch group in FP64).  Here the workgroup marches along z, one input plane per step, and keeps
// every intermediate on chip:
//
//   * Waves 0-3 (the column waves): lane t owns the output column (i,j) = (3 + t%16, 3 + output_row(t)), with
//     everything that couples planes along z in its registers: the previous input plane, the half-step z-flux, the
//     last three half-step primitive planes, the lower z-face state and the last full-step z-flux.  It does the
//     column's z work, its y work and the updates.
//   * Waves 4-7 (the side waves): lane g does the x reconstruction and the full-step x face of the column of lane g,
//     which need no z history.  Besides, side waves 0-1 each own one "arm" ghost column of the half step
//     (arm_column()); side waves 2-3 do the half-step x faces of two columns a lane; side wave 2 one single half-step
//     face per plane (face_task()), side wave 3 one reconstructed column next to the block and half of its lanes the
//     full-step face between the two (edge_column()); all of them stage the input planes.
//   * x/y neighbours go through LDS, one plane at a time.  A lane-private LDS ring keeps the input cells of the
//     output column for the planes between load and full-step update, so every input value is read from HBM once.
//
// Step t, input plane t staged (planes in input coordinates), with its two barriers:
//   [A] half-step z-flux at t-1/2 and half-step cell of plane t-1, half-step x/y fluxes of plane t, PLM of plane
//       r = t-2, x/y flux differences of plane t-3
//   [H] x/y half-step flux differences of plane t, half-step plane t-1 into LDS, full-step fluxes of plane r (x/y) and
//       at r-1/2 (z), full-step update and output of plane t-3, input plane t+1 into LDS
// Every LDS array is written in one interval and read in the other.  All branches around the barriers depend only on
// t, so every barrier is reached by the whole workgroup.
//
// What bounds it: a plane takes about 5,500 cycles (FP32), and a wave's chain of dependent operations (8 cycles each, 128
// and more for an LDS read) is most of that at any occupancy; the vector units issue half of the time (FP64) or three
// quarters (FP32).  So the work is split for the longest wave of each interval, by clock readings at the barriers:
// [A] columns 2,600, arms 2,500, side waves 2-3 2,500; [H] 2,700 to 3,000.  The previous layout, with all x work on the
// column waves and four barriers a plane, left the side waves waiting.  A spill costs more here than its instructions: a
// reload, also one placed in front of the loop, makes its first use wait for all outstanding prefetches and stores on
// every plane (the default kernel with 80 instead of 16 bytes of scratch a lane: 563 against 532 us).  FP64 HLLC and HLLE
// and FP32 HLLE with VL_GMINMOD run without scratch; FP32 HLLC holds 20 bytes (queue 40), Roe 88 (FP64 64 to 76), the
// kernels with a run-time limiter 40 to 92 (FP64 72 to 88), where 128 (FP64 256) registers do not hold the limiter's or
// Roe's temporaries beside the z history.  On 4096 patch groups FP32 654 -> 528 us (HLLE on 2048: 389 -> 249 before the
// cheaper solves of both), on 1331 FP64 516 -> 463 us; with HLLC's contact as weighted means 543 and 438 (with dt).

#include "hydro_math.hpp"
#include "hydro_kernels.hpp"

namespace gamer_amd {

namespace {

constexpr int NX  = 22;          // FLU_NXT for MHM_RP
constexpr int NC  = NX*NX;       // columns per plane
constexpr int PS  = 16;          // PS2
constexpr int NK  = 256;         // output columns (lanes of waves 0-3)
constexpr int NT  = 512;         // lanes per workgroup
constexpr int FS  = 18;          // LDS row stride of the full-step face arrays: rows 8 apart are 16 banks apart modulo 32
constexpr int HX  = 20*NX, HY = 21*NX, FX = 16*FS, FY = 17*FS;

// output row (j - 3) of lane t: wave w takes rows w, w+8, w+4, w+12, 16 lanes each.  The neighbour reads of a
// plane in LDS (row stride NX = 22 words) then put the two rows of each half wave 176 words apart, 16 banks
// modulo 32, so they meet no bank conflict, where rows 4w..4w+3 collided on 6 of 16 lanes per row pair.
__device__ __forceinline__ int output_row( int t )
{
   const int q = ( t & 63 ) >> 4;
   return ( t >> 6 ) + 8*( q & 1 ) + 4*( q >> 1 );
}

// The reconstruction reads half-step cells only in three slabs: the 16^2 output columns over z = 1..20, and the
// "arm" columns (i or j in {1,2,19,20}, the other in 3..18) over z = 3..18 -- 7,168 of the 8,000 cells the
// reference updates (CPU_FluidSolver_MHM.cpp:656-666 takes the whole 20^3 block).  Those cells need 22,656 of
// its 25,200 half-step faces.  The ghost work of the side waves is laid out so that each wave runs one task kind
// over one z range and skips the rest with wave-uniform branches:
//   side wave 0: the 64 arms next to the output block (i or j in {2,19}): half-step cell + low x and y faces
//   side wave 1: the 64 outer arms (i or j in {1,20}): the same
//   side wave 2: 40 single half-step faces (one x or y face per lane, read by an arm or output cell but owned by a
//           column that is neither): the low x face of column (21,j) at z = 3..18 and of column (19,j) at the
//           other planes, where the output cell (18,j) still needs it (and the y analogue); and the low x faces
//           of (19, {1,2,19,20}) and low y faces of ({1,2,19,20}, 19) at z = 3..18
// Arm column of side lane t (side waves 0-1); false = none.
__device__ __forceinline__ bool arm_column( int t, int &i, int &j )
{
   if ( t >= 128 ) { i = j = 0;  return false; }
   const int k = t & 63, a = 3 + ( k & 15 ), s = ( k >> 4 ) & 1;
   const int e = ( t < 64 ) ? ( s ? 19 : 2 ) : ( s ? 20 : 1 );
   if ( k < 32 ) { i = e;  j = a; }
   else          { i = a;  j = e; }
   return true;
}

// single half-step face of side lane t (side wave 2) at a plane (mid: a plane with arm cells): the column whose low
// face it is and whether the face is y-normal; false = no face at this plane
__device__ __forceinline__ bool face_task( int t, bool mid, int &c, bool &dy )
{
   const int k = t - 128;
   int i, j;
   dy = false;
   if ( k < 0 || k >= 40 ) return false;
   if ( k < 32 )
   {
      const int a = 3 + ( k & 15 ), e = mid ? 21 : 19;
      dy = ( k >= 16 );
      i = dy ? a : e;
      j = dy ? e : a;
   }
   else
   {
      const int q = k & 3, e = ( q < 2 ) ? 1 + q : 17 + q;     // 1, 2, 19, 20
      dy = ( k >= 36 );
      i = dy ? e : 19;
      j = dy ? 19 : e;
      if ( !mid ) return false;
   }
   c = i + NX*j;
   return true;
}

// column next to the output block reconstructed by side lane t of side wave 3 (along y if dy): the columns 2 give the
// left states of the block's first faces; the columns 19 own the full-step flux on the block's last face (face)
__device__ __forceinline__ bool edge_column( int t, int &i, int &j, bool &dy, bool &face )
{
   const int k = t - 192;
   dy = ( k >= 32 );
   const int e = k & 31;
   face = ( e >= 16 );
   const int a = face ? 19 : 2, b = 3 + ( e & 15 );
   i = dy ? b : a;
   j = dy ? a : b;
   return ( k >= 0 && k < 64 );
}

// cell quantities of one input cell: conserved + pressure (recovered in FP64), 1/rho, sound speed
template <typename R, typename IO>
__device__ __forceinline__ void derive_cell( const IO u[NV], R q[8], const Prm<R> &P )
{
   #pragma clang fp contract(off)      // fused where written: every launch mode rounds alike
   const double d = (double)u[0], mx = (double)u[1], my = (double)u[2], mz = (double)u[3], e = (double)u[4];
   const double eint = fmad( -0.5*fmad( mz, mz, fmad( my, my, mx*mx ) ), rcp_pres<R>( d ), e );
   const R p = floor_pres( (R)( eint*P.gm1_d ), P.min_pres );
   const R ir = rcp( (R)u[0] );
#  pragma unroll
   for (int v=0; v<NV; v++) q[v] = (R)u[v];
   q[5] = p;
   q[6] = ir;
   q[7] = sound_speed( P.gamma*p, q[0], ir );
}

// half-step cell update, floors and conversion to primitive (CPU_FluidSolver_MHM.cpp:846-933).  The update
// U - dt/(2dh) sum dF runs in the bulk type; the pressure recovery E - |m|^2/(2 rho) and the internal-energy
// floor run in FP64.
template <typename R>
__device__ __forceinline__ void half_cell( const R u[NV], const R dfxy[NV], const R hzl[NV], const R hzu[NV],
                                           const Prm<R> &P, R w[NV] )
{
   #pragma clang fp contract(off)
   R c[NV];
   const R k = (R)P.dt_dh2;
#  pragma unroll
   for (int v=0; v<NV; v++) c[v] = fmad( -k, dfxy[v] + ( hzu[v] - hzl[v] ), u[v] );
   c[0] = vmax( c[0], P.min_dens );
   const double d = (double)c[0], m1 = (double)c[1], m2 = (double)c[2], m3 = (double)c[3];
   const double q = -0.5*fmad( m3, m3, fmad( m2, m2, m1*m1 ) ), rd = rcp_pres<R>( d );
   double e = (double)c[4];
   double ein = fmad( q, rd, e );
   const double eout = ( ein == ein ) ? __builtin_fmax( ein, P.min_eint_d ) : ein;
   if ( ein != eout ) { e = e - ein + eout;  ein = fmad( q, rd, e ); }
   const R r = rcp( c[0] );
   w[0] = c[0];
   w[1] = c[1]*r;
   w[2] = c[2]*r;
   w[3] = c[3]*r;
   const double p = ein*P.gm1_d;
   w[4] = (R)( ( p == p ) ? __builtin_fmax( p, P.min_pres_d ) : p );
}

template <typename R>
__device__ __forceinline__ void ld_cell( const R (*a)[NC], int c, R q[8] )
{
#  pragma unroll
   for (int v=0; v<8; v++) q[v] = a[v][c];
}

template <int D, typename R>
__device__ __forceinline__ Side<R> side_at( const R (*a)[NC], int c ) { R q[8]; ld_cell( a, c, q ); return cell_side<D>( q ); }

template <int N, typename R>
__device__ __forceinline__ void ld5( const R (*a)[N], int c, R w[NV] )
{
#  pragma unroll
   for (int v=0; v<NV; v++) w[v] = a[v][c];
}
template <int N, typename R>
__device__ __forceinline__ void st5( R (*a)[N], int c, const R w[NV] )
{
#  pragma unroll
   for (int v=0; v<NV; v++) a[v][c] = w[v];
}

// LDS of one workgroup: 81,584 B (FP32, two workgroups per CU) or 163,160 B (FP64, one)
template <typename R>
struct SmemRP {
   R a[8][NC];                  // input plane (rho,mx,my,mz,E,P,1/rho,c_s)
   // x and y arrays of a field next to each other, so that a lane that does either adds one offset
   R h[NV][HX + HY];            // half-step fluxes of the low x (from HX: y) face of column (i,j) at i + NX (j-1)
   R l[NV][FX + FY];            // left states of the full-step x (from FX: y) faces: low face of column (i,j) at i-3 + FS (j-3)
   R g[NV][FX + FY];            // full-step fluxes of those faces
   R w[NV][HX];                 // half-step primitive plane read by the reconstruction, cell (i,j) at i + NX (j-1)
   R u3[3][NV][NK];             // lane-private ring: input cells of the own output column, planes t-3 .. t-1
   int fail, next;
   R cfl[8][4];                 // fused CFL: per-patch maxima of the 4 column waves (R is the I/O type)
};

// MODE 0: one patch group per workgroup; 1: persistent work queue; 2: the last patch groups in z slabs (slab_split())
template <typename R, typename IO, int RS, int LIM, int MODE>
__global__ void __launch_bounds__( NT ) __attribute__(( amdgpu_waves_per_eu( sizeof(R) == 4 ? 4 : 2 ) ))
mhm_rp_kernel( const IO *__restrict__ g_in, IO *__restrict__ g_out, IO *__restrict__ g_flux,
               int npg, int store_flux, int minmod_maxiter, R minmod_coeff, Prm<R> P0,
               IO *__restrict__ g_dt, double dh_safety0, Batch B )
{
   static_assert( sizeof( R ) == sizeof( IO ), "the input ring holds IO values in R storage" );
   __shared__ SmemRP<R> S;
   static_assert( sizeof( S ) <= ( sizeof( R ) == 4 ? 81920 : 163840 ), "two FP32 workgroups or one FP64 workgroup per CU" );

   const int tid  = threadIdx.x;
   const int wave = __builtin_amdgcn_readfirstlane( tid >> 6 );   // wave-uniform role switch
   const int g    = tid - NK;                                     // side lane (0..255 on waves 4-7)
   const int gw   = wave - 4;                                     // side wave: 0-1 arms, 2 single faces, 3 edges

   // the lane's output column: column lane tid, or the one whose x work side lane g does
   const int ki = 3 + ( tid & 15 ), kj = 3 + output_row( tid & ( NK - 1 ) );
   const int kc = ki + NX*kj, kh = kc - NX, kq = ( ki - 3 ) + FS*( kj - 3 );   // in S.a, in S.h and S.w, in S.l and S.g
   // lane-constant byte offsets of the global stores: output column in a 16^2 plane, and the coarse-fine flux
   // planes x = 0/8 (fx), y = 0/8 (fy) and x or y = 16 (edge lanes) at row kj, ki or the edge column
   const int  kxy    = ( ki - 3 ) + PS*( kj - 3 );
   const int  fx_off = ( ( ( ki - 3 )/8 )*NV*PS*PS + ( kj - 3 ) )*(int)sizeof( IO );
   const int  fy_off = ( ( 3 + ( kj - 3 )/8 )*NV*PS*PS + ( ki - 3 ) )*(int)sizeof( IO );

   int base = 0;
   for (int item = 0; ; item++)
   {
   // next patch group: blockIdx.x (of the last ones, a z slab: slab_split()), or the next PG of this workgroup's ticket of
   // the persistent work queue (a ticket covers B.claim consecutive PGs; the barrier before every PG also keeps the
   // previous PG's LDS reads ahead of the next PG's writes)
   int pg, slab_z = 0, slab_h = PS, half = -1;        // first output plane and output planes of the march; z half whose dt it writes
   if ( MODE == 1 )
   {
      const int sub = item % B.claim;
      __syncthreads();
      if ( sub == 0 )
      {
         if ( tid == 0 ) S.next = (int)atomicAdd( B.counter, 1u );
         __syncthreads();
         base = __builtin_amdgcn_readfirstlane( S.next )*B.claim;   // uniform: keep pointers and dt in SGPRs
      }
      pg = base + sub;
   }
   else
   {
      if ( item > 0 ) break;
      pg = blockIdx.x;
      if ( MODE == 2 && pg >= B.whole )
      {
         const int e = pg - B.whole, k = e % B.slabs;
         pg = B.whole + e / B.slabs;
         slab_h  = PS / B.slabs;
         slab_z = k*slab_h;
         half = ( B.slabs == 2 ) ? k : -1;
      }
   }
   if ( pg >= npg ) break;

   constexpr int SZ = sizeof( IO );
   const IO *in  = g_in  + (size_t)pg*NV*NC*NX;
   IO       *out = g_out + (size_t)pg*NV*PS*PS*PS;
   IO       *flx = store_flux ? g_flux + (size_t)pg*9*NV*PS*PS : nullptr;
   const int z0 = ( MODE == 2 ) ? slab_z : 0;
   // the march counts its planes from 0: the descriptors start at the slab's first plane (the x and y flux planes at its
   // first row)
   const __amdgpu_buffer_rsrc_t b_in  = make_buf( in + z0*NC,     ( NV*NC*NX - z0*NC )*SZ );
   const __amdgpu_buffer_rsrc_t b_out = make_buf( out + z0*PS*PS, ( NV*PS*PS*PS - z0*PS*PS )*SZ );
   const __amdgpu_buffer_rsrc_t b_flx = make_buf( flx ? flx + z0*PS : nullptr, flx ? ( 9*NV*PS*PS - z0*PS )*SZ : 0 );
   Prm<R> P = P0;
   double dh_safety = dh_safety0;
   if ( B.pg_dt_dh )
   {
      const double dt = B.pg_dt_dh[2*pg], dh = B.pg_dt_dh[2*pg + 1];
      P.dt_dh2 = 0.5*dt/dh;  P.dt_dh = dt/dh;  dh_safety = B.safety*dh;
   }

   for (int iter = 0; ; iter++)
   {
      Prm<R> Q = P;
      {
         R cf = ( minmod_maxiter == 0 ) ? minmod_coeff : minmod_coeff - (R)iter*minmod_coeff/(R)minmod_maxiter;
         Q.coeff = vmax( cf, (R)0 );
      }
      if ( tid == 0 ) S.fail = 0;
      IO cfl[2] = { (IO)0, (IO)0 };            // fused CFL: max(|v_d|+c_s) of this column in patches z=0,1
      __syncthreads();                         // the previous patch group / iteration is done with the LDS arrays

      auto march_columns = [&]()
      {
         const int z0 = ( MODE == 2 ) ? slab_z : 0, t1 = ( MODE == 2 ) ? slab_h + 5 : NX - 1;     // t1: last input plane
         R kU[8], kU1[8];                            // input cell of planes t and t-1 (+ pressure, 1/rho, c_s)
         R kHz[NV], kDh[NV];                         // half-step z-flux at t-3/2 ; half-step dFx+dFy of plane t-1
         R kW1[NV], kW2[NV], kW3[NV];                // half-step primitives of planes t-1, t-2, t-3
         R kFzR[NV], kFz[NV];                        // upper z face of plane r-1 ; full z-flux at r-3/2

         // two steps per iteration would rename the plane-to-plane register hand-offs instead of copying them, but spill
         // (FP64 HLLC on 1331 patch groups 564 us, rolled 511)
#        pragma unroll 1
         for (int t = 0; t <= t1; t++)
         {
            const int o = t - 3;                     // output plane of this step
            const int r = t - 2;                     // reconstructed plane of this step
            __syncthreads();                         // [A] input plane t and the full-step fluxes of plane t-3 visible

#           pragma unroll
            for (int v=0; v<8; v++) kU1[v] = kU[v];
            ld_cell( S.a, kc, kU );
#           pragma unroll
            for (int v=0; v<NV; v++) S.u3[( t + 2 ) % 3][v][tid] = kU1[v];     // plane t-1, read back at step t+2

            R df[NV];                                // full-step dFx+dFy of plane o
            if ( o >= 3 && o <= t1 - 3 )
#              pragma unroll
               for (int v=0; v<NV; v++) df[v] = ( S.g[v][kq + 1] - S.g[v][kq] ) + ( S.g[v][FX + kq + FS] - S.g[v][FX + kq] );

            // half-step z-flux at t-1/2 and half-step cell of plane t-1
            if ( t >= 1 )
            {
               R fz[NV], w[NV];
               solve<RS, 2, 0>( cell_side<2>( kU1 ), cell_side<2>( kU ), Q, fz );
               if ( t >= 2 )
               {
                  half_cell( kU1, kDh, kHz, fz, Q, w );
#                 pragma unroll
                  for (int v=0; v<NV; v++) { kW3[v] = kW2[v];  kW2[v] = kW1[v];  kW1[v] = w[v]; }
               }
#              pragma unroll
               for (int v=0; v<NV; v++) kHz[v] = fz[v];
            }
            // half-step y flux of plane t
            if ( t >= 1 && t <= t1 - 1 )
            {
               R f[NV];
               solve<RS, 1, 0>( side_at<1>( S.a, kc - NX ), cell_side<1>( kU ), Q, f );
               st5( S.h, HX + kh, f );
            }
            // PLM of plane r along z and y; the y neighbours come from the half-step plane r in S.w
            R zL[NV], zR[NV], yL[NV];
            if ( r >= 2 && r <= t1 - 2 )
            {
               plm_cell<LIM>( kW3, kW2, kW1, Q, zL, zR );
               if ( r >= 3 && r <= t1 - 3 )
               {
                  R a[NV], b[NV], fr[NV];
                  ld5( S.w, kh - NX, a );  ld5( S.w, kh + NX, b );
                  plm_cell<LIM>( a, kW2, b, Q, yL, fr );
                  st5( S.l, FX + kq + FS, fr );
               }
            }
            __syncthreads();                         // [H] half-step fluxes and left states of plane r visible


            if ( t >= 1 && t <= t1 - 1 )
#              pragma unroll
               for (int v=0; v<NV; v++) kDh[v] = ( S.h[v][kh + 1] - S.h[v][kh] ) + ( S.h[v][HX + kh + NX] - S.h[v][HX + kh] );
            if ( t >= 2 ) st5( S.w, kh, kW1 );  // plane t-1 replaces plane t-2 for the next reconstruction

            // full-step z-flux at r-1/2
            R fz[NV];
            if ( r >= 3 && r <= t1 - 2 )
            {
               solve<RS, 2, 1>( face_side<2>( kFzR, Q ), face_side<2>( zL, Q ), Q, fz );
               if ( flx && ( z0 + r - 3 ) % 8 == 0 && ( r < t1 - 2 || z0 + r == 19 ) )    // the next slab stores the face between
#                 pragma unroll
                  for (int v=0; v<NV; v++)
                     buf_store( (IO)fz[v], b_flx, kxy*SZ, ( ( ( 6 + ( z0 + r - 3 )/8 )*NV + v )*PS*PS - z0*PS )*SZ );
            }
            if ( r >= 2 )
#              pragma unroll
               for (int v=0; v<NV; v++) kFzR[v] = zR[v];
            // full-step y-flux of plane r
            if ( r >= 3 && r <= t1 - 3 )
            {
               R f[NV], q[NV];
               ld5( S.l, FX + kq, q );
               solve<RS, 1, 1>( face_side<1>( q, Q ), face_side<1>( yL, Q ), Q, f );
               st5( S.g, FX + kq, f );
               if ( flx && ( kj - 3 ) % 8 == 0 )
#                 pragma unroll
                  for (int v=0; v<NV; v++) buf_store( (IO)f[v], b_flx, fy_off, ( v*PS*PS + PS*( r - 3 ) )*SZ );
            }
            // full-step update and output of plane o
            if ( o >= 3 && o <= t1 - 3 )
            {
               IO res[NV], uo[NV];
               ld5( S.u3[t % 3], tid, uo );
               const bool bad = full_cell( uo, df, kFz, fz, Q, res );
#              pragma unroll
               for (int v=0; v<NV; v++) buf_store( res[v], b_out, kxy*SZ, ( v*PS*PS*PS + PS*PS*( o - 3 ) )*SZ );
               if ( bad ) S.fail = 1;
               if ( g_dt ) cfl[ ( z0 + o - 3 )/8 ] = vmax( cfl[ ( z0 + o - 3 )/8 ], cell_cfl( res, (double)Q.gamma, Q.gm1_d, Q.min_pres_d ) );
            }
            if ( r >= 3 && r <= t1 - 2 )
#              pragma unroll
               for (int v=0; v<NV; v++) kFz[v] = fz[v];
         }
      };
      auto march_sides = [&]()
      {
         const int t1 = ( MODE == 2 ) ? slab_h + 5 : NX - 1;     // t1: last input plane
         int oi, oj, ei, ej;
         bool e_dy, e_face;
         arm_column( g, oi, oj );
         const int  oc = oi + NX*oj, oh = oc - NX;
         const bool has_e = edge_column( g, ei, ej, e_dy, e_face );
         const int  eh = ei + NX*( ej - 1 );             // in S.w
         const int  e_st = e_dy ? NX : 1;                // neighbour stride of the edge column's direction
         // the edge column's face in S.l / S.g: the low face of a column 19, the high face of a column 2
         const int  eq = e_dy ? FX + ( ei - 3 ) + FS*( e_face ? 16 : 0 ) : ( e_face ? 16 : 0 ) + FS*( ej - 3 );
         const int  fe_off = ( ( e_dy ? 5 : 2 )*NV*PS*PS + ( ( e_dy ? ei : ej ) - 3 ) )*(int)sizeof( IO );
         // single half-step face of the lane at the planes with arm cells (tm) and at the others (tn), -1 = none
         int tm_c = -1, tn_c = -1;
         bool t_dy = false, t_d2;
         if ( !face_task( g, true, tm_c, t_dy ) ) tm_c = -1;
         if ( !face_task( g, false, tn_c, t_d2 ) ) tn_c = -1;
         // column of side waves 0-1 whose half-step x face this lane of side waves 2-3 does
         const int k2 = ki + NX*( 3 + output_row( ( g & 63 ) + ( gw & 1 )*64 ) );
         R oU[8], oU1[8], oHz[NV], oDh[NV], oW[NV];      // arm column: input cell of planes t, t-1, and as the output column

         // prefetch of the next input plane, two cells per lane (coalesced)
         IO pf[2][NV];
         auto issue = [&]( int t )
         {
#           pragma unroll
            for (int k=0; k<2; k++)
            {
               const int c = g + k*NK;
               if ( c < NC )
#                 pragma unroll
                  for (int v=0; v<NV; v++) buf_load( b_in, c*SZ, ( v*NC*NX + t*NC )*SZ, pf[k][v] );
            }
         };
         // input plane (prefetched) -> LDS, with pressure, 1/rho and c_s once per cell
         auto stage = [&]()
         {
#           pragma unroll
            for (int k=0; k<2; k++)
            {
               const int c = g + k*NK;
               if ( c < NC )
               {
                  R q[8];
                  derive_cell( pf[k], q, Q );
#                 pragma unroll
                  for (int v=0; v<8; v++) S.a[v][c] = q[v];
               }
            }
         };
         issue( 0 );
         stage();
         issue( 1 );

#        pragma unroll 1
         for (int t = 0; t <= t1; t++)
         {
            const int r = t - 2;
            __syncthreads();                         // [A]
            // arm half step: cells of planes 3 .. t1-3 (updated one step later), their z faces and low x/y faces
            const bool arm_ld = ( gw < 2 ) && t >= 2 && t <= t1 - 2;
            const bool arm_z  = ( gw < 2 ) && t >= 3 && t <= t1 - 2;
            const bool arm_xy = ( gw < 2 ) && t >= 3 && t <= t1 - 3;
#           pragma unroll
            for (int v=0; v<8; v++) oU1[v] = oU[v];
            if ( arm_ld ) ld_cell( S.a, oc, oU );
            if ( arm_z )
            {
               R fz[NV];
               solve<RS, 2, 0>( cell_side<2>( oU1 ), cell_side<2>( oU ), Q, fz );
               if ( t >= 4 ) half_cell( oU1, oDh, oHz, fz, Q, oW );
#              pragma unroll
               for (int v=0; v<NV; v++) oHz[v] = fz[v];
            }
            if ( arm_xy )
            {
               const Side<R> l[2] = { side_at<0>( S.a, oc - 1 ), side_at<1>( S.a, oc - NX ) }, q[2] = { cell_side<0>( oU ), cell_side<1>( oU ) };
               R f[2][NV], ox[NV], oy[NV];
               solve_n<RS, 0, 2>( l, q, Q, f );
               to_lab<0>( f[0], ox );  to_lab<1>( f[1], oy );
               st5( S.h, oh, ox );
               st5( S.h, HX + oh, oy );
            }
            if ( gw == 2 && t >= 1 && t <= t1 - 1 )
            {
               const bool fdy = t_dy;
               const int  fc = ( t >= 3 && t <= t1 - 3 ) ? tm_c : tn_c;
               if ( fc >= 0 )
               {
                  R ql[8], qr[8], f[NV];
                  ld_cell( S.a, fc - ( fdy ? NX : 1 ), ql );
                  ld_cell( S.a, fc, qr );
                  solve_xy<RS, 0>( cell_side_xy( ql, fdy ), cell_side_xy( qr, fdy ), Q, fdy, f );
                  st5( S.h, ( fdy ? HX - NX : -NX ) + fc, f );
               }
            }
            // half-step x fluxes of plane t
            if ( gw >= 2 && t >= 1 && t <= t1 - 1 )
            {
               const Side<R> l[2] = { side_at<0>( S.a, kc - 1 ), side_at<0>( S.a, k2 - 1 ) }, q[2] = { side_at<0>( S.a, kc ), side_at<0>( S.a, k2 ) };
               R f[2][NV], fx[NV], f2[NV];
               solve_n<RS, 0, 2>( l, q, Q, f );
               to_lab<0>( f[0], fx );  to_lab<0>( f[1], f2 );
               st5( S.h, kh, fx );
               st5( S.h, k2 - NX, f2 );
            }
            // PLM of plane r along x, and of the edge column
            R xL[NV], eL[NV];
            if ( r >= 3 && r <= t1 - 3 )
            {
               R a[NV], b[NV], c[NV], fr[NV];
               ld5( S.w, kh - 1, a );  ld5( S.w, kh, b );  ld5( S.w, kh + 1, c );
               plm_cell<LIM>( a, b, c, Q, xL, fr );
               st5( S.l, kq + 1, fr );
               if ( has_e )
               {
                  ld5( S.w, eh - e_st, a );  ld5( S.w, eh, b );  ld5( S.w, eh + e_st, c );
                  plm_cell<LIM>( a, b, c, Q, eL, fr );
                  if ( !e_face ) st5( S.l, eq, fr );
               }
            }
            __syncthreads();                         // [H]


            // input plane t+1 into LDS: every read of S.a of this step came before barrier [H].  First, as the wait for its
            // loads would also wait for the flux stores below
            if ( t + 1 <= t1 )
            {
               stage();
               if ( t + 2 <= t1 ) issue( t + 2 );
            }
            if ( arm_xy )
#              pragma unroll
               for (int v=0; v<NV; v++) oDh[v] = ( S.h[v][oh + 1] - S.h[v][oh] ) + ( S.h[v][HX + oh + NX] - S.h[v][HX + oh] );
            if ( arm_z && t >= 4 ) st5( S.w, oh, oW );

            // full-step x-flux of plane r, and the faces x = 16 and y = 16 of the block
            if ( r >= 3 && r <= t1 - 3 )
            {
               R f[NV], q[NV];
               ld5( S.l, kq, q );
               solve<RS, 0, 1>( face_side<0>( q, Q ), face_side<0>( xL, Q ), Q, f );
               st5( S.g, kq, f );
               if ( flx && ( ki - 3 ) % 8 == 0 )
#                 pragma unroll
                  for (int v=0; v<NV; v++) buf_store( (IO)f[v], b_flx, fx_off, ( v*PS*PS + PS*( r - 3 ) )*SZ );
               if ( has_e && e_face )
               {
                  ld5( S.l, eq, q );
                  solve_xy<RS, 1>( face_side_xy( q, e_dy, Q ), face_side_xy( eL, e_dy, Q ), Q, e_dy, f );
                  st5( S.g, eq, f );
                  if ( flx )                         // planes x = 16 (2) and y = 16 (5)
#                    pragma unroll
                     for (int v=0; v<NV; v++) buf_store( (IO)f[v], b_flx, fe_off, ( v*PS*PS + PS*( r - 3 ) )*SZ );
               }
            }
         }
      };
      if ( wave < 4 ) march_columns(); else march_sides();

      if ( g_dt ) fused_dt( cfl, ( ki - 3 )/8 + 2*( ( kj - 3 )/8 ), S.cfl, g_dt + (size_t)pg*8, dh_safety, half );
      __syncthreads();
      const bool redo = ( S.fail != 0 ) && ( iter + 1 <= minmod_maxiter );
      __syncthreads();
      if ( !redo ) break;
   } // MinMod retry
   } // work items
}

} // namespace

template <typename R, typename IO, int RS>
static void launch_rs( const IO *in, IO *out, IO *flux, int npg, int store_flux, int minmod_maxiter,
                       double minmod_coeff, const Prm<R> &P, IO *dt, double dh_safety, Batch B, int grid_blocks, hipStream_t stream )
{
   const bool pers = ( B.counter != nullptr );
   if ( !pers ) slab_split( npg, NX - PS, sizeof( R ) == 4 ? 2 : 1, minmod_maxiter, dt != nullptr, B );
   const dim3 grid( pers ? ( grid_blocks > 0 ? grid_blocks : npg ) : B.whole + ( npg - B.whole )*B.slabs ), block( NT );
   const int mode = pers ? 1 : ( B.slabs > 1 ) ? 2 : 0;
#  define GA_LAUNCH( LIM_, MODE_ ) hipLaunchKernelGGL( ( mhm_rp_kernel<R, IO, RS, LIM_, MODE_> ), grid, block, 0, stream, \
                                                      in, out, flux, npg, store_flux, minmod_maxiter, (R)minmod_coeff, P, dt, dh_safety, B )
#  define GA_MODE( LIM_ ) { if ( mode == 0 ) GA_LAUNCH( LIM_, 0 ); else if ( mode == 1 ) GA_LAUNCH( LIM_, 1 ); else GA_LAUNCH( LIM_, 2 ); }
   if ( kernel_limiter( P.limiter, minmod_coeff ) == 4 ) GA_MODE( 4 ) else GA_MODE( 0 )
#  undef GA_MODE
#  undef GA_LAUNCH
}

template <typename R, typename IO>
int launch_mhm_rp( const IO *in, IO *out, IO *flux, int npg, int rsolver, int store_flux, int minmod_maxiter,
                   double minmod_coeff, const Prm<R> &P, IO *dt, double dh_safety, const Batch &B, int grid_blocks, hipStream_t stream )
{
   if ( npg <= 0 ) return 0;
   switch ( rsolver )
   {
      case 4: launch_rs<R, IO, 4>( in, out, flux, npg, store_flux, minmod_maxiter, minmod_coeff, P, dt, dh_safety, B, grid_blocks, stream ); break;
      case 3: launch_rs<R, IO, 3>( in, out, flux, npg, store_flux, minmod_maxiter, minmod_coeff, P, dt, dh_safety, B, grid_blocks, stream ); break;
      case 2: launch_rs<R, IO, 2>( in, out, flux, npg, store_flux, minmod_maxiter, minmod_coeff, P, dt, dh_safety, B, grid_blocks, stream ); break;
      default: return -1;
   }
   return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
}

template int launch_mhm_rp<double, double>( const double*, double*, double*, int, int, int, int, double, const Prm<double>&, double*, double, const Batch&, int, hipStream_t );
template int launch_mhm_rp<float,  float >( const float*,  float*,  float*,  int, int, int, int, double, const Prm<float>&,  float*, double, const Batch&, int, hipStream_t );

} // namespace gamer_amd

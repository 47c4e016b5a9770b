// Coarse -> fine interpolation of ghost-zone data, and the same-level gather of patch-group inputs from per-patch
// data: the two halves of Prepare_PatchData for the fluid solver at a refinement boundary
// (src/Main/Prepare_PatchData.cpp:166, src/Main/InterpolateGhostZone.cpp, src/Interpolation/Interpolate.cpp:90).
//
//   interpolate_kernel   Interpolate() with Interpolate_Iterate (Interpolate.cpp:90-330) for INT_MINMOD3D, INT_MINMOD1D,
//                        INT_VANLEER, INT_CQUAD, INT_QUAD, INT_CQUAR and INT_QUAR (src/Interpolation/Int_*.cpp): one
//                        workgroup per coarse box, one lane per asked-for coarse cell (listed, or a column of a box
//                        marched along z: interp_launch) producing its 2x2x2 fine cells.  For the
//                        tensor-product schemes (all but INT_MINMOD1D) the lane evaluates the x pass on the
//                        (2G+1)x(2G+1) coarse (y,z) neighbourhood (G = 1, or 2 for the quartic schemes), then the y
//                        pass, then the z pass: the same operations in the same order as the reference's split
//                        temporaries.  Iterations (conserved
//                        variables, then primitive variables, then lower monotonic coefficients) redo only coarse
//                        cells whose fine cells failed the physicality test: the INTERP_MASK rule (include/Macro.h:947)
//                        at the granularity of 2x2x2 fine blocks.
//   prepare_patches_kernel, prepare_patches_vec_kernel  the same-level copies: window cell (x,y,z) of a patch group from
//                        the patch in its 4x4x4 slot table; a cell without a patch (-1) comes from the interpolated fine
//                        box, or keeps its value if there is none.  The second takes four cells a lane (FP32)
//   gather_boxes_kernel  the coarse data of InterpolateGhostZone (src/Main/InterpolateGhostZone.cpp): box cell (x,y,z)
//                        from the patch covering cell origin + (x,y,z) of the box's slot table (e.g. the father patch
//                        and its 26 siblings); gather_planes_kernel does the same plane by plane

#include <type_traits>
#include "hydro_math.hpp"
#include "hydro_kernels.hpp"

namespace gamer_amd {

namespace {

constexpr int PS = 16, H = 8, P3 = H*H*H;

template <typename T> __device__ __forceinline__ T sgn( T a ) { return ( a < (T)0 ) ? (T)-1 : (T)+1; }

template <typename T>
__device__ __forceinline__ T cquad_slope( T L, T C, T R, bool mono, T coeff, bool opp0, bool turn )
{
   #pragma clang fp contract(off)
   T s = (T)0.125*( R - L );
   if ( mono )
   {
      const T l = (T)0.25*( C - L ), r = (T)0.25*( R - C );
      // of one sign where it matters, so that R - L has it too: the smallest magnitude, the smaller side scaled.  A negative
      // coefficient (turn) turns the slope around
      const T m = vmin( vmin( vmin( vabs( l ), vabs( r ) )*coeff, vmax( vabs( l ), vabs( r ) ) ), vabs( s ) );
      s = ( l*r > (T)0 ) ? __builtin_copysign( m, l ) : (T)0;
      if ( turn ) s = -s;
   }
   if ( opp0 && L*R < (T)0 ) s = (T)0;
   return s;
}

// One split pass of a tensor-product scheme: stencil u = {L2, L1, C, R1, R2} along one direction -> the fine values
// (lo, hi) of the centre cell (x passes of Int_MinMod3D.cpp:93-103, Int_vanLeer.cpp:93-105, Int_CQuadratic.cpp,
// Int_Quadratic.cpp:104-160, Int_CQuartic.cpp:100-140, Int_Quartic.cpp:100-165; their y and z passes repeat them)
template <typename T, int SCHEME>
__device__ __forceinline__ void pass1d( const T u[5], bool mono, T coeff, bool opp0, bool turn, T &lo, T &hi )
{
   #pragma clang fp contract(off)
   const T L2 = u[0], L1 = u[1], C = u[2], R1 = u[3], R2 = u[4];
   T s;
   if ( SCHEME == 1 || SCHEME == 3 )               // MinMod-3D, van Leer
   {
      const T l = C - L1, r = R1 - C;
      if ( r*l <= (T)0 ) s = (T)0;
      else s = ( SCHEME == 1 ) ? (T)0.25*( vabs( r ) < vabs( l ) ? r : l ) : (T)0.5*l*r/( l + r );
      if ( opp0 && L1*R1 < (T)0 ) s = (T)0;
      lo = C - s;  hi = C + s;
   }
   else if ( SCHEME == 4 )                         // conservative quadratic
   {
      s = cquad_slope( L1, C, R1, mono, coeff, opp0, turn );
      lo = C - s;  hi = C + s;
   }
   else if ( SCHEME == 6 )                         // conservative quartic
   {
      s = (T)( 3.0/128.0)*L2 + (T)(-22.0/128.0)*L1 + (T)(22.0/128.0)*R1 + (T)(-3.0/128.0)*R2;
      if ( mono )
      {
         T l = (T)0.25*( C - L1 ), r = (T)0.25*( R1 - C );
         if ( l*r > (T)0 )
         {
            if ( s*l < (T)0 ) s = (T)0.125*( R1 - L1 );
            const T sg = sgn( l );
            s *= sg;  l *= sg;  r *= sg;
            if ( l < r ) l *= coeff; else r *= coeff;
            s = vmin( l, s );
            s = vmin( r, s );
            s *= sg;
         }
         else s = (T)0;
      }
      if ( opp0 && L1*R1 < (T)0 ) s = (T)0;
      lo = C - s;  hi = C + s;
   }
   else                                            // quadratic (5), quartic (7): Lagrange values at -/+ 1/4
   {
      if ( SCHEME == 5 )
      {
         lo = (T)( 5.0/32.0)*L1 + (T)(30.0/32.0)*C + (T)(-3.0/32.0)*R1;
         hi = (T)(-3.0/32.0)*L1 + (T)(30.0/32.0)*C + (T)( 5.0/32.0)*R1;
      }
      else
      {
         lo = (T)( -45.0/2048.0)*L2 + (T)( 420.0/2048.0)*L1 + (T)(1890.0/2048.0)*C + (T)(-252.0/2048.0)*R1
            + (T)(  35.0/2048.0)*R2;
         hi = (T)(  35.0/2048.0)*L2 + (T)(-252.0/2048.0)*L1 + (T)(1890.0/2048.0)*C + (T)( 420.0/2048.0)*R1
            + (T)( -45.0/2048.0)*R2;
      }
      if ( mono )
      {
         T l = C - L1, r = R1 - C;
         if ( l*r > (T)0 )
         {
            const T cmax = ( l > (T)0 ) ? R1 : L1, cmin = ( l > (T)0 ) ? L1 : R1;
            bool bad = ( vmax( lo, hi ) > cmax || vmin( lo, hi ) < cmin );
            if ( SCHEME == 7 ) bad = bad || ( hi - lo )*l < (T)0;
            if ( bad )
            {
               const T c4 = (T)0.25*coeff;
               s  = (T)0.125*( R1 - L1 );
               l *= c4;  r *= c4;
               const T sg = sgn( l );
               s *= sg;
               s  = vmin( sg*l, s );
               s  = vmin( sg*r, s );
               s *= sg;
               lo = C - s;  hi = C + s;
            }
         }
         else { lo = C;  hi = C; }
      }
      if ( opp0 && L1*R1 < (T)0 ) { lo = C;  hi = C; }
   }
}

// the 2x2x2 fine values of coarse cell i of one field: f[(k*2 + j)*2 + i]
template <typename T, int SCHEME>
__device__ __forceinline__ void interp_cell( const T *__restrict__ c, int i, int dy, int dz, bool mono, T coeff,
                                             bool opp0, bool turn, T f[8] )
{
   #pragma clang fp contract(off)
   if ( SCHEME != 2 )
   {
      constexpr int G = ( SCHEME == 6 || SCHEME == 7 ) ? 2 : 1, W = 2*G + 1;
      T X[W][W][2], Y[W][2][2], u[5];
#     pragma unroll
      for (int a=0; a<W; a++)
#        pragma unroll
         for (int b=0; b<W; b++)
         {
            const int q = i + ( a - G )*dz + ( b - G )*dy;
#           pragma unroll
            for (int k=0; k<5; k++) u[k] = ( k - 2 >= -G && k - 2 <= G ) ? c[q + k - 2] : (T)0;
            pass1d<T, SCHEME>( u, mono, coeff, opp0, turn, X[a][b][0], X[a][b][1] );
         }
#     pragma unroll
      for (int a=0; a<W; a++)
#        pragma unroll
         for (int x=0; x<2; x++)
         {
#           pragma unroll
            for (int k=0; k<5; k++) u[k] = ( k - 2 >= -G && k - 2 <= G ) ? X[a][k - 2 + G][x] : (T)0;
            pass1d<T, SCHEME>( u, mono, coeff, opp0, turn, Y[a][0][x], Y[a][1][x] );
         }
#     pragma unroll
      for (int y=0; y<2; y++)
#        pragma unroll
         for (int x=0; x<2; x++)
         {
#           pragma unroll
            for (int k=0; k<5; k++) u[k] = ( k - 2 >= -G && k - 2 <= G ) ? Y[k - 2 + G][y][x] : (T)0;
            pass1d<T, SCHEME>( u, mono, coeff, opp0, turn, f[( 0*2 + y )*2 + x], f[( 1*2 + y )*2 + x] );
         }
   }
   else
   {
      const int cd[3] = { 1, dy, dz };
      T sl[3];
#     pragma unroll
      for (int d=0; d<3; d++)
      {
         const T l = c[i] - c[i - cd[d]], r = c[i + cd[d]] - c[i];
         sl[d] = ( r*l <= (T)0 ) ? (T)0 : (T)0.25*( vabs( r ) < vabs( l ) ? r : l );
         if ( opp0 && c[i - cd[d]]*c[i + cd[d]] < (T)0 ) sl[d] = (T)0;
      }
#     pragma unroll
      for (int k=0; k<2; k++)
#        pragma unroll
         for (int j=0; j<2; j++)
#           pragma unroll
            for (int x=0; x<2; x++)
               f[( k*2 + j )*2 + x] = c[i] + ( k ? sl[2] : -sl[2] ) + ( j ? sl[1] : -sl[1] ) + ( x ? sl[0] : -sl[0] );
   }
}

// x pass of the rows y-1, y, y+1 of coarse plane z' around index q, then the y pass: Y[y-lo/hi][x-lo/hi] of that
// plane, exactly as interp_cell computes its Y[a] (3-point schemes)
template <typename T, int SCHEME>
__device__ __forceinline__ void xy_pass( const T *__restrict__ c, int q, int dy, bool mono, T coeff, bool opp0, T Y[2][2] )
{
   #pragma clang fp contract(off)
   T X[3][2], u[5];
#  pragma unroll
   for (int b=0; b<3; b++)
   {
      const int qq = q + ( b - 1 )*dy;
      u[0] = (T)0;  u[1] = c[qq - 1];  u[2] = c[qq];  u[3] = c[qq + 1];  u[4] = (T)0;
      pass1d<T, SCHEME>( u, mono, coeff, opp0, false, X[b][0], X[b][1] );
   }
#  pragma unroll
   for (int x=0; x<2; x++)
   {
      u[0] = (T)0;  u[1] = X[0][x];  u[2] = X[1][x];  u[3] = X[2][x];  u[4] = (T)0;
      pass1d<T, SCHEME>( u, mono, coeff, opp0, false, Y[0][x], Y[1][x] );
   }
}

template <typename T> struct Huge;
template <> struct Huge<double> { static constexpr double v = 1.7976931348623157e308; static constexpr double eps = 2.2204460492503131e-16; };
template <> struct Huge<float>  { static constexpr float  v = 3.40282346638528859812e+38f; static constexpr float eps = 1.1920928955078125e-07f; };

// Hydro_IsUnphysical in CONS mode (FluUtility.cpp:843-940)
template <typename T>
__device__ __forceinline__ bool cons_bad( const T u[NV] )
{
   #pragma clang fp contract(off)
   const T huge = Huge<T>::v;
   bool bad = false;
#  pragma unroll
   for (int v=0; v<NV; v++)
   {
      bad |= ( u[v] != u[v] );
      if ( v >= 1 && v <= 3 ) bad |= ( u[v] < -huge || u[v] > huge );
      else                    bad |= ( u[v] <= (T)0 || u[v] > huge );
   }
   const T e = u[4] - (T)0.5*( u[1]*u[1] + u[2]*u[2] + u[3]*u[3] )/u[0];
   bad |= ( e < (T)-3.0*u[4]*Huge<T>::eps || e > huge || e != e );
   return bad;
}

// Hydro_IsUnphysical in PRIM mode plus the interpolated internal energy from the EoS (Interpolate.cpp:234-262)
template <typename T>
__device__ __forceinline__ bool prim_bad( const T w[NV], double inv_gm1 )
{
   const T huge = Huge<T>::v;
   bool bad = false;
#  pragma unroll
   for (int v=0; v<NV; v++)
   {
      bad |= ( w[v] != w[v] );
      if ( v >= 1 && v <= 3 ) bad |= ( w[v] < -huge || w[v] > huge );
      else                    bad |= ( w[v] <= (T)0 || w[v] > huge );
   }
   const T e = w[4]*(T)inv_gm1;                      // P/(gamma-1) in the storage type, as EOS_GAMMA
   return bad || e < (T)0 || e > huge || e != e;
}

// the 2x2x2 fine values of one coarse cell: physicality test (when iterating), conversion back from primitive
// variables, store; false when the test failed (nothing stored)
template <typename T>
__device__ __forceinline__ bool store_fine( T f[NV][8], bool iterate, bool prim, const InterpPrm &p, T *F, int F3, int fo,
                                           int fdy, int fdz )
{
   #pragma clang fp contract(off)
   bool bad = false;
   if ( iterate )
#     pragma unroll
      for (int b=0; b<8; b++)
      {
         T t[NV];
#        pragma unroll
         for (int v=0; v<NV; v++) t[v] = f[v][b];
         bad |= prim ? prim_bad( t, p.inv_gm1 ) : cons_bad( t );
      }
   if ( bad ) return false;
#  pragma unroll
   for (int b=0; b<8; b++)
   {
      T t[NV];
#     pragma unroll
      for (int v=0; v<NV; v++) t[v] = f[v][b];
      if ( prim )
      {
         // Hydro_Pri2Con with EoS_DensPres2Eint
         const T ei = t[4]*(T)p.inv_gm1;
         t[1] = t[0]*t[1];  t[2] = t[0]*t[2];  t[3] = t[0]*t[3];
         t[4] = (T)0.5*( t[1]*t[1] + t[2]*t[2] + t[3]*t[3] )/t[0] + ei;
      }
      const int o = fo + ( b >> 2 )*fdz + ( ( b >> 1 ) & 1 )*fdy + ( b & 1 );
#     pragma unroll
      for (int v=0; v<NV; v++) F[ (size_t)v*F3 + o ] = t[v];
   }
   return true;
}

// One lane per asked-for coarse cell, from a list: a box next to a patch of its own level needs two layers of its 12^3 cells,
// and a lane's chain of 95 one-dimensional passes (19 a field) is the time, so the lanes must all have cells.  PLAIN: all
// fields monotonic, their coefficient not negative, and no clipping across 0 (the default); with these as run-time bits every pass had branches of its own,
// which kept the passes from overlapping.  512 boxes of the AMR step (216 ask for nothing, most others for 288 cells), CQUAD:
// FP32 118 -> 34 us, FP64 155 -> 48; every cell asked for 130 -> 65 and 217 -> 150; one box 95 -> 26.  The first form marched
// a lane per column through the box: 9 passes a cell and field in place of 19, but 24 lanes of 144 at work beside an x face,
// twelve planes in sequence; the list with the branches took 90.
// MARCH: no list, and the first pass (not of MINMOD1D) with a lane per column, marching along z with the y-pass results of planes z-1, z, z+1 in registers:
// 9 passes a cell and field in place of 19, with interp_cell's operations in its order, so the same bits.  interp_launch()
// says where that is the faster one, and how many lanes (NT) a block has and waves per SIMD (EU) its registers leave room
// for (0: as the compiler finds).
template <typename T, int SCHEME, bool PLAIN, bool MARCH, int NT, int EU>
__global__ void __launch_bounds__( NT ) __attribute__(( amdgpu_waves_per_eu( EU ) ))
interpolate_kernel( T *__restrict__ g_c, T *__restrict__ g_f, int nbox, InterpPrm p, int *__restrict__ nfail )
{
   #pragma clang fp contract(off)
   __shared__ int s_fail;
   __shared__ int s_n;
   __shared__ unsigned char s_done[INTERP_MAX_CELLS];
   __shared__ unsigned short s_todo[MARCH ? 1 : INTERP_MAX_CELLS];
   const int q = blockIdx.x, tid = threadIdx.x;
   if ( q >= nbox ) return;
   const int dy = p.cs[0], dz = p.cs[0]*p.cs[1], C3 = dz*p.cs[2];
   const int fdy = p.fs[0], fdz = p.fs[0]*p.fs[1], F3 = fdz*p.fs[2];
   const int ncell = p.cr[0]*p.cr[1]*p.cr[2];
   T *C = g_c + (size_t)q*NV*C3;
   T *F = g_f + (size_t)q*NV*F3;
   const bool iterate = p.int_prim || p.reduce;
   const int mono_max = p.reduce ? p.mono_max_iter : 0, max_iter = p.int_prim ? mono_max + 1 : mono_max;

   // the cells that are asked for, listed (in any order: they are independent)
   int ntodo = ncell;
   if constexpr ( MARCH )
   {
      for (int c = tid; c < ncell; c += NT) s_done[c] = p.need ? !p.need[ (size_t)q*ncell + c ] : 0;
      __syncthreads();
   }
   else
   {
      if ( tid == 0 ) s_n = 0;
      __syncthreads();
      for (int c = tid; c < ncell; c += NT)
      {
         const bool todo = !p.need || p.need[ (size_t)q*ncell + c ];
         s_done[c] = !todo;
         const unsigned long long m = __ballot( todo );
         const int lane = tid & 63, first = __ffsll( (long long)__ballot( true ) ) - 1;
         int at = 0;
         if ( lane == first ) at = atomicAdd( &s_n, __popcll( m ) );
         at = __shfl( at, first, 64 );
         if ( todo ) s_todo[ at + __popcll( m & ( ( 1ULL << lane ) - 1 ) ) ] = (unsigned short)c;
      }
      __syncthreads();
      ntodo = s_n;
      if ( ntodo == 0 ) return;
   }
   T coeff = (T)p.mono_coeff;
   bool prim = false;
   for (int it = 0; ; it++)
   {
      if ( it == 1 && p.int_prim )
      {
         // Hydro_Con2Pri of the whole coarse box, in place (Interpolate.cpp:148-170)
         for (int i = tid; i < C3; i += NT)
         {
            T u[NV];
#           pragma unroll
            for (int v=0; v<NV; v++) u[v] = C[ (size_t)v*C3 + i ];
            const T r = (T)1/u[0];
            const T e = u[4] - (T)0.5*( u[1]*u[1] + u[2]*u[2] + u[3]*u[3] )/u[0];
            T pr = (T)( (double)e*p.gm1 );
            pr = ( pr == pr ) ? vmax( pr, (T)p.min_pres ) : pr;
            C[ (size_t)1*C3 + i ] = u[1]*r;
            C[ (size_t)2*C3 + i ] = u[2]*r;
            C[ (size_t)3*C3 + i ] = u[3]*r;
            C[ (size_t)4*C3 + i ] = pr;
         }
         prim = true;
         __syncthreads();
      }
      else if ( it > 0 )
      {
         coeff -= (T)p.mono_coeff/(T)mono_max;
         coeff  = vmax( coeff, (T)0 );
      }
      if ( tid == 0 ) s_fail = 0;
      __syncthreads();

      if ( MARCH && SCHEME != 2 && it == 0 )
      {
         const int ncol = p.cr[0]*p.cr[1];
         for (int col = tid; col < ncol; col += NT)
         {
            const int x = col % p.cr[0], y = col / p.cr[0];
            const int q0 = p.c0[2]*dz + ( p.c0[1] + y )*dy + p.c0[0] + x;      // coarse index of (x, y, z = 0)
            T Yw[NV][3][2][2];
#           pragma unroll
            for (int v=0; v<NV; v++)
            {
               xy_pass<T, SCHEME>( C + (size_t)v*C3, q0 - dz, dy, ( p.mono >> v ) & 1, coeff, p.opp0, Yw[v][0] );
               xy_pass<T, SCHEME>( C + (size_t)v*C3, q0,      dy, ( p.mono >> v ) & 1, coeff, p.opp0, Yw[v][1] );
            }
            for (int z = 0; z < p.cr[2]; z++)
            {
               T f[NV][8], u[5];
#              pragma unroll
               for (int v=0; v<NV; v++)
               {
                  xy_pass<T, SCHEME>( C + (size_t)v*C3, q0 + ( z + 1 )*dz, dy, ( p.mono >> v ) & 1, coeff, p.opp0, Yw[v][2] );
#                 pragma unroll
                  for (int yy=0; yy<2; yy++)
#                    pragma unroll
                     for (int xx=0; xx<2; xx++)
                     {
                        u[0] = (T)0;  u[1] = Yw[v][0][yy][xx];  u[2] = Yw[v][1][yy][xx];  u[3] = Yw[v][2][yy][xx];  u[4] = (T)0;
                        pass1d<T, SCHEME>( u, ( p.mono >> v ) & 1, coeff, p.opp0, false, f[v][( 0*2 + yy )*2 + xx],
                                           f[v][( 1*2 + yy )*2 + xx] );
                     }
               }
               const int fo = ( p.f0[2] + 2*z )*fdz + ( p.f0[1] + 2*y )*fdy + p.f0[0] + 2*x;
               if ( store_fine( f, iterate, prim, p, F, F3, fo, fdy, fdz ) ) s_done[ col + z*ncol ] = 1; else s_fail = 1;
#              pragma unroll
               for (int v=0; v<NV; v++)
#                 pragma unroll
                  for (int yy=0; yy<2; yy++)
#                    pragma unroll
                     for (int xx=0; xx<2; xx++) { Yw[v][0][yy][xx] = Yw[v][1][yy][xx];  Yw[v][1][yy][xx] = Yw[v][2][yy][xx]; }
            }
         }
      }
      else
      for (int k = tid; k < ntodo; k += NT)
      {
         const int c = MARCH ? k : s_todo[k];
         if ( s_done[c] ) continue;
         const int x = c % p.cr[0], y = ( c/p.cr[0] ) % p.cr[1], z = c/( p.cr[0]*p.cr[1] );
         const int ic = ( p.c0[2] + z )*dz + ( p.c0[1] + y )*dy + p.c0[0] + x;
         T f[NV][8];
#        pragma unroll
         for (int v=0; v<NV; v++) interp_cell<T, SCHEME>( C + (size_t)v*C3, ic, dy, dz, PLAIN || ( ( p.mono >> v ) & 1 ), coeff,
                                                             !PLAIN && p.opp0, !PLAIN && p.mono_coeff < 0.0, f[v] );
         const int fo = ( p.f0[2] + 2*z )*fdz + ( p.f0[1] + 2*y )*fdy + p.f0[0] + 2*x;
         if ( store_fine( f, iterate, prim, p, F, F3, fo, fdy, fdz ) ) s_done[c] = 1; else s_fail = 1;
      }
      __syncthreads();
      const bool any = ( s_fail != 0 );
      if ( !iterate || !any ) break;
      if ( it == max_iter )
      {
         if ( tid == 0 ) atomicAdd( nfail, 1 );
         break;
      }
      __syncthreads();
   }
}

// Patch-group input window (N = 16 + 2 ghost <= 32 per axis): cell (x,y,z) from the patch slot[pg][Z/8][Y/8][X/8],
// (X,Y,Z) = (x,y,z) - ghost + 8; slot -1: from the fine box fbox at (x,y,z) + fb.origin, or kept if fbox == NULL.  Block
// (patch group, field, PREP_N cells of the window in linear order), a thread copies the cells t, t + 512, ...: every store
// instruction covers 64 consecutive cells and every load pieces of patch rows that lie side by side, and PREP_Q loads are in
// flight per lane.  (x,y,z) come from a float reciprocal: after the +0.5 shift, e/N^2 and r/N sit at least 1/(2 N^2) away
// from an integer, far above the float error for N <= 32.  The slot table goes through LDS, so that a cell's patch lookup is
// no second dependent global load.  Bound by memory.
// 512 patch groups with ghost 3 at a refinement boundary (218 MB FP32): 62 us within an AMR step, 48 alone; four consecutive
// cells a lane and one vector store 78 and 53.  FP64 alone 156 -> 100, without fine boxes 80 -> 73 (FP32 40 -> 44: what the
// caches hold); XCD-major blocks 89, 256 lanes with 6 cells 98, 21 cells 90.
constexpr int PREP_NT = 512, PREP_Q = 11, PREP_N = PREP_NT*PREP_Q;
template <typename IO>
__global__ void __launch_bounds__( PREP_NT )
prepare_patches_kernel( const IO *__restrict__ patch, const IO *__restrict__ fbox, IO *__restrict__ pg_in,
                        const int *__restrict__ slot, int ghost, BoxGeom fb )
{
   const int n = PS + 2*ghost, n2 = n*n, n3 = n2*n;
   const int p = blockIdx.x, v = blockIdx.y, bz = blockIdx.z;
   __shared__ int sl[64];
   if ( threadIdx.x < 64 ) sl[ threadIdx.x ] = slot[ (size_t)p*64 + threadIdx.x ];
   __syncthreads();
   const float rn = 1.0f/(float)n, rn2 = 1.0f/(float)n2;
   const int sx = fb.size[0], sxy = fb.size[1]*fb.size[0];
   const IO *pv = patch + (size_t)v*P3;
   const IO *fv = fbox ? fbox + ( (size_t)p*NV + v )*fb.size[2]*sxy + ( (size_t)fb.origin[2]*sxy + fb.origin[1]*sx + fb.origin[0] )
                       : nullptr;
   IO *dst = pg_in + ( (size_t)p*NV + v )*n3;
   IO   val[PREP_Q];
   bool put[PREP_Q];
#  pragma unroll
   for (int q=0; q<PREP_Q; q++)
   {
      const int e = bz*PREP_N + q*PREP_NT + (int)threadIdx.x;
      put[q] = false;
      if ( e >= n3 ) continue;
      const int z = (int)( ( (float)e + 0.5f )*rn2 ), r = e - z*n2, y = (int)( ( (float)r + 0.5f )*rn ), x = r - y*n;
      const int X = x - ghost + H, Y = y - ghost + H, Z = z - ghost + H;
      const int s = sl[ ( Z >> 3 )*16 + ( Y >> 3 )*4 + ( X >> 3 ) ];
      const IO *src = ( s >= 0 ) ? pv + ( (size_t)s*NV*P3 + ( Z & 7 )*H*H + ( Y & 7 )*H + ( X & 7 ) )
                                 : fv + ( (size_t)z*sxy + y*sx + x );
      put[q] = ( s >= 0 ) || fv;
      if ( put[q] ) val[q] = *src;
   }
#  pragma unroll
   for (int q=0; q<PREP_Q; q++)
      if ( put[q] ) dst[ bz*PREP_N + q*PREP_NT + (int)threadIdx.x ] = val[q];
}

// The same with four consecutive cells a lane, put as one vector where all are copied and the destination is aligned (N^3 is a
// multiple of 8, so a group never straddles two windows).  More blocks in flight for less work each: the faster one in FP32 for
// narrow windows and for few patch groups (us, caches warm / cold, against the form above: 512 patch groups without ghost zones
// 14.6 / 28 and 19 / 31; with ghost 3 64 8.6 / 11.7 and 11 / 13, 729 58 / 89 and 68 / 87, 216 with fine boxes 21 / 30 and 24 / 32),
// the slower one else (2000 with ghost 3 226 / 251 and 216 / 224; 512 with fine boxes in an AMR step 78 and 62; FP64 1024 265 and 177).
constexpr int PV_NT = 256, PV_N = 4;
template <typename IO> struct Vec4;
template <> struct Vec4<float>  { typedef float  type __attribute__(( ext_vector_type( 4 ) )); };
template <typename IO>
__global__ void __launch_bounds__( PV_NT )
prepare_patches_vec_kernel( const IO *__restrict__ patch, const IO *__restrict__ fbox, IO *__restrict__ pg_in,
                            const int *__restrict__ slot, int ghost, BoxGeom fb )
{
   const int p = blockIdx.x, v = blockIdx.y, n = PS + 2*ghost, n2 = n*n, n3 = n2*n;
   __shared__ int sl[64];
   if ( threadIdx.x < 64 ) sl[ threadIdx.x ] = slot[ (size_t)p*64 + threadIdx.x ];
   __syncthreads();
   const int e0 = ( blockIdx.z*PV_NT + threadIdx.x )*PV_N;
   if ( e0 >= n3 ) return;
   int z = (int)( ( (float)e0 + 0.5f )*( 1.0f/(float)n2 ) );
   const int r = e0 - z*n2;
   int y = (int)( ( (float)r + 0.5f )*( 1.0f/(float)n ) );
   int x = r - y*n;
   const IO *pv = patch + (size_t)v*P3;
   const IO *fv = fbox ? fbox + ( (size_t)p*NV + v )*fb.size[2]*fb.size[1]*fb.size[0] : nullptr;
   IO   val[PV_N];
   bool put[PV_N];
#  pragma unroll
   for (int k = 0; k < PV_N; k++)
   {
      const int X = x - ghost + H, Y = y - ghost + H, Z = z - ghost + H;
      const int s = sl[ ( Z >> 3 )*16 + ( Y >> 3 )*4 + ( X >> 3 ) ];
      put[k] = true;
      if ( s >= 0 )  val[k] = pv[ (size_t)s*NV*P3 + ( Z & 7 )*H*H + ( Y & 7 )*H + ( X & 7 ) ];
      else if ( fv ) val[k] = fv[ ( (size_t)( z + fb.origin[2] )*fb.size[1] + y + fb.origin[1] )*fb.size[0] + x + fb.origin[0] ];
      else           put[k] = false;
      // next cell of the window
      x++;
      const bool wx = ( x == n );
      x = wx ? 0 : x;
      y = wx ? y + 1 : y;
      const bool wy = ( y == n );
      y = wy ? 0 : y;
      z = wy ? z + 1 : z;
   }
   IO *dst = pg_in + ( (size_t)p*NV + v )*n3 + e0;
   const bool aligned = ( reinterpret_cast<size_t>( dst ) % sizeof( typename Vec4<IO>::type ) ) == 0;
   if ( aligned && put[0] && put[1] && put[2] && put[3] )
   {
      typename Vec4<IO>::type q;
      q.x = val[0];  q.y = val[1];  q.z = val[2];  q.w = val[3];
      *reinterpret_cast<typename Vec4<IO>::type*>( dst ) = q;
   }
   else
   {
#     pragma unroll
      for (int k = 0; k < PV_N; k++) if ( put[k] ) dst[k] = val[k];
   }
}

// box[q][v][z][y][x] (size) = patch[ slot[q][Z/8][Y/8][X/8] ][v][Z%8][Y%8][X%8], (X,Y,Z) = origin + (x,y,z);
// slot -1 keeps the box value.  Blocks of GB_N consecutive cells across boxes and fields, a thread copies the cells t, t + 256, ...,
// as above, with GB_Q loads in flight.  With patch2, half the sum of the cells of both: coarse data halfway between two times, where
// two passes over the whole level made them first (20 + 23 us of a two-level step of 4096 patches).  A cell's coordinates come from
// reciprocals instead of integer divisions, which are most of the instructions otherwise (512 boxes of 14^3 FP32 cells 18 us and
// 23): (e + 0.5)/nxy lies at least 1/(2 nxy) from an integer, and its error is below nz/2^22 in float, less than that for
// nxy*nz < 2^21 (SMALL: boxes of at most GB_SMALL cells), and far below it in double for the others.
// Bound by memory.  Blocks of one box and field each, of 512 x 6 cells, leave what a box does not fill: us, FP32, 4096 boxes: 1^3
// cells 49 -> 9.2, 8^3 52 -> 27, 9 x 9 x 9 51 -> 37, 16^3 252 -> 193; 512 of 14^3 the same 20.
constexpr int GB_NT = 256, GB_Q = 4, GB_N = GB_NT*GB_Q, GB_SMALL = 1 << 20;
template <typename IO, bool SMALL>
__global__ void __launch_bounds__( GB_NT )
gather_boxes_kernel( const IO *__restrict__ patch, const IO *__restrict__ patch2, IO *__restrict__ box, BoxGeom g,
                     const int *__restrict__ slot, long first, long total )
{
   using R = std::conditional_t<SMALL, float, double>;
   using I = std::conditional_t<SMALL, unsigned, unsigned long>;
   const I nx = g.size[0], nxy = nx*g.size[1], n = nxy*g.size[2];
   const size_t nt = (size_t)g.tdim[0]*g.tdim[1]*g.tdim[2];
   const R rx = (R)1/(R)nx, rxy = (R)1/(R)nxy;
   const ptrdiff_t other = patch2 ? patch2 - patch : 0;
   const IO *src[GB_Q];
   IO val[GB_Q];
   const long e0 = first + (long)blockIdx.x*GB_N + threadIdx.x;
#  pragma unroll
   for (int k=0; k<GB_Q; k++)
   {
      const long e = e0 + k*GB_NT;
      src[k] = nullptr;
      if ( e >= total ) continue;
      const unsigned long w = ( total >> 32 ) ? (unsigned long)e / n : (unsigned)e / (unsigned)n;
      const unsigned long q = ( total >> 32 ) ? w / NV : (unsigned)w / NV;
      const int v = (int)( w - q*NV );
      const I c = (I)( e - (long)( w*n ) );
      const I z = (I)( ( (R)c + (R)0.5 )*rxy ), r = c - z*nxy, y = (I)( ( (R)r + (R)0.5 )*rx ), x = r - y*nx;
      const int X = (int)x + g.origin[0], Y = (int)y + g.origin[1], Z = (int)z + g.origin[2];
      const int s = slot[ q*nt + ( (size_t)( Z >> 3 )*g.tdim[1] + ( Y >> 3 ) )*g.tdim[0] + ( X >> 3 ) ];
      if ( s >= 0 ) src[k] = patch + ( ( (size_t)s*NV + v )*P3 + ( Z & 7 )*H*H + ( Y & 7 )*H + ( X & 7 ) );
   }
#  pragma unroll
   for (int k=0; k<GB_Q; k++) if ( src[k] ) val[k] = *src[k];
   if ( patch2 )
#     pragma unroll
      for (int k=0; k<GB_Q; k++) if ( src[k] ) val[k] = ( val[k] + src[k][other] )*(IO)0.5;
#  pragma unroll
   for (int k=0; k<GB_Q; k++) if ( src[k] ) box[ e0 + k*GB_NT ] = val[k];
}

// The same, a block per (box, field, z plane) whose lanes take the plane's cells in linear order: the faster one for planes of many
// cells if there are enough of them, which keep the memory streams long (us, FP32: 64 boxes of 64^3 cells 172 -> 151, 8 of 128^3 186
// -> 166, 4096 of 256 x 16 x 1 150 -> 125), in FP64 only for thin boxes (2048 of 64 x 64 x 2 211 -> 202; 64 of 64^3 247 -> 280).
constexpr int GP_NT = 256;
template <typename IO>
__global__ void __launch_bounds__( GP_NT )
gather_planes_kernel( const IO *__restrict__ patch, const IO *__restrict__ patch2, IO *__restrict__ box, BoxGeom g,
                      const int *__restrict__ slot )
{
   const int q = blockIdx.x, v = blockIdx.y, z = blockIdx.z, Z = z + g.origin[2], nxy = g.size[0]*g.size[1];
   const int *sl = slot + (size_t)q*g.tdim[0]*g.tdim[1]*g.tdim[2] + (size_t)( Z >> 3 )*g.tdim[1]*g.tdim[0];
   IO *dst = box + ( ( (size_t)q*NV + v )*g.size[2] + z )*nxy;
   for (int e = threadIdx.x; e < nxy; e += GP_NT)
   {
      const int y = e / g.size[0], x = e - y*g.size[0], X = x + g.origin[0], Y = y + g.origin[1];
      const int s = sl[ (size_t)( Y >> 3 )*g.tdim[0] + ( X >> 3 ) ];
      if ( s < 0 ) continue;
      const size_t o = ( ( (size_t)s*NV + v )*H + ( Z & 7 ) )*H*H + ( Y & 7 )*H + ( X & 7 );
      dst[e] = patch2 ? ( patch[o] + patch2[o] )*(IO)0.5 : patch[o];
   }
}

} // namespace

// Boxes of one launch: 512 lanes each, and a grid dimension holds less than 2^32 lanes (a launch of more runs the number
// modulo 2^32, without an error)
constexpr long BOX_GRID = ( 1L << 23 ) - 1;
static unsigned boxes_from( long q0, long nbox ) { return (unsigned)( nbox - q0 < BOX_GRID ? nbox - q0 : BOX_GRID ); }

// Which form a call takes.  A list takes 19 one-dimensional passes a cell and field, a march 9 and 10 more a column, but the
// march's registers leave room for fewer waves and its planes are in sequence; and a block holds the registers of all its
// waves, busy or not, so that with many boxes idle lanes cost what busy ones would.  us, against a march of 256 lanes for all:
//   * few boxes: a list of as many lanes as cells, up to 512 (256 for the wide stencils in FP64 and QUAR).
//   * many boxes of up to 128 cells: a list of 64 or 128 lanes (CQUAD with clipping FP32, 2048 boxes of 2^3: 95 -> 11; VANLEER
//     FP64, 4096 of 8 x 8 x 2: 240 -> 87, with 512 lanes 300); of up to 256 cells 256 lanes.
//   * many boxes with a mask, of which few cells may be asked for: 128 lanes up to 512 cells (CQUAD with clipping FP32, 4096 of
//     8 x 8 x 2: 134 -> 48, with 512 lanes 193), 256 up to 1331; MINMOD3D and CQUAD without options in FP32, whose lists are short
//     of nothing but lanes, 512 from 257 on (MINMOD3D, 2048 of 8^3: 45, 128 lanes 54).
//   * the march for many boxes where options are in the kernel or the passes hold divisions in FP64 (`heavy`: there lists get
//     two waves per SIMD at most too): from three boxes per unit on, 128 lanes for 65 to 128 columns (QUAD with clipping FP32,
//     1024 of 10^3: 272 -> 150, list 203), 256 for more; 64 lanes for 33 to 64 columns from eight boxes per unit on (VANLEER with
//     clipping FP32, 4096 of 8 x 8 x 2: 163 -> 71, list 78).  Without options, in FP32, only for thin boxes of more than 128
//     columns (VANLEER, 1400 of 16 x 16 x 3: 94, list 123).
//   * CQUAD with a negative coefficient never takes the march, whose passes do not turn slopes around.
//   * CQUAR in FP32, many boxes: 256 lanes, or 128 where those hold all boxes at once; without options large boxes take four waves
//     per SIMD with some registers in scratch (512 of 12^3: 373 -> 280).
//   * MINMOD1D has one pass a cell: cell by cell, without a list, where the list takes as long as the passes, or where 256 lanes
//     hold all boxes at once and 512 do not (masked FP32, 1024 of 10^3: 31, list 41).
template <typename T, int S>
static void interp_launch( T *cdata, T *fdata, int nbox, const InterpPrm &p, int *nfail, hipStream_t stream )
{
   constexpr bool F64 = ( sizeof( T ) == 8 ), WIDE = ( S == 6 || S == 7 );
   const bool plain = ( p.mono & 0x1F ) == 0x1F && !p.opp0 && !( p.mono_coeff < 0.0 );
   const int  ncell = p.cr[0]*p.cr[1]*p.cr[2], ncol = p.cr[0]*p.cr[1], cus = device_cus();
   const bool many  = nbox >= 2*cus, full = nbox >= 3*cus, one_round = ( full && nbox <= 6*cus ), big = ncell >= 2048;
#  define GA_LAUNCH( PLAIN_, MARCH_, NT_, EU_ ) { hipLaunchKernelGGL( ( interpolate_kernel<T, S, PLAIN_, MARCH_, NT_, EU_> ), dim3( nbox ), dim3( NT_ ), \
                                                                0, stream, cdata, fdata, nbox, p, nfail );  return; }
#  define GA_LIST( NT_ ) { if ( plain ) GA_LAUNCH( true, false, NT_, 0 ) else GA_LAUNCH( false, false, NT_, 0 ) }
   if constexpr ( S == 2 )
   {
      if ( many && ( ncell <= 256 || ( p.need && ncell <= 600 && ( F64 || nbox >= 4*cus ) ) || ( p.need && !F64 && one_round && ncell <= 2000 ) ) )
         GA_LAUNCH( false, true, 256, 0 )
      if ( ncell <= 64 ) GA_LIST( 64 )
      GA_LIST( 512 )
   }
   else
   {
      if constexpr ( !WIDE )
         if ( !p.need && ncell > 64 && !( S == 4 && p.mono_coeff < 0.0 ) )
         {
            const bool heavy = !plain || ( F64 && ( S == 1 || S == 3 ) );
            if ( heavy && full && ncol > 64 && ncol <= 128 && ncell >= ( F64 && S == 1 ? 300 : 200 ) ) GA_LAUNCH( false, true, 128, 0 )
            if ( heavy && nbox >= 8*cus && ncol > 32 && ncol <= 64 && ncell >= 128 ) GA_LAUNCH( false, true, 64, 0 )
            if ( ( heavy && many && ( ( ncol > 128 && ncell > 256 ) || ncell >= 1200 ) ) || ( !plain && F64 && S != 4 && big ) ||
                 ( plain && !F64 && S != 4 && full && ncol > 128 && ncell >= 512 && p.cr[2] <= 4 ) || ( plain && S == 1 && many && big ) )
               GA_LAUNCH( false, true, 256, 0 )
         }
      const bool light = plain && !F64 && ( S == 1 || S == 4 );
      if ( ncell <= 64 ) GA_LIST( 64 )
      if ( ncell <= 128 || ( p.need && many && ncell <= ( light ? 256 : 512 ) ) || ( S == 6 && !F64 && plain && one_round && ncell <= 256 ) ) GA_LIST( 128 )
      if constexpr ( S == 6 && !F64 )
         if ( many && !p.need )
         {
            if ( !plain || ncell <= 256 ) GA_LIST( 256 )
            GA_LAUNCH( true, false, 512, 4 )
         }
      if ( S == 7 || ( S == 6 && F64 ) || ncell <= 256 || ( p.need && many && !light && ( ncell <= 1331 || WIDE ) ) || ( full && ncell <= 512 && !p.need ) ||
           ( S == 5 && F64 && many ) ) GA_LIST( 256 )
      if constexpr ( S != 7 && !( S == 6 && F64 ) ) GA_LIST( 512 )
   }
#  undef GA_LIST
#  undef GA_LAUNCH
}

template <typename T>
static int interpolate_boxes( T *cdata, T *fdata, int nbox, const InterpPrm &p, int *nfail, hipStream_t stream )
{
   switch ( p.scheme )
   {
      case 1: interp_launch<T, 1>( cdata, fdata, nbox, p, nfail, stream ); break;
      case 2: interp_launch<T, 2>( cdata, fdata, nbox, p, nfail, stream ); break;
      case 3: interp_launch<T, 3>( cdata, fdata, nbox, p, nfail, stream ); break;
      case 4: interp_launch<T, 4>( cdata, fdata, nbox, p, nfail, stream ); break;
      case 5: interp_launch<T, 5>( cdata, fdata, nbox, p, nfail, stream ); break;
      case 6: interp_launch<T, 6>( cdata, fdata, nbox, p, nfail, stream ); break;
      case 7: interp_launch<T, 7>( cdata, fdata, nbox, p, nfail, stream ); break;
      default: return -1;
   }
   return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
}

template <typename T>
int launch_interpolate( T *cdata, T *fdata, int nbox, const InterpPrm &p, int *nfail, hipStream_t stream )
{
   const long C3 = (long)p.cs[0]*p.cs[1]*p.cs[2], F3 = (long)p.fs[0]*p.fs[1]*p.fs[2], ncell = (long)p.cr[0]*p.cr[1]*p.cr[2];
   int rc = 0;
   for (long q0 = 0; q0 < nbox && rc == 0; q0 += BOX_GRID)
   {
      InterpPrm part = p;
      if ( p.need ) part.need = p.need + q0*ncell;
      rc = interpolate_boxes( cdata + q0*NV*C3, fdata + q0*NV*F3, (int)boxes_from( q0, nbox ), part, nfail, stream );
   }
   return rc;
}

template <typename IO>
int launch_prepare_patches( const IO *patch, IO *pg_in, int npg, const int *slot, int ghost, hipStream_t stream )
{
   return launch_assemble<IO>( patch, nullptr, pg_in, npg, slot, ghost, BoxGeom{}, stream );
}

template <typename IO>
int launch_gather_boxes( const IO *patch, const IO *patch2, IO *box, int nbox, const BoxGeom &g, const int *slot, hipStream_t stream )
{
   if ( nbox <= 0 ) return 0;
   const long nxy = (long)g.size[0]*g.size[1], n = nxy*g.size[2], total = (long)nbox*NV*n, planes = (long)nbox*NV*g.size[2];
   if ( nxy >= ( sizeof( IO ) == 4 ? 512 : 1024 ) && ( sizeof( IO ) == 4 || g.size[2] <= 4 ) && planes >= 1900 && nxy < ( 1L << 30 ) && nbox <= BOX_GRID )
   {
      hipLaunchKernelGGL( gather_planes_kernel<IO>, dim3( nbox, NV, g.size[2] ), dim3( GP_NT ), 0, stream, patch, patch2, box, g, slot );
      return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
   }
   constexpr long most = BOX_GRID*GB_N;                                     // cells of one launch
   for (long first = 0; first < total; first += most)
   {
      const long left = total - first, part = left < most ? left : most;
      const dim3 grid( (unsigned)( ( part + GB_N - 1 )/GB_N ) );
      if ( n <= GB_SMALL ) hipLaunchKernelGGL( ( gather_boxes_kernel<IO, true> ), grid, dim3( GB_NT ), 0, stream, patch, patch2, box, g, slot, first, total );
      else hipLaunchKernelGGL( ( gather_boxes_kernel<IO, false> ), grid, dim3( GB_NT ), 0, stream, patch, patch2, box, g, slot, first, total );
   }
   return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
}

template <typename IO>
int launch_assemble( const IO *patch, const IO *fbox, IO *pg_in, int npg, const int *slot, int ghost, const BoxGeom &fb,
                     hipStream_t stream )
{
   if ( npg <= 0 ) return 0;
   const int n = PS + 2*ghost;
   if constexpr ( sizeof( IO ) == 4 )
      if ( ghost <= 2 || npg <= ( fbox ? 1 : 3 )*device_cus() )
      {
         hipLaunchKernelGGL( prepare_patches_vec_kernel<IO>, dim3( npg, NV, ( n*n*n + PV_NT*PV_N - 1 )/( PV_NT*PV_N ) ), dim3( PV_NT ), 0, stream,
                             patch, fbox, pg_in, slot, ghost, fb );
         return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
      }
   hipLaunchKernelGGL( prepare_patches_kernel<IO>, dim3( npg, NV, ( n*n*n + PREP_N - 1 )/PREP_N ), dim3( PREP_NT ), 0, stream,
                       patch, fbox, pg_in, slot, ghost, fb );
   return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
}

#define GA_INSTANTIATE( T ) \
template int launch_gather_boxes<T>( const T*, const T*, T*, int, const BoxGeom&, const int*, hipStream_t ); \
template int launch_assemble<T>( const T*, const T*, T*, int, const int*, int, const BoxGeom&, hipStream_t ); \
template int launch_interpolate<T>( T*, T*, int, const InterpPrm&, int*, hipStream_t ); \
template int launch_prepare_patches<T>( const T*, T*, int, const int*, int, hipStream_t );
// INTERP_PRECISION (32 or 64; both if undefined): the build compiles the two precisions as two objects at the same time
#if !defined( INTERP_PRECISION ) || INTERP_PRECISION == 64
GA_INSTANTIATE( double )
#endif
#if !defined( INTERP_PRECISION ) || INTERP_PRECISION == 32
GA_INSTANTIATE( float )
#endif
#undef GA_INSTANTIATE

} // namespace gamer_amd

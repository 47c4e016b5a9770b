// Adjoint (vector-Jacobian product) and tangent-linear (Jacobian-vector product) of one MHM_RP step, FP64.
//
// The step is the map U_in (22^3 x 5 per patch group) -> U_out (16^3 x 5) of the forward kernel
// (src/Model_Hydro/CPU_Hydro/CPU_FluidSolver_MHM.cpp:263-589 with the half-step prediction of :615-949).
// Explicit phases over a per-PG global workspace, one kernel for one or two phases over all patch groups:
//
//   forward   F1 + F2, z plane by z plane: half-step fluxes (Hydro_RiemannPredict_Flux) in LDS, then the half-step
//                update, floors and primitive W (Hydro_RiemannPredict) -> ws
//             F4 (tangent / plain forward only) PLM faces (Hydro_DataReconstruction) and the full-step flux of
//                each face, then the update of the 16^3 output cells
//   reverse   R4 lambda_F of each full-step face from lambda_out (transpose of Hydro_FullStepUpdate),
//                lambda_FC = J_RS^T lambda_F (transpose of Hydro_ComputeFlux), with the two PLM faces of the
//                face recomputed from W
//             R3 + R2, z plane by z plane: lambda_W = sum over the three stencil cells of J_PLM^T lambda_FC
//                (transpose of the limiter, face clamp and mirror) in LDS, then lambda_U_half = J_Con2Pri^T lambda_W
//                (transpose of the floors and primitive conversion) -> ws
//             R1 + R0, z plane by z plane: lambda of every half-step face, J_RS^T of the cell-centred half-step
//                solve per side, and lambda_in = lambda_out (core) + lambda_U_half + the half-step face contributions
//
// The reverse sweep is written out by hand.  The Riemann solves (HLLC, HLLE and Roe) run backwards as hand-written
// reverse-mode sweeps (hydro_reverse.hpp: solver + interface-state builders, one pass per face for all ten
// inputs).  The PLM reconstruction (face clamps and mirror) is reversed by hand for every
// limiter, with the limited slope's two partials from a two-direction dual evaluation (written out for VL_GMINMOD).  The half-step conversion
// with floors takes its local Jacobian from forward-mode dual numbers (hydro_dual.hpp) pushed through the same
// templated device function, one input direction at a time.  All forms take exactly the branches of the forward
// evaluation of this file (F12, F4), which solves the interfaces by rs_hllc(), rs_hlle() and rs_roe().  The marching
// kernels solve them by hllc_flux() and its twins of hydro_math.hpp: the same functions rounded differently, so that a
// face within rounding of a kink (a floor, a wave speed of 0) may be on the other side of it there.
// The reverse phases are gathers: every workspace entry has one writer, so there are no atomics and the result
// is deterministic.
//
// Scope: MHM_RP, FP64, any Riemann solver and limiter of the forward path.  The MinMod retry is not
// differentiated (the first-iteration coefficient is used); dt and dh are constants.
//
// No floating-point contraction of values in this translation unit (it holds only the derivative kernels, and the
// pragma comes before the solver headers it instantiates).  Every value is then the rounded result of its own
// source expression, with fused multiply-adds only where fmad() is written, so the dual-number evaluation, the
// plain recomputation inside the reverse sweeps and the forward phases all produce bitwise equal values and
// split ties the same way.  hydro_reverse.hpp turns contraction on for the adjoints alone, from which no branch depends.  Ties are common: a uniform floored region puts the HLLC star pressure on the
// pressure floor up to rounding, and the floor decides whether its derivative passes.

#pragma clang fp contract(off)

// the derivative phases and their dual-number twins take the sound speed as sqrt(gamma P / rho) (see sound_speed)
#define HYDRO_IEEE_SOUND_SPEED
#include "hydro_dual.hpp"
#include "hydro_kernels.hpp"
#include "hydro_reverse.hpp"

namespace gamer_amd {

namespace {

constexpr int NX = 22, N2 = NX*NX, N3 = NX*N2;
constexpr int PS = 16;
constexpr int NT = 256;
constexpr int STRIDE[3] = { 1, NX, N2 };

// workspace layout per patch group, in units of N3 doubles.  Written / last read by:
constexpr int WS_W   = 0;            // [5]       half-step primitives (cells 1..20)            F1+F2 / R3
constexpr int WS_LFC = 5;            // [3][2][5][NLC] lambda of the full-step faces, dense     R4 / R3
constexpr int WS_LU  = 40;           // [5]       lambda of the half-step conserved state       R2 / R0
constexpr int WS_H   = 45;           // [5]       half-step conserved state                     F1+F2 / R2
constexpr int WS_ADJ = 50;
// lambda of the full-step faces, per direction, side and field a dense block over the reconstruction's centres (normal 2..19,
// tangential 3..18) with x fastest, so that rows are whole cache lines: as rows of 16 out of 22 cells,
// R4 on 512 patch groups took 357 us, this takes 273.
constexpr int NLC = 18*16*16;
constexpr int LFC0 = ( WS_LFC*N3 + 15 )/16*16;           // its first element, on a cache line
static_assert( LFC0 + 30*NLC <= WS_LU*N3 && WS_H + NV <= WS_ADJ, "workspace slots overlap" );
__device__ __forceinline__ int lfc_cell( int d, int i, int j, int k )
{
   return ( d == 0 ) ? ( i - 2 ) + 18*( ( j - 3 ) + 16*( k - 3 ) )
        : ( d == 1 ) ? ( i - 3 ) + 16*( ( j - 2 ) + 18*( k - 3 ) )
        :              ( i - 3 ) + 16*( ( j - 3 ) + 16*( k - 2 ) );
}

__device__ __forceinline__ void coords( int c, int &i, int &j, int &k ) { i = c % NX;  j = ( c / NX ) % NX;  k = c / N2; }
__device__ __forceinline__ bool in_rng( int x, int lo, int hi ) { return x >= lo && x <= hi; }

// face c + 1/2 e_d with normal coordinate n, tangential a, b
__device__ __forceinline__ void split( int d, int i, int j, int k, int &n, int &a, int &b )
{
   n = ( d == 0 ) ? i : ( d == 1 ) ? j : k;
   a = ( d == 0 ) ? j : i;
   b = ( d == 2 ) ? j : k;
}
__device__ __forceinline__ bool half_face( int n, int a, int b ) { return in_rng( n, 0, 20 ) && in_rng( a, 1, 20 ) && in_rng( b, 1, 20 ); }
__device__ __forceinline__ bool core3( int i, int j, int k ) { return in_rng( i, 3, 18 ) && in_rng( j, 3, 18 ) && in_rng( k, 3, 18 ); }
__device__ __forceinline__ int  out_index( int i, int j, int k ) { return ( i - 3 ) + PS*( ( j - 3 ) + PS*( k - 3 ) ); }

// The phases enumerate only the cells or faces they work on (a box [lo, lo + len) per axis, x fastest, so that
// neighbouring lanes read neighbouring cells) instead of striding over the whole 22^3 block and skipping.
struct Box { int lx, ly, lz, nx, ny, nz; };
__device__ __forceinline__ int box_cell( const Box &b, int e, int &i, int &j, int &k )
{
   const int x = e % b.nx, r = e / b.nx, y = r % b.ny, z = r / b.ny;
   i = b.lx + x;  j = b.ly + y;  k = b.lz + z;
   return i + NX*j + N2*k;
}
// d-normal faces c + 1/2 e_d with normal coordinate in [n0, n0 + nn) and both tangential ones in [t0, t0 + nt)
__device__ __forceinline__ Box face_box( int d, int n0, int nn, int t0, int nt )
{
   Box b;
   b.lx = ( d == 0 ) ? n0 : t0;  b.nx = ( d == 0 ) ? nn : nt;
   b.ly = ( d == 1 ) ? n0 : t0;  b.ny = ( d == 1 ) ? nn : nt;
   b.lz = ( d == 2 ) ? n0 : t0;  b.nz = ( d == 2 ) ? nn : nt;
   return b;
}
constexpr int NHF = 21*20*20;        // half-step faces per direction: normal 0..20, tangential 1..20
constexpr int NFF = 17*16*16;        // full-step faces per direction: normal 2..18, tangential 3..18
constexpr Box CORE_CELLS = { 3, 3, 3, 16, 16, 16 };

// ---------------- pieces of the step, generic in the arithmetic type ----------------
// cell-centred interface state of the half step (pressure recovery + floor, 1/rho, sound speed)
template <typename T>
__device__ __forceinline__ St<T> cell_st( int d, const T u[NV], const Prm<T> &P )
{
   const T ir = rcp( u[0] );
   const T eint = u[4] - (T)0.5*( u[1]*u[1] + u[2]*u[2] + u[3]*u[3] )*ir;
   const T p = floor_pres( eint*P.gm1, P.min_pres );
   return cell_state( d, u, p, ir, vsqrt( P.gamma*p*ir ) );
}

template <int RS, typename T>
__device__ __forceinline__ void half_flux( int d, const T uL[NV], const T uR[NV], const Prm<T> &P, T f[NV] )
{
   riemann<RS>( d, cell_st( d, uL, P ), cell_st( d, uR, P ), P, f );
}

template <int RS, typename T>
__device__ __forceinline__ void full_flux( int d, const T wL[NV], const T wR[NV], const Prm<T> &P, T f[NV] )
{
   riemann<RS>( d, face_state( d, wL, P ), face_state( d, wR, P ), P, f );
}

// reverse sweeps of half_flux / full_flux: bL, bR = (d flux / d input side)^T bf, one pass
template <int RS>
__device__ __forceinline__ void half_flux_rev( int d, const double uL[NV], const double uR[NV], const Prm<double> &P,
                                               const double bf[NV], double bL[NV], double bR[NV] )
{
   const StD L = cell_st( d, uL, P ), Q = cell_st( d, uR, P );
   StD sL, sQ;
   riemann_rev<RS>( d, L, Q, P, bf, sL, sQ );
   cell_st_rev( d, uL, L, sL, P, bL );
   cell_st_rev( d, uR, Q, sQ, P, bR );
}

template <int RS>
__device__ __forceinline__ void full_flux_rev( int d, const double wL[NV], const double wR[NV], const Prm<double> &P,
                                               const double bf[NV], double bL[NV], double bR[NV] )
{
   const StD L = face_state( d, wL, P ), Q = face_state( d, wR, P );
   StD sL, sQ;
   riemann_rev<RS>( d, L, Q, P, bf, sL, sQ );
   face_state_rev( d, wL, L, sL, P, bL );
   face_state_rev( d, wR, Q, sQ, P, bR );
}

// half-step conserved state -> density floor, internal-energy floor, primitive variables with pressure floor
// (CPU_FluidSolver_MHM.cpp:900-933)
template <typename T>
__device__ __forceinline__ void con2pri_floor( const T u[NV], const Prm<T> &P, T w[NV] )
{
   T c[NV];
#  pragma unroll
   for (int v=0; v<NV; v++) c[v] = u[v];
   c[0] = vmax( c[0], P.min_dens );
   const T r  = rcp( c[0] );
   const T ke = (T)0.5*( c[1]*c[1] + c[2]*c[2] + c[3]*c[3] )*r;
   T ein = c[4] - ke;
   const T eout = ( ein == ein ) ? vmax( ein, P.min_eint ) : ein;
   if ( ein != eout ) { c[4] = c[4] - ein + eout;  ein = c[4] - ke; }
   w[0] = c[0];
   w[1] = c[1]*r;
   w[2] = c[2]*r;
   w[3] = c[3]*r;
   const T p = ein*P.gm1;
   w[4] = ( p == p ) ? vmax( p, P.min_pres ) : p;
}

template <int LIM, typename T>
__device__ __forceinline__ void plm( const T &L, const T &C, const T &R, const Prm<T> &P, T &fL, T &fR )
{
   plm_face<LIM>( L, C, R, P.limiter, P.coeff, fL, fR );
}

// ---------------- workspace views ----------------
// The adjoint keeps h (read by R2) in its own slots; the tangent kernels store W as dual
// numbers (two doubles each).
static_assert( 2*NV <= WS_ADJ, "tangent workspace must fit the per-PG slot" );

template <typename T>
struct Fwd {
   T *W;
   __device__ Fwd( T *base ) : W( base + WS_W*N3 ) {}
   __device__ T &w( int v, int c ) { return W[ v*N3 + c ]; }
};

// load cell c of the input (value, and tangent for Dual<1>)
template <typename T> struct Load;
template <> struct Load<double>
{
   __device__ static void cell( const double *in, const double *, int c, double u[NV] )
   {
#     pragma unroll
      for (int v=0; v<NV; v++) u[v] = in[ v*N3 + c ];
   }
};
template <> struct Load< Dual<1> >
{
   __device__ static void cell( const double *in, const double *tin, int c, Dual<1> u[NV] )
   {
#     pragma unroll
      for (int v=0; v<NV; v++) { u[v] = Dual<1>( in[ v*N3 + c ] );  u[v].d[0] = tin[ v*N3 + c ]; }
   }
};

// ---------------- phases: one kernel each, one element per lane ----------------
// Every phase is a gather over the faces or cells of each patch group that reads only what earlier phases wrote, so the
// phases run as separate kernels in stream order, each over many workgroups per patch group: R4 and F4 over flat grids of
// bpp(count) workgroups (element e of patch group pg is lane e % NT of workgroup pg*bpp + e / NT), the others over blocks of
// rows and planes.  One workgroup marching through all phases of its patch group kept only 4 waves per patch group busy;
// spread over the grid, a phase keeps as many patch groups' workspace traffic in flight as its registers allow.
constexpr int bpp( int count ) { return ( count + NT - 1 ) / NT; }
constexpr int N_F4 = PS*PS*PS, N_R4 = 3*NFF;

// Consecutive logical blocks of a phase share data (the planes k-1..k+1 of a plane-per-workgroup phase, the W
// stencils of neighbouring face blocks), so every phase takes its block index from xcd_block() (hydro_kernels.hpp).
struct Elem { int pg, e; };
__device__ __forceinline__ Elem elem( int count )
{
   const int b = bpp( count ), l = (int)xcd_block();       // grids_fit keeps the grid below 2^31 blocks
   return { l / b, ( l % b )*NT + (int)threadIdx.x };
}

template <typename T>
__device__ __forceinline__ Prm<T> phase_prm( const Prm<double> &P0, double minmod_coeff )
{
   Prm<T> P = prm_as<T>( P0 );
   P.coeff = vmax( (T)minmod_coeff, (T)0.0 );
   return P;
}

template <typename T> struct Store;
template <> struct Store<double>
{
   __device__ static void put( double *out, double *, size_t o, const double &x ) { out[o] = x; }
};
template <> struct Store< Dual<1> >
{
   __device__ static void put( double *out, double *tout, size_t o, const Dual<1> &x ) { if ( out ) out[o] = x.v;  tout[o] = x.d[0]; }
};

constexpr size_t NIN = (size_t)NV*N3, NOUT = (size_t)NV*PS*PS*PS;

// F1 + F2: a workgroup takes JR rows (y) of KS planes (z), plane by plane.  The half-step fluxes of the plane's x
// and y faces and of the z faces above it (Hydro_RiemannPredict_Flux) go to LDS, where the z faces below it are from the
// plane before (solved first for the first plane), then the cells take the half-step update (x and y flux differences,
// then z, as the production kernel), the floors and the primitive conversion (Hydro_RiemannPredict).  The fluxes never
// reach memory; the price is that faces between workgroups are solved by both.  h_off >= 0 (FP64 only): the half-step state h
// is stored too, for R2.  With one whole plane per workgroup every z face was solved twice: 512 patch groups 264 us, this
// takes 238; half as many rows 240, five planes 242.  What the cell contributes to its six faces (pressure, 1/rho, sound
// speed) kept in LDS instead of recomputed took 265: the solves wait, the vector units do not bound it.  Calls of few patch
// groups take blocks of one plane (few_blocks()).
template <int JR_, int KS_>
struct F12
{
   static constexpr int JR = JR_, KS = KS_, RB = 20/JR, KB = 20/KS, BPP = RB*KB;
   static constexpr int NXF = 21*JR, NYF = 20*( JR + 1 ), NZF = 20*JR;
   static_assert( 20 % JR == 0 && 20 % KS == 0, "the blocks must tile the 20 x 20 half-step rows and planes" );
};
constexpr int F12_NT = 256;
typedef F12<10, 4> F12Large;
typedef F12<5, 1>  F12Small;

template <int RS, typename T, typename B>
__global__ void __launch_bounds__( F12_NT )
f12_kernel( const double *__restrict__ g_in, const double *__restrict__ g_tin, double *__restrict__ g_ws, int h_off,
            Prm<double> P0, double minmod_coeff )
{
   __shared__ double s_raw[NV*( B::NXF + B::NYF + 2*B::NZF )*( sizeof( T )/sizeof( double ) )];
   T *sX = reinterpret_cast<T*>( s_raw ), *sY = sX + NV*B::NXF, *sZ = sY + NV*B::NYF;      // [v][face]; sZ [k % 2][v][face]
   const int tid = threadIdx.x, lb = (int)xcd_block(), rb = lb % B::RB, kb = ( lb / B::RB ) % B::KB, pg = lb / B::BPP;
   const int j0 = rb*B::JR, ka = 1 + kb*B::KS;                 // rows j0 + 1 .. j0 + JR, planes ka .. ka + KS - 1
   const Prm<T> P = phase_prm<T>( P0, minmod_coeff );
   const double *in = g_in + pg*NIN, *tin = g_tin ? g_tin + pg*NIN : nullptr;
   Fwd<T> F( reinterpret_cast<T*>( g_ws + (size_t)pg*WS_ADJ*N3 ) );
   constexpr bool ONE = ( B::KS == 1 );                          // one plane: the z faces below it come with its own
#  pragma unroll 1
   for (int k = ONE ? ka : ka - 1; k < ka + B::KS; k++)
   {
      // faces, stored at their low cell: x (normal i = 0..20), y (normal j0 .. j0 + JR), then the z faces with low cell
      // in plane k (ONE: and those in plane k - 1); lanes run along x
      const int f0 = ( !ONE && k < ka ) ? B::NXF + B::NYF : 0;
      for (int f = f0 + tid; f < B::NXF + B::NYF + ( ONE ? 2 : 1 )*B::NZF; f += F12_NT)
      {
         int d, i, j, kf = k, r = f, n = B::NXF;
         T *dst = sX;
         if ( f < B::NXF )                 { d = 0;  i = r % 21;  j = j0 + 1 + r / 21; }
         else if ( f < B::NXF + B::NYF )  { d = 1;  r = f - B::NXF;  i = 1 + r % 20;  j = j0 + r / 20;  dst = sY;  n = B::NYF; }
         else
         {
            d = 2;  r = f - B::NXF - B::NYF;
            if ( ONE && r >= B::NZF ) { r -= B::NZF;  kf = k - 1; }
            i = 1 + r % 20;  j = j0 + 1 + r / 20;  dst = sZ + ( kf & 1 )*NV*B::NZF;  n = B::NZF;
         }
         const int c = i + NX*j + N2*kf;
         T uL[NV], uR[NV], fl[NV];
         Load<T>::cell( in, tin, c, uL );
         Load<T>::cell( in, tin, c + ( d == 0 ? 1 : d == 1 ? NX : N2 ), uR );
         half_flux<RS>( d, uL, uR, P, fl );
#        pragma unroll
         for (int v=0; v<NV; v++) dst[ v*n + r ] = fl[v];
      }
      __syncthreads();
      if ( k >= ka )
      for (int e = tid; e < B::NZF; e += F12_NT)
      {
         const int i = 1 + e % 20, jr = e / 20, c = i + NX*( j0 + 1 + jr ) + N2*k;
         const int xh = i + 21*jr, yh = ( i - 1 ) + 20*( jr + 1 );
         const T *zu = sZ + ( k & 1 )*NV*B::NZF + e, *zl = sZ + ( ( k - 1 ) & 1 )*NV*B::NZF + e;
         T u[NV], h[NV], w[NV];
         Load<T>::cell( in, tin, c, u );
#        pragma unroll
         for (int v=0; v<NV; v++)
         {
            const T *fx = sX + v*B::NXF + xh, *fy = sY + v*B::NYF + yh;
            const T dxy = ( fx[0] - fx[-1] ) + ( fy[0] - fy[-20] );
            h[v] = u[v] - P.dt_dh2*( dxy + ( zu[v*B::NZF] - zl[v*B::NZF] ) );
         }
         con2pri_floor( h, P, w );
#        pragma unroll
         for (int v=0; v<NV; v++) F.w( v, c ) = w[v];
         if constexpr ( std::is_same<T, double>::value )
            if ( h_off >= 0 )
            {
               double *H = g_ws + (size_t)pg*WS_ADJ*N3 + (size_t)h_off*N3;
#              pragma unroll
               for (int v=0; v<NV; v++) H[ v*N3 + c ] = h[v];
            }
      }
      __syncthreads();
   }
}

// F4 (tangent / plain forward), in two kernels.  f4_face_kernel: the full-step flux of each of the 13,056 faces
// (3 x 17 x 16 x 16, low cell 2..18 along the normal, tangential 3..18), once per face, with its two PLM faces
// recomputed from the half-step primitives W as the adjoint's R4 does; the fluxes go to the workspace.
// f4_update_kernel: the full-step update of the 16^3 output cells from the fluxes of their faces.
// T = Dual<1>: out = U_out (optional), tout = J v; T = double: out = U_out.
constexpr int WS_TF = 2*NV;          // tangent flux slots: [3][5][NFF] values of T, after W (5 values of T per cell)
static_assert( WS_TF*N3 + 3*NV*NFF*2 <= WS_ADJ*N3, "tangent fluxes must fit the per-PG workspace" );

// index of the d-normal face with low cell (i, j, k) in face_box(d, 2, 17, 3, 16)
__device__ __forceinline__ int full_face_index( int d, int i, int j, int k )
{
   return ( d == 0 ) ? ( i - 2 ) + 17*( ( j - 3 ) + 16*( k - 3 ) )
        : ( d == 1 ) ? ( i - 3 ) + 16*( ( j - 2 ) + 17*( k - 3 ) )
        :              ( i - 3 ) + 16*( ( j - 3 ) + 16*( k - 2 ) );
}

template <int RS, int LIM, typename T>
__global__ void __launch_bounds__( NT )
f4_face_kernel( double *__restrict__ g_ws, Prm<double> P0, double minmod_coeff )
{
   const Elem x = elem( 3*NFF );
   if ( x.e >= 3*NFF ) return;
   const Prm<T> P = phase_prm<T>( P0, minmod_coeff );
   T *ws = reinterpret_cast<T*>( g_ws + (size_t)x.pg*WS_ADJ*N3 );
   Fwd<T> F( ws );
   T *tf = ws + (size_t)WS_TF*N3/( sizeof( T )/sizeof( double ) );
   const int d = x.e / NFF, q = x.e - d*NFF;
   int i, j, k;
   const int c = box_cell( face_box( d, 2, 17, 3, 16 ), q, i, j, k );
   const int s = STRIDE[d];
   T wl[NV], wr[NV], f[NV];
#  pragma unroll
   for (int v=0; v<NV; v++)
   {
      const T wm = F.w( v, c - s ), w0 = F.w( v, c ), w1 = F.w( v, c + s ), w2 = F.w( v, c + 2*s );
      T dummy;
      plm<LIM>( wm, w0, w1, P, dummy, wl[v] );      // R face of the low cell
      plm<LIM>( w0, w1, w2, P, wr[v], dummy );      // L face of the high cell
   }
   // Roe on dual numbers needs more than 256 registers with run-time selects of the direction: a copy of the solve per
   // direction, chosen for the whole workgroup, takes 64 patch groups from 208 to 190 us for the whole call and 512 from
   // 1697 to 1563.  HLLC gains 1% at 64, HLLE loses 2% at 512
   if constexpr ( RS == 2 )
   {
      static_assert( NFF % NT == 0, "a workgroup's faces have one direction" );
      const int du = __builtin_amdgcn_readfirstlane( d );
      if      ( du == 0 ) full_flux<RS>( 0, wl, wr, P, f );
      else if ( du == 1 ) full_flux<RS>( 1, wl, wr, P, f );
      else                full_flux<RS>( 2, wl, wr, P, f );
   }
   else
      full_flux<RS>( d, wl, wr, P, f );
#  pragma unroll
   for (int v=0; v<NV; v++) tf[ ( d*NV + v )*NFF + q ] = f[v];
}

template <typename T>
__global__ void __launch_bounds__( NT )
f4_update_kernel( const double *__restrict__ g_in, const double *__restrict__ g_tin, double *__restrict__ g_out,
                  double *__restrict__ g_tout, double *__restrict__ g_ws, Prm<double> P0, double minmod_coeff )
{
   const Elem x = elem( N_F4 );
   if ( x.e >= N_F4 ) return;
   const Prm<T> P = phase_prm<T>( P0, minmod_coeff );
   const double *in = g_in + x.pg*NIN, *tin = g_tin ? g_tin + x.pg*NIN : nullptr;
   double *out = g_out ? g_out + x.pg*NOUT : nullptr, *tout = g_tout ? g_tout + x.pg*NOUT : nullptr;
   const T *tf = reinterpret_cast<const T*>( g_ws + (size_t)x.pg*WS_ADJ*N3 ) + (size_t)WS_TF*N3/( sizeof( T )/sizeof( double ) );
   int i, j, k;
   const int c = box_cell( CORE_CELLS, x.e, i, j, k );
   T u[NV], dF[3][NV];
   Load<T>::cell( in, tin, c, u );
   for (int d=0; d<3; d++)
   {
      const int qp = full_face_index( d, i, j, k );                                 // face c + 1/2
      const int qm = full_face_index( d, i - ( d == 0 ), j - ( d == 1 ), k - ( d == 2 ) );   // face c - 1/2
#     pragma unroll
      for (int v=0; v<NV; v++) dF[d][v] = tf[ ( d*NV + v )*NFF + qp ] - tf[ ( d*NV + v )*NFF + qm ];
   }
   const size_t o = out_index( i, j, k );
#  pragma unroll
   for (int v=0; v<NV; v++)
      Store<T>::put( out, tout, (size_t)v*PS*PS*PS + o, u[v] - P.dt_dh*( ( dF[0][v] + dF[1][v] ) + dF[2][v] ) );
}

// ---------------- reverse phases ----------------
struct Adj {
   double *LU, *LFC;
   __device__ Adj( double *base ) : LU( base + WS_LU*N3 ), LFC( base + LFC0 ) {}
   __device__ double &lu( int v, int c )                { return LU[ v*N3 + c ]; }
   __device__ double &lfc( int d, int s, int v, int e ) { return LFC[ ( ( d*2 + s )*NV + v )*NLC + e ]; }     // e: lfc_cell()
};

typedef Dual<1> D1;

// R4 full-step faces: lambda_F = dt/dh (lambda_out(c+e_d) - lambda_out(c)), then J_RS^T per side.  Only the
// faces that feed a full-step flux receive a value; R3 reads the others as zero.
template <int RS, int LIM>
__global__ void __launch_bounds__( NT )
r4_kernel( const double *__restrict__ g_lout, double *__restrict__ g_ws, Prm<double> P0, double minmod_coeff )
{
   const Elem x = elem( N_R4 );
   if ( x.e >= N_R4 ) return;
   const Prm<double> P = phase_prm<double>( P0, minmod_coeff );
   const double *lout = g_lout + x.pg*NOUT;
   double *ws = g_ws + (size_t)x.pg*WS_ADJ*N3;
   Fwd<double> F( ws );
   Adj A( ws );
   const int d = x.e / NFF;
   int i, j, k;
   const int c = box_cell( face_box( d, 2, 17, 3, 16 ), x.e - d*NFF, i, j, k );
   const int s = STRIDE[d];
   int i2 = i, j2 = j, k2 = k;
   if ( d == 0 ) i2++; else if ( d == 1 ) j2++; else k2++;
   double lf[NV];
   const bool lo = core3( i, j, k ), hi = core3( i2, j2, k2 );
#  pragma unroll
   for (int v=0; v<NV; v++)
   {
      const double ll = lo ? lout[ (size_t)v*PS*PS*PS + out_index( i, j, k ) ] : 0.0;
      const double lh = hi ? lout[ (size_t)v*PS*PS*PS + out_index( i2, j2, k2 ) ] : 0.0;
      lf[v] = P.dt_dh*( lh - ll );
   }
   // the R face of c and the L face of c + e_d (F3's values, recomputed from the half-step primitives)
   double wl[NV], wr[NV];
#  pragma unroll
   for (int v=0; v<NV; v++)
   {
      const double wm = F.w( v, c - s ), w0 = F.w( v, c ), w1 = F.w( v, c + s ), w2 = F.w( v, c + 2*s );
      double fl, fr;
      plm<LIM>( wm, w0, w1, P, fl, wl[v] );
      plm<LIM>( w0, w1, w2, P, wr[v], fr );
   }
   // one reverse sweep for both sides
   double gl[NV] = { 0.0, 0.0, 0.0, 0.0, 0.0 }, gr[NV] = { 0.0, 0.0, 0.0, 0.0, 0.0 };
   full_flux_rev<RS>( d, wl, wr, P, lf, gl, gr );
   const int e = lfc_cell( d, i, j, k ), es = ( d == 0 ) ? 1 : ( d == 1 ) ? 16 : 256;
#  pragma unroll
   for (int v=0; v<NV; v++) { A.lfc( d, 1, v, e ) = gl[v];  A.lfc( d, 0, v, e + es ) = gr[v]; }
}

// R3 + R2: a workgroup takes R32_KS planes of the half-step cells.  Step n: every lane reverses reconstruction stencils
// (plm_face_rev) of all fields, those along z with centre plane n and those along x and y in plane n - 1, whose z neighbours
// are done by then.  The stencils along x and y leave the adjoints of their three cells in LDS; those along z march, a lane
// per (field, column), with the two cell adjoints still open in registers, and leave the one that is complete.  Then each
// cell of plane n - 1 sums x, y and z in this order (each from the lower centre up) and takes lambda of the half-step
// conserved state: J_Con2Pri^T lambda_W (floors included), at the state F2 stored.  lambda_W never reaches memory.
// Only the 16^2 lines with both tangential coordinates in 3..18 carry face adjoints (the L face of a centre at normal
// coordinate 3..19, the R face at 2..18).  Bound by the workspace's traffic (860 MB for 512 patch groups, 174 us at the
// card's copy rate) and the stencils' chains: 380 us, where the phases one by one (x lines, y lines, z lines, conversion),
// with lambda_W through memory between them, took 288 + 157 + 157 + 150.  Two planes a workgroup: 64 patch groups 187 us
// for the whole adjoint against 199 with four; the recomputed z stencils cost nothing on 512 (383 against 377).
constexpr int R32_KS = 2, R32_NT = 512, R32_BPP = 20/R32_KS;
constexpr int R32_XY = 18*16, R32_Z = 16*16, R32_ZT = ( NV*R32_Z + R32_NT - 1 )/R32_NT;
static_assert( 20 % R32_KS == 0, "the blocks must tile the 20 half-step planes" );

template <int LIM>
__global__ void __launch_bounds__( R32_NT )
r32_kernel( double *__restrict__ g_ws, Prm<double> P0, double minmod_coeff )
{
   __shared__ double sX[3][NV][R32_XY], sY[3][NV][R32_XY], sZ[NV][R32_Z];      // x, y: [lower cell, centre, upper cell][v][stencil]
   const int tid = threadIdx.x, lb = (int)xcd_block(), pg = lb / R32_BPP, ka = 1 + ( lb % R32_BPP )*R32_KS, ke = ka + R32_KS;
   const Prm<double> P = phase_prm<double>( P0, minmod_coeff );
   const Prm<D1> PD = prm_as<D1>( P );
   double *ws = g_ws + (size_t)pg*WS_ADJ*N3;
   const double *H = ws + (size_t)WS_H*N3;
   Fwd<double> F( ws );
   Adj A( ws );
   double wm[R32_ZT], w0[R32_ZT], am[R32_ZT], a0[R32_ZT];
#  pragma unroll
   for (int t=0; t<R32_ZT; t++)
   {
      const int x = tid + t*R32_NT, v = x / R32_Z, ln = x - v*R32_Z, c = ( 3 + ln % 16 ) + NX*( 3 + ln / 16 );
      const int n = ( ka - 1 < 2 ) ? 2 : ka - 1;                               // first centre
      am[t] = a0[t] = wm[t] = w0[t] = 0.0;
      if ( x < NV*R32_Z ) { wm[t] = F.w( v, c + N2*( n - 1 ) );  w0[t] = F.w( v, c + N2*n ); }
   }
#  pragma unroll 1
   for (int n = ka - 1; n <= ke; n++)
   {
      const int q = n - 1;                                                     // plane that is completed
#     pragma unroll
      for (int t=0; t<R32_ZT; t++)
      {
         const int x = tid + t*R32_NT, v = x / R32_Z, ln = x - v*R32_Z;
         if ( x >= NV*R32_Z ) continue;
         double br = 0.0;
         if ( n >= 2 && n <= 19 )
         {
            const int c = ( 3 + ln % 16 ) + NX*( 3 + ln / 16 ) + N2*n, e = ln + 256*( n - 2 );
            const double wp = F.w( v, c + N2 );
            const double gl = ( n >= 3 )  ? A.lfc( 2, 0, v, e ) : 0.0;
            const double gr = ( n <= 18 ) ? A.lfc( 2, 1, v, e ) : 0.0;
            plm_face_rev<LIM>( wm[t], w0[t], wp, P.limiter, P.coeff, gl, gr, am[t], a0[t], br );
            wm[t] = w0[t];
            w0[t] = wp;
         }
         sZ[v][ln] = am[t];
         am[t] = a0[t];
         a0[t] = br;
      }
      if ( q >= ka && q >= 3 && q <= 18 )
         for (int x = tid; x < 2*NV*R32_XY; x += R32_NT)
         {
            const int d = x / ( NV*R32_XY ), y = x - d*NV*R32_XY, v = y / R32_XY, r = y - v*R32_XY;
            const int m = d ? 2 + r / 16 : 2 + r % 18;                         // centre along d
            const int i = d ? 3 + r % 16 : m, j = d ? m : 3 + r / 18, c = i + NX*j + N2*q, s = d ? NX : 1;
            const int e = d*2*NV*NLC + v*NLC + R32_XY*( q - 3 ) + r;
            const double gl = ( m >= 3 )  ? A.LFC[ e ] : 0.0;
            const double gr = ( m <= 18 ) ? A.LFC[ e + NV*NLC ] : 0.0;
            double bl = 0.0, bc = 0.0, br = 0.0;
            plm_face_rev<LIM>( F.w( v, c - s ), F.w( v, c ), F.w( v, c + s ), P.limiter, P.coeff, gl, gr, bl, bc, br );
            double *o = ( d ? &sY[0][0][0] : &sX[0][0][0] ) + v*R32_XY + r;
            o[0] = bl;  o[NV*R32_XY] = bc;  o[2*NV*R32_XY] = br;
         }
      __syncthreads();
      if ( q >= ka )
         for (int x = tid; x < 400; x += R32_NT)
         {
            const int i = 1 + x % 20, j = 1 + x / 20, c = i + NX*j + N2*q;
            const bool ci = in_rng( i, 3, 18 ), cj = in_rng( j, 3, 18 ), ck = in_rng( q, 3, 18 );
            double h[NV], lw[NV];
#           pragma unroll
            for (int v=0; v<NV; v++)
            {
               h[v] = H[ v*N3 + c ];
               double lx = 0.0, ly = 0.0;
               if ( cj && ck )
               {
                  const int r = 18*( j - 3 ) + i - 2;                          // stencil centred here
                  if ( i >= 3 )           lx += sX[2][v][r - 1];
                  if ( i >= 2 && i <= 19 ) lx += sX[1][v][r];
                  if ( i <= 18 )          lx += sX[0][v][r + 1];
               }
               if ( ci && ck )
               {
                  const int r = 16*( j - 2 ) + i - 3;
                  if ( j >= 3 )           ly += sY[2][v][r - 16];
                  if ( j >= 2 && j <= 19 ) ly += sY[1][v][r];
                  if ( j <= 18 )          ly += sY[0][v][r + 16];
               }
               lw[v] = lx + ly;
               if ( ci && cj ) lw[v] += sZ[v][ 16*( j - 3 ) + i - 3 ];
            }
            for (int u=0; u<NV; u++)
            {
               D1 hd[NV], w[NV];
#              pragma unroll
               for (int v=0; v<NV; v++) { hd[v] = D1( h[v] );  hd[v].d[0] = ( u == v ) ? 1.0 : 0.0; }
               con2pri_floor( hd, PD, w );
               double g = 0.0;
#              pragma unroll
               for (int v=0; v<NV; v++) g = fmad( lw[v], w[v].d[0], g );
               A.lu( u, c ) = g;
            }
         }
      __syncthreads();
   }
}

// R1 + R0: a workgroup takes JR rows (y) of about 22/KB planes (z), plane by plane.  R1: lambda_Fh = dt/(2dh)
// (lambda_U(c+e_d) - lambda_U(c)) of every half-step face, then J_RS^T per side; the side contributions of the plane's x
// and y faces and of the z face above it (normal k) stay in LDS.  R0: lambda_in of the plane's cells = lambda_out (output
// cells) + lambda_U_half (half-step cells) + the face contributions in the order x low, x high, y low, y high, z low, z high,
// the last one from the plane before (solved first for the first plane).  Faces between workgroups are solved by both.
// 3 waves per SIMD (<= 170 VGPRs); Roe's reverse solve needs about 230, 2 waves.  512 patch groups 514 us; one whole plane of
// 768 lanes, with the z faces' high sides added by a kernel of their own through memory, 525 + 95.  192 lanes against 256
// (610) and 128 (608); Roe 128 lanes against 256: 1724 and 1917 us for the whole adjoint.  Calls of few patch groups take
// blocks of one plane (few_blocks()).
template <int JR_, int KB_>
struct R10
{
   static constexpr int JR = JR_, KB = KB_, RB = 20/JR, BPP = RB*KB;
   static constexpr int NXF = 21*JR, NYF = 20*( JR + 1 ), NZF = 20*JR;
   static constexpr bool ONE = ( KB == NX );            // one plane: the z faces below it come with its own
   static constexpr int nt( int rs ) { return ( rs == 2 && !ONE ) ? 128 : 192; }
   static_assert( 20 % JR == 0, "the blocks must tile the 20 half-step rows" );
};
typedef R10<5, 4>  R10Large;
typedef R10<5, NX> R10Small;

template <int RS, typename B>
__global__ void __launch_bounds__( B::nt( RS ) )
r10_kernel( const double *__restrict__ g_in, const double *__restrict__ g_lout, double *__restrict__ g_lin,
            double *__restrict__ g_ws, Prm<double> P0, double minmod_coeff )
{
   constexpr int R10_NT = B::nt( RS );
   constexpr bool ONE = B::ONE;
   // [low/high side][v][face]; sZh [k % 2][v][face]: the z faces' high sides, read one plane later
   __shared__ double sX[2][NV][B::NXF], sY[2][NV][B::NYF], sZ[NV][B::NZF], sZh[2][NV][B::NZF];
   const int tid = threadIdx.x, lb = (int)xcd_block(), rb = lb % B::RB, kb = ( lb / B::RB ) % B::KB, pg = lb / B::BPP;
   const int j0 = rb*B::JR, ka = 22*kb/B::KB, ke = 22*( kb + 1 )/B::KB;      // half-step rows j0 + 1 .. j0 + JR, planes [ka, ke)
   const int ja = ( rb == 0 ) ? 0 : j0 + 1, je = ( rb == B::RB - 1 ) ? NX : j0 + B::JR + 1;      // rows of lambda_in [ja, je)
   const Prm<double> P = phase_prm<double>( P0, minmod_coeff );
   const double *in = g_in + pg*NIN, *lout = g_lout + pg*NOUT;
   double *lin = g_lin + pg*NIN;
   Adj A( g_ws + (size_t)pg*WS_ADJ*N3 );
#  pragma unroll 1
   for (int k = ( !ONE && ka > 0 ) ? ka - 1 : ka; k < ke; k++)
   {
      // faces with low cell in plane k: x (normal i = 0..20), y (normal j0 .. j0 + JR), z; plane 0 and the plane
      // before the first have only their z faces, plane 21 none (ONE: and those with low cell in plane k - 1)
      const int nxy = B::NXF + B::NYF;
      const int f0 = ( k == 0 || k < ka ) ? nxy : ( ONE && k == NX - 1 ) ? nxy + B::NZF : 0;
      const int f1 = ( ONE && k > 0 ) ? nxy + 2*B::NZF : ( k <= 20 ) ? nxy + B::NZF : 0;
      for (int f = f0 + tid; f < f1; f += R10_NT)
      {
         int d, i, j, kf = k, r = f, n;
         if ( f < B::NXF )                 { d = 0;  i = r % 21;  j = j0 + 1 + r / 21;  n = i; }
         else if ( f < B::NXF + B::NYF )  { d = 1;  r = f - B::NXF;  i = 1 + r % 20;  j = j0 + r / 20;  n = j; }
         else
         {
            d = 2;  r = f - nxy;
            if ( ONE && r >= B::NZF ) { r -= B::NZF;  kf = k - 1; }
            i = 1 + r % 20;  j = j0 + 1 + r / 20;  n = kf;
         }
         const int c = i + NX*j + N2*kf, s = ( d == 0 ? 1 : d == 1 ? NX : N2 );
         const bool lo = in_rng( n, 1, 20 ), hi = in_rng( n + 1, 1, 20 );   // tangential range is 1..20 already
         double lf[NV];
#        pragma unroll
         for (int v=0; v<NV; v++) lf[v] = P.dt_dh2*( ( hi ? A.lu( v, c + s ) : 0.0 ) - ( lo ? A.lu( v, c ) : 0.0 ) );
         double uL[NV], uR[NV];
#        pragma unroll
         for (int v=0; v<NV; v++) { uL[v] = in[ v*N3 + c ];  uR[v] = in[ v*N3 + c + s ]; }
         double gl[NV] = { 0.0, 0.0, 0.0, 0.0, 0.0 }, gr[NV] = { 0.0, 0.0, 0.0, 0.0, 0.0 };
         half_flux_rev<RS>( d, uL, uR, P, lf, gl, gr );
         double *pl = ( d == 0 ) ? &sX[0][0][r] : ( d == 1 ) ? &sY[0][0][r] : &sZ[0][r];
         double *ph = ( d == 0 ) ? &sX[1][0][r] : ( d == 1 ) ? &sY[1][0][r] : &sZh[kf & 1][0][r];
         const int m = ( d == 0 ) ? B::NXF : ( d == 1 ) ? B::NYF : B::NZF;
#        pragma unroll
         for (int v=0; v<NV; v++)
         {
            if ( !ONE || kf == k ) pl[ v*m ] = gl[v];
            ph[ v*m ] = gr[v];
         }
      }
      __syncthreads();
      if ( k >= ka )
      for (int e = ja*NX + tid; e < je*NX; e += R10_NT)
      {
         const int i = e % NX, j = e / NX, c = i + NX*j + N2*k;
         const bool core = core3( i, j, k ), half = in_rng( i, 1, 20 ) && in_rng( j, 1, 20 ) && in_rng( k, 1, 20 );
         const bool xl = half_face( i, j, k ), xh = half_face( i - 1, j, k ), yl = half_face( j, i, k ),
                    yh = half_face( j - 1, i, k ), zl = half_face( k, i, j ), zh = half_face( k - 1, i, j );
         const int rx = i + 21*( j - j0 - 1 ), ry = ( i - 1 ) + 20*( j - j0 ), rz = ( i - 1 ) + 20*( j - j0 - 1 );
#        pragma unroll
         for (int v=0; v<NV; v++)
         {
            double acc = core ? lout[ (size_t)v*PS*PS*PS + out_index( i, j, k ) ] : 0.0;
            if ( half ) acc += A.lu( v, c );
            if ( xl ) acc += sX[0][v][rx];
            if ( xh ) acc += sX[1][v][rx - 1];
            if ( yl ) acc += sY[0][v][ry];
            if ( yh ) acc += sY[1][v][ry - 20];
            if ( zl ) acc += sZ[v][rz];
            if ( zh ) acc += sZh[( k - 1 ) & 1][v][rz];
            lin[ v*N3 + c ] = acc;
         }
      }
      __syncthreads();
   }
}

// ---------------- transpose of the periodic ghost-zone preparation ----------------
// level_lam[v][z][y][x] = sum over every patch-group input element that copies level cell (x,y,z)
// (gather form: each level cell collects its copies, so there is one writer per element)
// The window copies of level coordinate x along one axis of G patch groups: its own patch group's, and one more within
// `ghost` (<= 8) cells of a patch-group face, in the neighbour across that face (the same patch group if G == 1), in
// ascending order of the patch groups q-1, q, q+1 and, within one, of the index.
__device__ __forceinline__ int copies( int x, int G, int ghost, int pl[2], int il[2] )
{
   const int q = x/PS, r = x - q*PS;
   pl[0] = pl[1] = q;
   il[0] = il[1] = r + ghost;
   const bool lo = r < ghost, hi = r >= PS - ghost;
   if ( !lo && !hi ) return 1;
   const int p = lo ? ( q > 0 ? q - 1 : G - 1 ) : ( q < G - 1 ? q + 1 : 0 ), i = lo ? r + PS + ghost : r - PS + ghost;
   const int k = ( G == 1 ) ? ( lo ? 1 : 0 ) : ( lo || G == 2 ) ? 0 : 1;      // place of the neighbour's copy
   pl[k] = p;
   il[k] = i;
   return 2;
}

// one level cell per lane, a row of cells per (y, z, field), neighbouring rows on one XCD: at most 8 copies, most cells
// have one.  Element index divisions and a search over candidate patch groups took 34 us for 64 FP64 patch groups and
// 397 us for 960 FP32 ones, this takes 12.9 and 133 us; lanes over 16 x 16 cells took 16 and 134 us.  THIN, for rows of less than
// 64 cells and for few rows: lx lanes a row, and the rows in xs pieces (1 x 1 x 32 patch groups with ghost 8 22 -> 9.8 us, 32 x 1
// x 1 FP64 27 -> 12; as run-time values for all levels they cost 5 to 15% of the others).
template <typename IO, bool THIN>
__global__ void __launch_bounds__( 256 )
prepare_adjoint_kernel( const IO *__restrict__ pg_lam, IO *__restrict__ lam, int nx, int ny, int nz, int ghost, long rows, int lx_, int xs_ )
{
   const int lx = THIN ? lx_ : 64, xs = THIN ? xs_ : 1;
   const int n = PS + 2*ghost, n3 = n*n*n, gx = nx/PS, gy = ny/PS;
   const int tx = threadIdx.x & ( lx - 1 ), lr = (unsigned)threadIdx.x / (unsigned)lx, nr = 256 / lx;      // lx cells of nr rows per pass
   const long lb = xcd_block(), rb = THIN ? lb / xs : lb;
   const int  xc = THIN ? (int)( lb - rb*xs )*lx : 0;
   for (long row = rb*nr + lr; row < rows; row += (long)( gridDim.x/xs )*nr)
   {
      const int  y = (int)( row % ny );
      const long vz = row / ny;
      const int  z = (int)( vz % nz ), v = (int)( vz / nz );
      int py[2], iy[2], pz[2], iz[2];
      const int my = copies( y, gy, ghost, py, iy ), mz = copies( z, nz/PS, ghost, pz, iz );
      for (int x = xc + tx; x < nx; x += lx*xs)
      {
         int px[2], ix[2];
         const int mx = copies( x, gx, ghost, px, ix );
         double acc = 0.0;
         for (int c=0; c<mz; c++)
            for (int b=0; b<my; b++)
            {
               const IO *w = pg_lam + iy[b]*n + iz[c]*n*n + (size_t)v*n3;
               const size_t pr = ( (size_t)pz[c]*gy + py[b] )*gx;
               acc += (double)w[ ( pr + px[0] )*NV*n3 + ix[0] ];
               if ( mx > 1 ) acc += (double)w[ ( pr + px[1] )*NV*n3 + ix[1] ];
            }
         lam[ row*nx + x ] = (IO)acc;
      }
   }
}

} // namespace

size_t adjoint_workspace_bytes( int npg ) { return (size_t)( npg > 0 ? npg : 0 )*WS_ADJ*N3*sizeof( double ); }

namespace {

// one flat grid of bpp(count) workgroups per patch group
void phase_grid( int npg, int count, dim3 &grid ) { grid = dim3( (unsigned)( (long)npg*bpp( count ) ) ); }
// whether every phase's grid of npg patch groups fits one launch (R4 has the most lanes)
bool grids_fit( int npg ) { return (long)npg*bpp( N_R4 )*NT < ( 1L << 32 ); }
static_assert( F12Large::BPP*F12_NT <= bpp( N_R4 )*NT && R10Large::BPP*R10Large::nt( 4 ) <= bpp( N_R4 )*NT && R32_BPP*R32_NT <= bpp( N_R4 )*NT,
               "R4 has the most lanes" );

// Whether a phase of `blocks` marching workgroups leaves the chip idle, most of them per compute unit
bool few_blocks( long blocks, double most ) { return (double)blocks <= most*device_cus(); }

// The marching blocks for calls that fill the chip with them, blocks of one plane for those that do not: a march of four to
// six planes takes its time however few patch groups there are.  us of the whole call, marching -> one plane, adjoint HLLC 1
// patch group 84 -> 45, 16 97 -> 70, 64 183 -> 171, 128 372 -> 360, 256 702 -> 711; Roe 8 121 -> 62, 48 207 -> 192, 64 249
// -> 257 (its blocks of one plane alone 263), 128 480 -> 530; tangent HLLC 4 38 -> 21, 64 126 -> 120, 96 175 -> 182; Roe 4 60 -> 27, 64 218 -> 209,
// 96 310 -> 317.  So the lines: 2.5 marching blocks of F1 + F2 per compute unit, of R1 + R0 eight, with Roe three.
template <int RS, typename T>
void launch_f12( const double *in, const double *tin, double *ws, int h_off, int npg, double minmod_coeff, const Prm<double> &P, hipStream_t stream )
{
#  define GA_F12( B ) hipLaunchKernelGGL( ( f12_kernel<RS, T, B> ), dim3( (unsigned)( B::BPP*npg ) ), dim3( F12_NT ), 0, stream, in, tin, ws, h_off, P, minmod_coeff )
   if ( few_blocks( (long)F12Large::BPP*npg, 2.5 ) ) GA_F12( F12Small ); else GA_F12( F12Large );
#  undef GA_F12
}

template <int RS>
void launch_r10( const double *in, const double *lam_out, double *lam_in, double *ws, int npg, double minmod_coeff, const Prm<double> &P, hipStream_t stream )
{
#  define GA_R10( B ) hipLaunchKernelGGL( ( r10_kernel<RS, B> ), dim3( (unsigned)( B::BPP*npg ) ), dim3( B::nt( RS ) ), 0, stream, in, lam_out, lam_in, ws, P, minmod_coeff )
   if ( few_blocks( (long)R10Large::BPP*npg, RS == 2 ? 3.0 : 8.0 ) ) GA_R10( R10Small ); else GA_R10( R10Large );
#  undef GA_R10
}

template <int RS, int LIM>
int adjoint_phases( const double *in, const double *lam_out, double *lam_in, double *ws, int npg, double minmod_coeff,
                    const Prm<double> &P, hipStream_t stream )
{
   const dim3 block( NT );
   dim3 g;
   // forward: F1 + F2 (the PLM faces are recomputed where they are needed instead of stored)
   if ( !grids_fit( npg ) ) return -3;
   launch_f12<RS, double>( in, nullptr, ws, WS_H, npg, minmod_coeff, P, stream );
   // reverse: R4, R3 + R2, R1 + R0
   phase_grid( npg, N_R4, g );
   hipLaunchKernelGGL( ( r4_kernel<RS, LIM> ), g, block, 0, stream, lam_out, ws, P, minmod_coeff );
   hipLaunchKernelGGL( ( r32_kernel<LIM> ), dim3( (unsigned)( npg*R32_BPP ) ), dim3( R32_NT ), 0, stream, ws, P, minmod_coeff );
   launch_r10<RS>( in, lam_out, lam_in, ws, npg, minmod_coeff, P, stream );
   return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
}

template <int RS, int LIM, typename T>
int tangent_phases( const double *in, const double *tin, double *out, double *tout, double *ws, int npg,
                    double minmod_coeff, const Prm<double> &P, hipStream_t stream )
{
   const dim3 block( NT );
   dim3 g;
   if ( !grids_fit( npg ) ) return -3;
   launch_f12<RS, T>( in, tin, ws, -1, npg, minmod_coeff, P, stream );
   phase_grid( npg, 3*NFF, g );
   hipLaunchKernelGGL( ( f4_face_kernel<RS, LIM, T> ), g, block, 0, stream, ws, P, minmod_coeff );
   phase_grid( npg, N_F4, g );
   hipLaunchKernelGGL( ( f4_update_kernel<T> ), g, block, 0, stream, in, tin, out, tout, ws, P, minmod_coeff );
   return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
}

} // namespace

int launch_mhm_rp_adjoint( const double *in, const double *lam_out, double *lam_in, double *ws, int npg, int rsolver,
                           double minmod_coeff, const Prm<double> &P, hipStream_t stream )
{
   if ( npg <= 0 ) return 0;
   const bool l4 = ( kernel_limiter( P.limiter, minmod_coeff ) == 4 );
#  define GA_ADJ( RS_ ) ( l4 ? adjoint_phases<RS_, 4>( in, lam_out, lam_in, ws, npg, minmod_coeff, P, stream ) \
                             : adjoint_phases<RS_, 0>( in, lam_out, lam_in, ws, npg, minmod_coeff, P, stream ) )
   switch ( rsolver )
   {
      case 4: return GA_ADJ( 4 );
      case 3: return GA_ADJ( 3 );
      case 2: return GA_ADJ( 2 );
      default: return -1;
   }
#  undef GA_ADJ
}

int launch_mhm_rp_tangent( const double *in, const double *tin, double *out, double *tout, double *ws, int npg,
                           int rsolver, double minmod_coeff, const Prm<double> &P, hipStream_t stream )
{
   if ( npg <= 0 ) return 0;
   const bool l4 = ( kernel_limiter( P.limiter, minmod_coeff ) == 4 ), tl = ( tin != nullptr );
#  define GA_TAN( RS_, T_ ) ( l4 ? tangent_phases<RS_, 4, T_>( in, tin, out, tout, ws, npg, minmod_coeff, P, stream ) \
                                 : tangent_phases<RS_, 0, T_>( in, tin, out, tout, ws, npg, minmod_coeff, P, stream ) )
   switch ( rsolver )
   {
      case 4: return tl ? GA_TAN( 4, D1 ) : GA_TAN( 4, double );
      case 3: return tl ? GA_TAN( 3, D1 ) : GA_TAN( 3, double );
      case 2: return tl ? GA_TAN( 2, D1 ) : GA_TAN( 2, double );
      default: return -1;
   }
#  undef GA_TAN
}

template <typename IO>
int launch_prepare_adjoint( const IO *pg_lam, IO *lam, int nx, int ny, int nz, int ghost, hipStream_t stream )
{
   const long rows = (long)NV*ny*nz;
   if ( rows <= 0 || nx <= 0 ) return 0;
   const int  lx = ( nx < 32 ) ? 16 : ( nx < 64 ) ? 32 : 64, nr = 256/lx;
   const long b = ( rows + nr - 1 )/nr, blocks = b < 65536 ? b : 65536;
   int xs = 1;
   while ( xs*lx < nx && blocks*xs < 4L*device_cus() ) xs *= 2;
   if ( lx < 64 || xs > 1 ) hipLaunchKernelGGL( ( prepare_adjoint_kernel<IO, true> ), dim3( (unsigned)( blocks*xs ) ), dim3( 256 ), 0, stream, pg_lam, lam,
                                                nx, ny, nz, ghost, rows, lx, xs );
   else hipLaunchKernelGGL( ( prepare_adjoint_kernel<IO, false> ), dim3( (unsigned)blocks ), dim3( 256 ), 0, stream, pg_lam, lam, nx, ny, nz, ghost,
                            rows, lx, xs );
   return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
}

template int launch_prepare_adjoint<double>( const double*, double*, int, int, int, int, hipStream_t );
template int launch_prepare_adjoint<float> ( const float*,  float*,  int, int, int, int, hipStream_t );

} // namespace gamer_amd

// Kernels around the patch-group solver: the hydro CFL time step, ghost-zone preparation of patch-group inputs
// from a periodic uniform level, and the scatter of patch-group outputs back to that level.
//
//   dt_cfl_kernel       CPU_dtSolver_HydroCFL / CUFLU_dtSolver_HydroCFL (src/Model_Hydro/CPU_Hydro/
//                       CPU_dtSolver_HydroCFL.cpp:57-209): per 8^3 patch, dt = Safety*dh / max_cells max_d(|v_d|+c_s),
//                       block max-reduction with wave64 shuffles (the reference's CUUTI_BlockReduction_Shuffle
//                       assumes 32-lane warps).
//   gather_pg_kernel    the same-level, periodic case of Prepare_PatchData for the fluid solver
//                       (src/Fluid/Flu_Prepare.cpp:91-94, src/Main/Prepare_PatchData.cpp:166): 16^3 interior +
//                       ghost zones, layout [PG][var][N^3].
//   scatter_pg_kernel   the copy-back of Flu_Close (src/Fluid/Flu_Close.cpp:133-217) into the level array.
// The level array is [var][Z][Y][X], x fastest; patch groups are numbered x fastest, then y, then z.

#include "hydro_math.hpp"
#include "hydro_kernels.hpp"

namespace gamer_amd {

namespace {

constexpr int PS = 16;

__device__ __forceinline__ float  wave_max( float v )
{
#  pragma unroll
   for (int o = 32; o > 0; o >>= 1) v = vmax( v, __shfl_xor( v, o, 64 ) );
   return v;
}
__device__ __forceinline__ double wave_max( double v )
{
#  pragma unroll
   for (int o = 32; o > 0; o >>= 1) v = vmax( v, __shfl_xor( v, o, 64 ) );
   return v;
}

template <typename IO>
__global__ void __launch_bounds__( 256 )
dt_cfl_kernel( const IO *__restrict__ in, IO *__restrict__ dt, int npatch, double dh_safety, double gamma,
               double min_pres )
{
   __shared__ IO red[4];
   const int p = blockIdx.x, tid = threadIdx.x;
   if ( p >= npatch ) return;
   const IO *u0 = in + (size_t)p*NV*512;
   IO m = (IO)0;
#  pragma unroll
   for (int k=0; k<2; k++)
   {
      const int c = tid + 256*k;
      IO u[NV];
#     pragma unroll
      for (int v=0; v<NV; v++) u[v] = u0[ v*512 + c ];
      m = vmax( m, cell_cfl( u, gamma, gamma - 1.0, min_pres ) );
   }
   m = wave_max( m );
   if ( ( tid & 63 ) == 0 ) red[tid >> 6] = m;
   __syncthreads();
   if ( tid == 0 ) dt[p] = (IO)( dh_safety / (double)vmax( vmax( red[0], red[1] ), vmax( red[2], red[3] ) ) );
}

template <typename IO> struct Vec4;
template <> struct Vec4<float>  { typedef float  type __attribute__(( ext_vector_type( 4 ) )); };
template <> struct Vec4<double> { typedef double type __attribute__(( ext_vector_type( 4 ) )); };

// Patch-group inputs from the periodic level: block (patch group, field, GATHER_N cells of the window in linear order), a
// thread copies the cells t, t + 512, ...: every load and store instruction then covers 64 consecutive cells, whose rows
// are rows of the level.  (x, y, z) of a cell come from a float reciprocal: after the +0.5 shift, e/N^2 and r/N sit at
// least 1/(2 N^2) away from an integer, far above the float error for N <= 32; the wrap is one conditional add, as
// ghost <= 8 < nx.  Patch groups next to each other in x share cache lines of the level, so the blocks are laid out
// XCD-major, patch group fastest (xcd_block).  Bound by memory: 283 MB for 960 FP32 patch groups take 58 us at the card's
// copy rate.  One element per lane with 64-bit index divisions took 287 us (64 FP64 patch groups 25.6 us), four
// consecutive cells per lane with a vector store 110, 11 cells in flight per lane 98 to 121, this takes 90 (10.7); on 512
// FP64 patch groups with ghost 2 the XCD-major layout takes 48 us in place of 66, the first form 130.
constexpr int GATHER_NT = 512, GATHER_Q = 11, GATHER_N = GATHER_NT*GATHER_Q;
template <typename IO>
__global__ void __launch_bounds__( GATHER_NT )
gather_pg_kernel( const IO *__restrict__ grid, IO *__restrict__ pg_in, int nx, int ny, int nz, int ghost )
{
   const int n = PS + 2*ghost, n2 = n*n, n3 = n2*n;
   const long lb = xcd_block();
   const unsigned pg = (unsigned)( lb % gridDim.x ), lv = (unsigned)( lb / gridDim.x ), v = lv % NV, bz = lv / NV;
   const unsigned gx = nx/PS, gy = ny/PS, row = pg / gx;
   const int x0 = (int)( pg - row*gx )*PS - ghost, y0 = (int)( row % gy )*PS - ghost, z0 = (int)( row / gy )*PS - ghost;
   const float rn = 1.0f/(float)n, rn2 = 1.0f/(float)n2;
   const IO *src = grid + (size_t)v*nz*ny*nx;
   IO *dst = pg_in + ( (size_t)pg*NV + v )*n3;
   IO val[GATHER_Q];
#  pragma unroll
   for (int q=0; q<GATHER_Q; q++)
   {
      const int e = (int)bz*GATHER_N + q*GATHER_NT + (int)threadIdx.x;
      if ( e >= n3 ) continue;
      const int k = (int)( ( (float)e + 0.5f )*rn2 ), r = e - k*n2, j = (int)( ( (float)r + 0.5f )*rn ), i = r - j*n;
      int x = x0 + i, y = y0 + j, z = z0 + k;
      x += ( x < 0 ) ? nx : ( x >= nx ) ? -nx : 0;
      y += ( y < 0 ) ? ny : ( y >= ny ) ? -ny : 0;
      z += ( z < 0 ) ? nz : ( z >= nz ) ? -nz : 0;
      val[q] = src[ ( (size_t)z*ny + y )*nx + x ];
   }
#  pragma unroll
   for (int q=0; q<GATHER_Q; q++)
   {
      const int e = (int)bz*GATHER_N + q*GATHER_NT + (int)threadIdx.x;
      if ( e < n3 ) dst[e] = val[q];
   }
}

// Patch-group outputs into the level: block (patch group, field, 4 planes), a thread moves 4 consecutive cells of a row
// (nx is a multiple of 16), as one vector where both sides are aligned.  158 MB for 960 FP32 patch groups; one element
// per lane with 64-bit index divisions took 66 us, this takes 24.
template <typename IO>
__global__ void __launch_bounds__( 256 )
scatter_pg_kernel( const IO *__restrict__ pg_out, IO *__restrict__ grid, int nx, int ny, int nz, bool vec )
{
   const unsigned pg = blockIdx.x, gx = nx/PS, gy = ny/PS, row = pg / gx;
   const int x0 = (int)( pg - row*gx )*PS, y0 = (int)( row % gy )*PS, z0 = (int)( row / gy )*PS;
   const int v = blockIdx.y >> 2, t = threadIdx.x;
   const int i = 4*( t & 3 ), j = ( t >> 2 ) & 15, k = 4*( blockIdx.y & 3 ) + ( t >> 6 );
   const IO *src = pg_out + ( (size_t)pg*NV + v )*PS*PS*PS + ( k*PS + j )*PS + i;
   IO *dst = grid + ( ( (size_t)v*nz + z0 + k )*ny + y0 + j )*nx + x0 + i;
   typedef typename Vec4<IO>::type V4;
   if ( vec ) *reinterpret_cast<V4*>( dst ) = *reinterpret_cast<const V4*>( src );
   else
#     pragma unroll
      for (int q=0; q<4; q++) dst[q] = src[q];
}

__global__ void reset_counter_kernel( unsigned *c ) { if ( threadIdx.x == 0 ) *c = 0u; }

template <typename IO> bool vec4_aligned( const void *p ) { return reinterpret_cast<size_t>( p ) % ( 4*sizeof( IO ) ) == 0; }

} // namespace

template <typename IO>
int launch_dt_cfl( const IO *in, IO *dt, int npatch, double dh, double safety, double gamma, double min_pres,
                   hipStream_t stream )
{
   if ( npatch <= 0 ) return 0;
   hipLaunchKernelGGL( dt_cfl_kernel<IO>, dim3( npatch ), dim3( 256 ), 0, stream, in, dt, npatch, safety*dh, gamma, min_pres );
   return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
}

template <typename IO>
int launch_gather( const IO *grid, IO *pg_in, int nx, int ny, int nz, int ghost, hipStream_t stream )
{
   const long npg = (long)( nx/PS )*( ny/PS )*( nz/PS ), n = PS + 2*ghost;
   if ( npg <= 0 ) return 0;
   hipLaunchKernelGGL( gather_pg_kernel<IO>, dim3( (unsigned)npg, NV, (unsigned)( ( n*n*n + GATHER_N - 1 )/GATHER_N ) ), dim3( GATHER_NT ), 0, stream,
                       grid, pg_in, nx, ny, nz, ghost );
   return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
}

template <typename IO>
int launch_scatter( const IO *pg_out, IO *grid, int nx, int ny, int nz, hipStream_t stream )
{
   const long npg = (long)( nx/PS )*( ny/PS )*( nz/PS );
   if ( npg <= 0 ) return 0;
   hipLaunchKernelGGL( scatter_pg_kernel<IO>, dim3( (unsigned)npg, NV*4 ), dim3( 256 ), 0, stream, pg_out, grid, nx, ny, nz,
                       vec4_aligned<IO>( pg_out ) && vec4_aligned<IO>( grid ) );
   return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
}

int launch_reset_counter( unsigned *counter, hipStream_t stream )
{
   hipLaunchKernelGGL( reset_counter_kernel, dim3( 1 ), dim3( 64 ), 0, stream, counter );
   return ( hipGetLastError() == hipSuccess ) ? 0 : -2;
}

template int launch_dt_cfl<double>( const double*, double*, int, double, double, double, double, hipStream_t );
template int launch_dt_cfl<float> ( const float*,  float*,  int, double, double, double, double, hipStream_t );
template int launch_gather<double>( const double*, double*, int, int, int, int, hipStream_t );
template int launch_gather<float> ( const float*,  float*,  int, int, int, int, hipStream_t );
template int launch_scatter<double>( const double*, double*, int, int, int, hipStream_t );
template int launch_scatter<float> ( const float*,  float*,  int, int, int, hipStream_t );

} // namespace gamer_amd

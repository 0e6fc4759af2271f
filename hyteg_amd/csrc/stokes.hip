// P2-P1 Taylor-Hood Stokes operator with the blended, variable-viscosity
// full-viscous velocity block (P2P1ElementwiseBlendingFullViscousStokesOperator,
// P2P1ElementwiseBlendingStokesOperator.hpp:125-216): host set-up, HIP kernels
// and C-ABI entry points.
//
// One tiled kernel evaluates any combination of the three blocks of
//   [ A  B^T ] [u]
//   [ B   0  ] [p]
// per micro-cell: A = 2 eta eps(u):eps(v) - 2/3 eta div u div v with the
// 5-point degree-3 rule (p2_full_stokesvar_*_blending_q3), B = -(q, div u) and
// B^T with the 4-point degree-2 rule (p2_to_p1_div_blending_q2,
// p1_to_p2_divt_blending_q2); eta = exp(c0 + c1 |F(x)|) at the blended points.
// The element matrices are never formed: per quadrature point the velocity
// gradient is built from the 30 element values, turned into the stress and
// tested against the 30 basis gradients, the same sums the reference's 9 + 6
// sub-operators form one block at a time.
//
// The shell map is used in rank-one form, DF = q I + x w^T, beta = q + w.x:
// DF^-T v = (v - w (x.v)/beta)/q, DF^-1 s = (s - x (w.s)/beta)/q and
// |det DF| = q^2 |beta|, so the powers of q cancel in the viscous block and one
// power remains in the divergence blocks.
#include <array>
#include <type_traits>
#include <cmath>
#include <mutex>

#include "abi_util.hpp"
#include "halo.hpp"
#include "hyteg_amd.h"
#include "p2tile.hpp"
#include "runtime.hpp"

namespace hg {

namespace {
// Stokes quadrature: points 0..4 are the degree-3 rule of the viscous block
// (centroid with weight -2/15, then the points with barycentric coordinate 1/2
// at vertex 3, 2, 1, 0 with weight 3/40), points 5..8 the degree-2 rule of the
// divergence blocks ((a,a,a,b) permutations, weight 1/24)
__constant__ double cSQ4[9][4];  // 4 lam_k
__constant__ double cSQ4m[9][4]; // 4 lam_k - 1
__constant__ double cSQL[9][4];  // lam_k
__constant__ double cSQW[9];

constexpr double kQa = 0.1381966011250105, kQb = 0.5854101966249685;
const double     kSQP[9][4] = { { 0.25, 0.25, 0.25, 0.25 },
                                { 1.0 / 6.0, 1.0 / 6.0, 1.0 / 6.0, 0.5 },
                                { 1.0 / 6.0, 1.0 / 6.0, 0.5, 1.0 / 6.0 },
                                { 1.0 / 6.0, 0.5, 1.0 / 6.0, 1.0 / 6.0 },
                                { 0.5, 1.0 / 6.0, 1.0 / 6.0, 1.0 / 6.0 },
                                { kQa, kQa, kQa, kQb },
                                { kQa, kQa, kQb, kQa },
                                { kQa, kQb, kQa, kQa },
                                { kQb, kQa, kQa, kQa } };
const double     kSQW[9]    = { -2.0 / 15.0, 3.0 / 40.0, 3.0 / 40.0,  3.0 / 40.0, 3.0 / 40.0,
                                1.0 / 24.0,  1.0 / 24.0, 1.0 / 24.0,  1.0 / 24.0 };

constexpr int kPBox  = kTile + 1; // pressure box: the tile's level-L vertices
constexpr int kPBox3 = kPBox * kPBox * kPBox;

// FP32 copies of the quadrature tables for the reduced-precision velocity block
__constant__ float cSQ4f[9][4];
__constant__ float cSQ4mf[9][4];
__constant__ float cSQLf[9][4];
__constant__ float cSQWf[9];

template < class R >
struct SQ;
template <>
struct SQ< double >
{
   static __device__ __forceinline__ const double* a4( int q ) { return cSQ4[q]; }
   static __device__ __forceinline__ const double* b4( int q ) { return cSQ4m[q]; }
   static __device__ __forceinline__ const double* lam( int q ) { return cSQL[q]; }
   static __device__ __forceinline__ double        w( int q ) { return cSQW[q]; }
};
template <>
struct SQ< float >
{
   static __device__ __forceinline__ const float* a4( int q ) { return cSQ4f[q]; }
   static __device__ __forceinline__ const float* b4( int q ) { return cSQ4mf[q]; }
   static __device__ __forceinline__ const float* lam( int q ) { return cSQLf[q]; }
   static __device__ __forceinline__ float        w( int q ) { return cSQWf[q]; }
};

__device__ __forceinline__ double rexp( double v ) { return exp( v ); }
__device__ __forceinline__ float  rexp( float v ) { return expf( v ); }

// barycentric derivatives g_k = sum_j u_j dphi_j / dlam_k of a P2 function
template < class R >
__device__ __forceinline__ void baryGrad( const R* a4, const R* b4, const R u[10], R g[4] )
{
   g[0] = b4[0] * u[0] + a4[1] * u[4] + a4[2] * u[5] + a4[3] * u[6];
   g[1] = b4[1] * u[1] + a4[0] * u[4] + a4[2] * u[7] + a4[3] * u[8];
   g[2] = b4[2] * u[2] + a4[0] * u[5] + a4[1] * u[7] + a4[3] * u[9];
   g[3] = b4[3] * u[3] + a4[0] * u[6] + a4[1] * u[8] + a4[2] * u[9];
}

// y_j += grad phi_j . tau for the 10 P2 functions; e_k = grad lam_k . tau, k = 1..3
template < class R >
__device__ __forceinline__ void testGrad( const R* a4, const R* b4, R e1, R e2, R e3, R y[10] )
{
   const R e0 = -( e1 + e2 + e3 );
   y[0] += b4[0] * e0;
   y[1] += b4[1] * e1;
   y[2] += b4[2] * e2;
   y[3] += b4[3] * e3;
   y[4] += a4[1] * e0 + a4[0] * e1;
   y[5] += a4[2] * e0 + a4[0] * e2;
   y[6] += a4[3] * e0 + a4[0] * e3;
   y[7] += a4[2] * e1 + a4[1] * e2;
   y[8] += a4[3] * e1 + a4[1] * e3;
   y[9] += a4[3] * e2 + a4[2] * e3;
}

// With T = q DF^-T the gradient of component c is G_c = T D^T (g_k - g_0); M = T D^T
// (3 x 3, M[d][k - 1] = d-th component of T grad lam_k) serves all three components and,
// transposed, their test functions: T = I - w x^T / beta, a rank-one correction of D^T.
template < class R >
__device__ __forceinline__ void mapGradients( const R* Dc, const R x[3], const R w[3], R ib, R M[3][3] )
{
#pragma unroll
   for ( int k = 0; k < 3; ++k )
   {
      const R z = ib * ( x[0] * Dc[3 * k] + x[1] * Dc[3 * k + 1] + x[2] * Dc[3 * k + 2] );
#pragma unroll
      for ( int d = 0; d < 3; ++d )
         M[d][k] = Dc[3 * k + d] - w[d] * z;
   }
}

// quadrature point q of the thread's micro-cell: computational point x, the
// shell scalars (q = 1, w = 0, beta = 1 without blending), 1/beta and |F(x)|
template < class R >
struct QPoint
{
   R x[3], qq, w[3], beta, ib, r;
};

template < class R >
__device__ __forceinline__ QPoint< R > qpoint( const P2CellGeomT< R >& g, const TileThread< R >& th, int q )
{
   QPoint< R > P;
   const R*    xq = g.XQ[th.t][q];
#pragma unroll
   for ( int d = 0; d < 3; ++d )
      P.x[d] = th.p0[d] + xq[d];
   if ( g.kind )
   {
      const R ls = th.ls0 + xq[3];
      shellScalars( g, P.x, ls, P.qq, P.w, P.beta );
      P.ib = fastRcp( P.beta );
      P.r  = g.r0 + fabs( ls ) * g.dr;
   }
   else
   {
      P.qq = P.beta = P.ib = R( 1 );
      P.w[0] = P.w[1] = P.w[2] = R( 0 );
      P.r                      = sqrt( P.x[0] * P.x[0] + P.x[1] * P.x[1] + P.x[2] * P.x[2] );
   }
   return P;
}

// y (=|+=) the selected blocks on the cell lattices (halo positions included):
// MASK bit 1: yu = A u, bit 2: yu += B^T p, bit 4: yp = B u; MASK 8 alone:
// yp = M_k p, the P1 mass with k = 1/eta (the Schur-complement approximation
// of the block-factorisation preconditioner), 4-point degree-2 rule.
// T is the value type of the functions (double; float or half for the
// reduced-precision velocity block), the arithmetic runs in Acc<T>.
//
// Three forms, chosen by stokesForm:
// kStokesWide: stokesTiles tiles a workgroup, one micro-cell type a wavefront.  Results go
//   through copies of the result box, one a wavefront, one component after the other, with
//   plain LDS reads and writes in the spread layout.  Bound by FP64 issue and its latencies
//   at three wavefronts a SIMD (11.1 ms for 117 GFLOP, the vector unit about half busy).
//   168 registers a lane (masks 3 and 7 spill three and four, 16 and 20 bytes of scratch):
//   two of the three velocity components are read from LDS again at each point of the
//   viscous block (HELD in registers), box points and anchors are formed again for the
//   write-back.
// kStokesShared: one tile a workgroup, one result box filled with LDS atomics, the three
//   components in registers.  Two barriers where the wide form has seven: the shortest
//   chain, for launches that are bound by one workgroup's latency.
// kStokesLast: a last-layer tile (tileList) by one wavefront, its 64 micro-cells with the
//   type varying over the lanes -- a workgroup of the other forms would run six wavefronts
//   for them.
constexpr int kPBox3P = 128; // a pressure box, padded
enum StokesForm
{
   kStokesWide   = 0,
   kStokesShared = 1,
   kStokesLast   = 2
};
// Tiles a workgroup of the wide form: two, for three wavefronts on each SIMD; of a workgroup
// of six two of the four SIMDs hold two (full operator 11.5 against 10.3 ms, mask 6 11.1
// against 9.2 ms, shell level 5).  B^T alone has registers for two workgroups of one tile a
// CU, which overlap one's memory phases with the other's arithmetic (5.2 against 6.2 ms).
constexpr int stokesTiles( int mask, int form ) { return form != kStokesWide || mask == 2 ? 1 : 2; }
// wavefronts a SIMD that the registers leave room for (the shared form's merged divergence
// loop needs 192 registers)
constexpr int stokesWaves( int mask, int form )
{
   return form == kStokesLast || ( form == kStokesShared && ( ( mask & 1 ) || mask == 6 ) ) ? 2 : 3;
}
// The form of a launch over n tiles of lattices with mm micro-edges; kStokesLast: the
// interior tiles in the wide form and the last layer behind them.  Kernel times in us of
// shared / wide / wide and last, n tiles, on 256 CUs:
//   mask 7: 19 / 29 / 44 (cube level 4, 120), 35 / 33 / 48 (480), 50 / 57 / 49 (720),
//           428 / 439 / 365 (7200); level 1: 17 / 28 (36), 118 / 109 (1920)
//   mask 2: 9.5 / 11 / 19 (24), 21 / 23 / 26 (720), 274 / 306 / 306 (14400),
//           737 / 864 / 717 (38400); level 3: 144 / 173 / 111 (7680)
//   mask 4: 9.2 / 9.9 / 17 (24), 25 / 25 / 26 (1200), 44 / 39 / 35 (2400)
//   mask 6: 12 / 18 / 29 (24), 51 / 58 / 57 (1200), 93 / 94 / 86 (2400)
//   mask 8: 7.4 / 7.7 / 12 (24), 13 / 14 / 16 (1200), 23 / 20 / 19 (2400)
//   FP32 velocities: 22 / 16 / 28 (24), 141 / 70 / 73 (2400), 258 / 136 / 115 (4800);
//           level 1: 11 / 15 (36)
// Up to a tile a CU the chain of one workgroup counts (shared; FP32 has cheap wavefront
// boxes and expensive atomics), up to two a CU the wide form still is one round; beyond,
// the last layer by wavefronts saves more than its launch costs, later for the masks with
// less arithmetic.  On levels 0 and 1 a tile holds few micro-cells.
inline int stokesForm( int mask, bool fp32, int64_t mm, int64_t n )
{
   const bool viscous = mask & 1;
   if ( mm < kTile )
      return n <= 512 || mask == 2 || fp32 ? kStokesShared : kStokesWide;
   if ( mm == kTile ) // every tile is in the last layer
      return n <= 256 && ( fp32 || !( viscous || mask == 8 ) ) ? kStokesShared : kStokesLast;
   if ( fp32 )
      return n <= 3072 ? kStokesWide : kStokesLast;
   if ( mask == 2 )
      return n <= ( mm == 2 * kTile ? 512 : 16384 ) ? kStokesShared : kStokesLast;
   if ( n <= ( mask == 8 ? 2048 : 512 ) )
      return n <= 256 ? kStokesShared : kStokesWide;
   // (of eight micro-edges three tiles in four are in the last layer)
   return viscous || mask == 8 || n > 1440 || mm == 2 * kTile ? kStokesLast : kStokesShared;
}
template < int MASK, class T, int FORM >
__global__ __launch_bounds__( FORM == kStokesLast ? 64 : stokesTiles( MASK, FORM ) * kTileThreads,
                              stokesWaves( MASK, FORM ) ) void kStokesTileApply(
    const P2CellGeomT< typename Acc< T >::type >* __restrict__ geom, typename Acc< T >::type c0,
    typename Acc< T >::type c1, int64_t mm, int64_t ntiles, int64_t sc1, int64_t w1, int64_t sc0, int64_t w0,
    const T* __restrict__ u0, const T* __restrict__ u1, const T* __restrict__ u2, const T* __restrict__ pin,
    T* __restrict__ y0, T* __restrict__ y1, T* __restrict__ y2, T* __restrict__ yp, const uint64_t* __restrict__ tiles )
{
   using R  = typename Acc< T >::type;
   using QC = SQ< R >;
   constexpr bool DO_A = MASK & 1, DO_BT = MASK & 2, DO_B = MASK & 4, DO_M = MASK & 8;
   constexpr bool LAST = FORM == kStokesLast, SHARED = FORM == kStokesShared;
   constexpr int HELD = LAST || SHARED || sizeof( R ) == 4 ? 3 : 1;
   constexpr bool MERGED = SHARED && DO_B && DO_BT; // one loop over the divergence points
   constexpr bool NEED_U = DO_A || DO_B, OUT_U = DO_A || DO_BT, NEED_P = DO_BT || DO_M, OUT_P = DO_B || DO_M;
   constexpr int  kThreads = LAST ? 64 : kTileThreads, kWaves = kThreads / 64;
   constexpr int  kPoints  = LAST ? kDiagBoxP / 64 : 2; // velocity box points a thread
   constexpr int  kPPoints = LAST ? 2 : 1;              // and pressure box points
   static_assert( LAST || kBox3 <= 2 * kTileThreads, "box points per thread" );
   // the tile's velocity values and, when they have been used, the wavefronts' result boxes
   // (SHARED: the one result box behind them)
   constexpr int kULds = ( SHARED ? ( NEED_U ? 3 : 0 ) + ( OUT_U ? 3 : 0 ) : OUT_U && kWaves > 3 ? kWaves : 3 ) * kSpreadBox;
   constexpr int kTiles = stokesTiles( MASK, FORM ), kPCopies = SHARED ? 1 : kWaves;
   __shared__ R  suAll[kTiles][NEED_U || OUT_U ? kULds : 1];
   __shared__ R  spAll[kTiles][NEED_P ? kPBox3P : 1];
   __shared__ R  apAll[kTiles][OUT_P ? kPCopies * kPBox3P : 1];
   const int64_t lw = xcdBlock( ( ntiles + kTiles - 1 ) / kTiles );
   if ( lw * kTiles >= ntiles )
      return;
   const int     lane = int( threadIdx.x ) & 63, wgWave = LAST ? 0 : __builtin_amdgcn_readfirstlane( int( threadIdx.x ) >> 6 );
   const int     sub = LAST ? 0 : wgWave / kWaves, wave = wgWave - sub * kWaves; // tile of the workgroup
   R* const      su  = suAll[sub];
   R* const      sp  = spAll[sub];
   R* const      ap  = apAll[sub];
   R* const      au  = su + ( SHARED && NEED_U ? 3 * kSpreadBox : 0 ); // result boxes
   const int     tid0 = wave * 64 + lane; // thread number in the tile
   const bool    live = lw * kTiles + sub < ntiles;
   const int64_t lb   = live ? lw * kTiles + sub : ntiles - 1;
   int64_t         full;
   const TileCoord tc    = tileFromList( tiles, lb, mm, full );
   const int64_t   base1 = tc.c * sc1, base0 = tc.c * sc0;
   const T*        uin[3] = { u0, u1, u2 };
   const int       pair = LAST ? cDiagPairs[lane] : 0;
   const int       t = LAST ? pair & 7 : wave, a = LAST ? pair >> 3 : lane;
   // all loads issued before the first LDS write, so their latencies overlap
   const BoxOffsets box1( int32_t( w1 ), 2 * int32_t( tc.x0 ), 2 * int32_t( tc.y0 ), 2 * int32_t( tc.z0 ) );
   const BoxOffsets box0( int32_t( w0 ), int32_t( tc.x0 ), int32_t( tc.y0 ), int32_t( tc.z0 ) );
   const int32_t    rest0 = live ? int32_t( mm ) - int32_t( tc.x0 + tc.y0 + tc.z0 ) : -1, rest1 = 2 * rest0; // -1: no points
   // the thread's j-th box points: their LDS positions and lattice offsets (-1: none)
   auto velocityPoint = [&]( int tid, int j, int32_t& bp, int32_t& off ) {
      const int p   = tid + j * kThreads;
      const int box = LAST ? cDiagBox[p] : ( p < kBox3 ? p : -1 );
      int32_t   lx, ly, lz;
      boxPoint( box, lx, ly, lz );
      bp  = box >= 0 ? spreadPos( lx, ly, lz ) : -1;
      off = box >= 0 && lx + ly + lz <= rest1 ? box1.at( lx, ly, lz ) : -1;
   };
   auto pressurePoint = [&]( int tid, int j ) {
      const int p = tid + j * kThreads, lx = p % kPBox, ly = ( p / kPBox ) % kPBox, lz = p / ( kPBox * kPBox );
      return p < kPBox3 && lx + ly + lz <= rest0 ? box0.at( lx, ly, lz ) : -1;
   };
   int32_t bp[kPoints], off[kPoints], poff[kPPoints];
   T       uv[kPoints][3], pvl[kPPoints];
   if constexpr ( NEED_U )
#pragma unroll
      for ( int j = 0; j < kPoints; ++j )
      {
         velocityPoint( tid0, j, bp[j], off[j] );
#pragma unroll
         for ( int c = 0; c < 3; ++c )
            uv[j][c] = off[j] >= 0 ? ( uin[c] + base1 )[uint32_t( off[j] )] : T( 0 );
      }
   if constexpr ( NEED_P )
#pragma unroll
      for ( int j = 0; j < kPPoints; ++j )
      {
         poff[j] = pressurePoint( tid0, j );
         pvl[j]  = poff[j] >= 0 ? ( pin + base0 )[uint32_t( poff[j] )] : T( 0 );
      }
   if constexpr ( SHARED )
   {
      // cleared while the loads are in flight
      if constexpr ( OUT_U )
         for ( int p = tid0; p < 3 * kSpreadBox; p += kThreads )
            au[p] = R( 0 );
      if constexpr ( OUT_P )
         if ( tid0 < kPBox3P )
            ap[tid0] = R( 0 );
   }
   if constexpr ( NEED_U )
   {
#pragma unroll
      for ( int j = 0; j < kPoints; ++j )
         if ( bp[j] >= 0 )
#pragma unroll
            for ( int c = 0; c < 3; ++c )
               su[c * kSpreadBox + bp[j]] = toAcc( uv[j][c] );
   }
   if constexpr ( NEED_P )
   {
#pragma unroll
      for ( int j = 0; j < kPPoints; ++j )
         if ( tid0 + j * kThreads < kPBox3P )
            sp[tid0 + j * kThreads] = toAcc( pvl[j] );
   }
   __syncthreads();
   const P2CellGeomT< R >& g  = geom[tc.c];
   TileThread< R >         th; // (32-bit tile coordinates: 64-bit ones held two registers each)
   {
      th.t  = t;
      th.ax = a & 3;
      th.ay = ( a >> 2 ) & 3;
      th.az = a >> 4;
      const R vx = R( int32_t( tc.x0 ) + th.ax + vertexOffset< 0 >( t, 0 ) ), vy = R( int32_t( tc.y0 ) + th.ay + vertexOffset< 1 >( t, 0 ) ),
              vz = R( int32_t( tc.z0 ) + th.az + vertexOffset< 2 >( t, 0 ) );
#pragma unroll
      for ( int d = 0; d < 3; ++d )
         th.p0[d] = g.v0[d] + g.hE[3 * d] * vx + g.hE[3 * d + 1] * vy + g.hE[3 * d + 2] * vz;
      th.ls0   = g.nl[0] * th.p0[0] + g.nl[1] * th.p0[1] + g.nl[2] * th.p0[2] - g.lam0;
      th.valid = LAST || th.ax + th.ay + th.az < rest0 - MicroCells::rowShift[t];
   }
   int                     lanePos[LAST ? 10 : 1];
   const int               b1 = LAST ? 0 : spreadPos( 2 * th.ax, 2 * th.ay, 2 * th.az );
   if constexpr ( LAST )
   {
      laneBoxPositions( t, a, lanePos );
#pragma unroll
      for ( int i = 0; i < 10; ++i )
      {
         int32_t lx, ly, lz;
         boxPoint( lanePos[i], lx, ly, lz );
         lanePos[i] = spreadPos( lx, ly, lz );
      }
   }
   // f( at ): at( i ) = box position of local DoF i, from b1
   auto withPositions = [&]( auto&& f ) {
      if constexpr ( LAST )
         f( [&]( int i ) { return lanePos[i]; } );
      else
         forType( t, [&]( auto box ) { f( [&]( int i ) { return spreadOf( box.at( i ) ); } ); } );
   };
   auto ppos = [&]( int k ) {
      return ( th.ax + vertexOffset< 0 >( t, k ) ) +
             kPBox * ( ( th.ay + vertexOffset< 1 >( t, k ) ) + kPBox * ( th.az + vertexOffset< 2 >( t, k ) ) );
   };
   // LDS accesses of a wavefront to its own copies: volatile, they complete in order
   using LdsR = volatile __attribute__( ( address_space( 3 ) ) ) R;
   LdsR* const apw = (LdsR*) ( ap + ( OUT_P && !SHARED ? wave * kPBox3P : 0 ) );
   auto pressureResults = [&]( const R yq[4] ) {
      if constexpr ( !SHARED )
      {
         apw[lane]      = R( 0 );
         apw[lane + 64] = R( 0 );
      }
      if ( th.valid )
      {
         if constexpr ( LAST || SHARED )
#pragma unroll
            for ( int k = 0; k < 4; ++k )
               atomicAdd( &ap[ppos( k )], yq[k] );
         else
#pragma unroll
            for ( int k = 0; k < 4; ++k )
               apw[ppos( k )] = apw[ppos( k )] + yq[k];
      }
   };
   const R* Dc   = g.Dc[t];
   const R  adet = g.adet[t];
   R        u[3][10], y[3][10];
   // (one opaque base address: the loops would keep the address of every value otherwise)
   using LdsIn = const __attribute__( ( address_space( 3 ) ) ) R;
   auto component = [&]( int c ) {
      LdsIn* base = (LdsIn*) su + c * kSpreadBox + b1;
      asm volatile( "" : "+v"( base ) );
      withPositions( [&]( auto at ) {
#pragma unroll
         for ( int i = 0; i < 10; ++i )
            u[c][i] = base[at( i )];
      } );
   };
   auto clear = [&]() {
#pragma unroll
      for ( int c = 0; c < 3; ++c )
#pragma unroll
         for ( int i = 0; i < 10; ++i )
            y[c][i] = R( 0 );
   };
   // y += s (q div of the test functions)
   auto gradientTests = [&]( const R* a4, const R* b4, R s, const R M[3][3] ) {
#pragma unroll
      for ( int c = 0; c < 3; ++c )
         testGrad( a4, b4, s * M[c][0], s * M[c][1], s * M[c][2], y[c] );
   };
   if constexpr ( NEED_U )
#pragma unroll
      for ( int c = 0; c < 3; ++c )
         component( c );
   // a wavefront without micro-cells in the macro-cell (lattices of one or two micro-edges)
   // has no quadrature points
   const bool work = __any( th.valid );
   const int  qA = work ? 5 : 0, qB = work ? 9 : 0;
   if constexpr ( MERGED )
      clear();
   if constexpr ( DO_B )
   {
      R pv[4], yq[4] = { R( 0 ), R( 0 ), R( 0 ), R( 0 ) };
      if constexpr ( MERGED )
#pragma unroll
         for ( int k = 0; k < 4; ++k )
            pv[k] = sp[ppos( k )];
#pragma unroll 1
      for ( int q = 5; q < qB; ++q )
      {
         const R*          a4  = QC::a4( q );
         const R*          b4  = QC::b4( q );
         const R*          lam = QC::lam( q );
         const QPoint< R > P   = qpoint( g, th, q );
         const R           cc  = QC::w( q ) * adet * fabs( P.beta ) * P.qq;
         R                 M[3][3];
         mapGradients( Dc, P.x, P.w, P.ib, M );
         // q div u = trace of q grad u
         R dq = R( 0 );
#pragma unroll
         for ( int c = 0; c < 3; ++c )
         {
            R gm[4];
            baryGrad( a4, b4, u[c], gm );
            dq += ( gm[1] - gm[0] ) * M[c][0] + ( gm[2] - gm[0] ) * M[c][1] + ( gm[3] - gm[0] ) * M[c][2];
         }
         const R s = -cc * dq;
#pragma unroll
         for ( int k = 0; k < 4; ++k )
            yq[k] += lam[k] * s;
         if constexpr ( MERGED )
            gradientTests( a4, b4, -cc * ( lam[0] * pv[0] + lam[1] * pv[1] + lam[2] * pv[2] + lam[3] * pv[3] ), M );
      }
      pressureResults( yq );
   }
   if constexpr ( !MERGED )
      clear();
   if constexpr ( DO_A )
   {
#pragma unroll 1
      for ( int q = 0; q < qA; ++q )
      {
         const R* a4 = QC::a4( q );
         const R* b4 = QC::b4( q );
         R        M[3][3], cc;
         {
            const QPoint< R > P = qpoint( g, th, q );
            cc                  = QC::w( q ) * adet * fabs( P.beta ) * rexp( c0 + c1 * P.r );
            mapGradients( Dc, P.x, P.w, P.ib, M );
         }
         // S = G + G^T, G[c][d]: q times the d-th derivative of component c
         R S[3][3];
#pragma unroll
         for ( int c = 0; c < 3; ++c )
         {
            R gm[4];
            if ( c >= HELD )
            {
               __builtin_amdgcn_sched_barrier( 0 );
               component( c );
            }
            baryGrad( a4, b4, u[c], gm );
            const R d1 = gm[1] - gm[0], d2 = gm[2] - gm[0], d3 = gm[3] - gm[0];
#pragma unroll
            for ( int d = 0; d < 3; ++d )
            {
               const R G = d1 * M[d][0] + d2 * M[d][1] + d3 * M[d][2];
               if ( d < c )
                  S[d][c] += G;
               else
                  S[c][d] = G; // the upper triangle
            }
         }
         // stress times the weight and the coefficient
         const R tr = ( R( 2 ) / R( 3 ) ) * ( S[0][0] + S[1][1] + S[2][2] );
#pragma unroll
         for ( int c = 0; c < 3; ++c )
         {
            S[c][c] = cc * ( R( 2 ) * S[c][c] - tr );
#pragma unroll
            for ( int d = c + 1; d < 3; ++d )
               S[d][c] = S[c][d] = cc * S[c][d];
         }
#pragma unroll
         for ( int c = 0; c < 3; ++c )
            testGrad( a4, b4, M[0][0] * S[c][0] + M[1][0] * S[c][1] + M[2][0] * S[c][2],
                      M[0][1] * S[c][0] + M[1][1] * S[c][1] + M[2][1] * S[c][2],
                      M[0][2] * S[c][0] + M[1][2] * S[c][1] + M[2][2] * S[c][2], y[c] );
      }
   }
   if constexpr ( NEED_P && !MERGED )
   {
      R pv[4], yq[4] = { R( 0 ), R( 0 ), R( 0 ), R( 0 ) };
#pragma unroll
      for ( int k = 0; k < 4; ++k )
         pv[k] = sp[ppos( k )];
#pragma unroll 1
      for ( int q = 5; q < qB; ++q )
      {
         const R*          lam = QC::lam( q );
         const QPoint< R > P   = qpoint( g, th, q );
         const R           pq  = lam[0] * pv[0] + lam[1] * pv[1] + lam[2] * pv[2] + lam[3] * pv[3];
         const R           cc  = QC::w( q ) * adet * fabs( P.beta ) * P.qq;
         if constexpr ( DO_M )
         {
            // |det D(F J)| = q^2 |beta| adet; k = 1/eta at the blended point
            const R s = cc * P.qq * rexp( -( c0 + c1 * P.r ) ) * pq;
#pragma unroll
            for ( int k = 0; k < 4; ++k )
               yq[k] += lam[k] * s;
         }
         else
         {
            const R* a4 = QC::a4( q );
            const R* b4 = QC::b4( q );
            R        M[3][3];
            mapGradients( Dc, P.x, P.w, P.ib, M );
            gradientTests( a4, b4, -cc * pq, M );
         }
      }
      if constexpr ( DO_M )
         pressureResults( yq );
   }
   if constexpr ( SHARED && OUT_U )
      if ( th.valid )
         withPositions( [&]( auto at ) {
#pragma unroll
            for ( int c = 0; c < 3; ++c )
#pragma unroll
               for ( int i = 0; i < 10; ++i )
                  atomicAdd( &au[c * kSpreadBox + b1 + at( i )], y[c][i] );
         } );
   __syncthreads(); // the velocity values are read (SHARED: the results added)
   // lane, anchor and box points again, rather than kept through the quadrature loops
   int ones = -1;
   asm volatile( "" : "+s"( ones ) );
   const int  laneEnd = int( __builtin_amdgcn_mbcnt_hi( uint32_t( ones ), __builtin_amdgcn_mbcnt_lo( uint32_t( ones ), 0 ) ) );
   const int  tid = wave * 64 + laneEnd, axEnd = laneEnd & 3, ayEnd = ( laneEnd >> 2 ) & 3, azEnd = laneEnd >> 4;
   if constexpr ( OUT_P )
   {
#pragma unroll
      for ( int j = 0; j < kPPoints; ++j )
      {
         const int32_t o = pressurePoint( tid, j );
         if ( o >= 0 )
         {
            R v = ap[tid + j * kThreads];
#pragma unroll
            for ( int w = 1; w < kPCopies; ++w )
               v += ap[w * kPBox3P + tid];
            sharedAdd( yp + base0 + uint32_t( o ), v );
         }
      }
   }
   if constexpr ( OUT_U )
   {
      // atomics for every point: a read-modify-write of the box interior would wait for
      // the outstanding atomics of the box surface
      T* yout[3] = { y0, y1, y2 };
#pragma unroll
      for ( int j = 0; j < kPoints; ++j )
         velocityPoint( tid, j, bp[j], off[j] );
      auto writeBoxes = [&]( const R* box ) {
#pragma unroll
         for ( int j = 0; j < kPoints; ++j )
            if ( off[j] >= 0 )
#pragma unroll
               for ( int c = 0; c < 3; ++c )
                  sharedAdd( yout[c] + base1 + uint32_t( off[j] ), box[c * kSpreadBox + bp[j]] );
      };
      if constexpr ( SHARED )
         writeBoxes( au );
      else if constexpr ( LAST )
      {
         for ( int p = tid; p < 3 * kSpreadBox; p += 64 )
            su[p] = R( 0 );
         __syncthreads();
#pragma unroll
         for ( int c = 0; c < 3; ++c )
#pragma unroll
            for ( int i = 0; i < 10; ++i )
               atomicAdd( &su[c * kSpreadBox + lanePos[i]], y[c][i] ); // every pair is a micro-cell
         __syncthreads();
         writeBoxes( su );
      }
      else
      {
         LdsR* const own = (LdsR*) ( su + wave * kSpreadBox );
         const int   b1e = spreadPos( 2 * axEnd, 2 * ayEnd, 2 * azEnd );
#pragma unroll
         for ( int c = 0; c < 3; ++c )
         {
            if ( c > 0 )
               __syncthreads(); // the component before is summed
#pragma unroll
            for ( int p = 0; p < kSpreadBox; p += 64 )
               if ( p + 64 <= kSpreadBox || laneEnd < kSpreadBox - p )
                  own[p + laneEnd] = R( 0 );
            if ( axEnd + ayEnd + azEnd < rest0 - MicroCells::rowShift[t] )
               withPositions( [&]( auto at ) {
#pragma unroll
                  for ( int i = 0; i < 10; ++i )
                     own[b1e + at( i )] = own[b1e + at( i )] + y[c][i];
               } );
            __syncthreads();
#pragma unroll
            for ( int j = 0; j < kPoints; ++j )
               if ( off[j] >= 0 )
               {
                  const R* b = su + bp[j];
                  sharedAdd( yout[c] + base1 + uint32_t( off[j] ),
                             ( ( b[0] + b[kSpreadBox] ) + ( b[2 * kSpreadBox] + b[3 * kSpreadBox] ) ) +
                                 ( b[4 * kSpreadBox] + b[5 * kSpreadBox] ) );
               }
         }
      }
   }
}

// diagonal of the three diagonal blocks of A:
//   sum_q w |det M| eta (|grad phi_j|^2 + (d_c phi_j)^2 / 3)
// added into the cell lattices (halo positions included)
__global__ __launch_bounds__( kTileThreads ) void kStokesTileDiag( const P2CellGeom* __restrict__ geom, double c0,
                                                                   double c1, int64_t mm, int64_t ntiles, int64_t sc1,
                                                                   int64_t w1, double* __restrict__ d0,
                                                                   double* __restrict__ d1, double* __restrict__ d2 )
{
   const int64_t lb = blockIdx.x;
   if ( lb >= ntiles )
      return;
   const TileCoord            tc = tileOf( lb, mm );
   const P2CellGeom&          g  = geom[tc.c];
   const TileThread< double > th = tileThread( g, tc, mm );
   if ( !th.valid )
      return;
   const double* Dc   = g.Dc[th.t];
   const double  adet = g.adet[th.t];
   double        dg[3][10] = {};
   for ( int q = 0; q < 5; ++q )
   {
      const double*          a4 = cSQ4[q];
      const double*          b4 = cSQ4m[q];
      const QPoint< double > P  = qpoint( g, th, q );
      const double           cc = cSQW[q] * adet * fabs( P.beta ) * exp( c0 + c1 * P.r );
      // computational gradients of lam_0..3
      double gl[4][3];
      for ( int d = 0; d < 3; ++d )
      {
         gl[1][d] = Dc[d];
         gl[2][d] = Dc[3 + d];
         gl[3][d] = Dc[6 + d];
         gl[0][d] = -( gl[1][d] + gl[2][d] + gl[3][d] );
      }
      for ( int j = 0; j < 10; ++j )
      {
         double v[3];
         if ( j < 4 )
            for ( int d = 0; d < 3; ++d )
               v[d] = b4[j] * gl[j][d];
         else
         {
            const int a = cP2E[j - 4][0], b = cP2E[j - 4][1];
            for ( int d = 0; d < 3; ++d )
               v[d] = a4[b] * gl[a][d] + a4[a] * gl[b][d];
         }
         const double t = ( P.x[0] * v[0] + P.x[1] * v[1] + P.x[2] * v[2] ) * P.ib;
         for ( int d = 0; d < 3; ++d )
            v[d] -= P.w[d] * t;
         const double n2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
         for ( int c = 0; c < 3; ++c )
            dg[c][j] += cc * ( n2 + v[c] * v[c] / 3.0 );
      }
   }
   const int64_t gx = tc.x0 + th.ax, gy = tc.y0 + th.ay, gz = tc.z0 + th.az;
   int64_t       vx[4][3];
   for ( int k = 0; k < 4; ++k )
   {
      vx[k][0] = gx + cVof[th.t][k][0];
      vx[k][1] = gy + cVof[th.t][k][1];
      vx[k][2] = gz + cVof[th.t][k][2];
   }
   double* dout[3] = { d0, d1, d2 };
   for ( int j = 0; j < 10; ++j )
   {
      int64_t X, Y, Z;
      if ( j < 4 )
         X = 2 * vx[j][0], Y = 2 * vx[j][1], Z = 2 * vx[j][2];
      else
      {
         const int a = cP2E[j - 4][0], b = cP2E[j - 4][1];
         X = vx[a][0] + vx[b][0], Y = vx[a][1] + vx[b][1], Z = vx[a][2] + vx[b][2];
      }
      const int64_t idx = tc.c * sc1 + tetRowStart32( int32_t( w1 ), int32_t( Y ), int32_t( Z ) ) + X;
      for ( int c = 0; c < 3; ++c )
         atomicAdd( dout[c] + idx, dg[c][j] );
   }
}

// P1 diagonal operators on the affine micro-cells of level L (kind 0: the
// PSPG diagonal -(|T|^(2/3)/12) |T| |grad lam_k|^2, kind 1: the lumped mass
// |T|/4), added into the level-L cell lattices
__global__ __launch_bounds__( kTileThreads ) void kP1AffineDiag( const P2CellGeom* __restrict__ geom, int kind,
                                                                 int64_t mm, int64_t ntiles, int64_t sc0, int64_t w0,
                                                                 double* __restrict__ dst )
{
   const int64_t lb = blockIdx.x;
   if ( lb >= ntiles )
      return;
   const TileCoord            tc = tileOf( lb, mm );
   const P2CellGeom&          g  = geom[tc.c];
   const TileThread< double > th = tileThread( g, tc, mm );
   if ( !th.valid )
      return;
   const double* Dc  = g.Dc[th.t];
   const double  vol = g.adet[th.t] / 6.0;
   const double  s   = -cbrt( vol * vol ) / 12.0 * vol;
   for ( int k = 0; k < 4; ++k )
   {
      double gk[3];
      for ( int d = 0; d < 3; ++d )
         gk[d] = k == 0 ? -( Dc[d] + Dc[3 + d] + Dc[6 + d] ) : Dc[3 * ( k - 1 ) + d];
      const double  v   = kind == 0 ? s * ( gk[0] * gk[0] + gk[1] * gk[1] + gk[2] * gk[2] ) : 0.25 * vol;
      const int64_t X   = tc.x0 + th.ax + cVof[th.t][k][0];
      const int64_t Y   = tc.y0 + th.ay + cVof[th.t][k][1];
      const int64_t Z   = tc.z0 + th.az + cVof[th.t][k][2];
      const int64_t idx = tc.c * sc0 + tetRowStart32( int32_t( w0 ), int32_t( Y ), int32_t( Z ) ) + X;
      atomicAdd( dst + idx, v );
   }
}
} // namespace

// v += value on the flagged DoFs of a single-vector FP64 function
__global__ void kAddConst( int64_t ncell, int64_t nb, const uint8_t* __restrict__ bndFlag, int flag, double value,
                           double* __restrict__ v )
{
   const int64_t i = int64_t( blockIdx.x ) * blockDim.x + threadIdx.x;
   const int64_t n = ( flag & kInner ? ncell : 0 ) + nb;
   if ( i >= n )
      return;
   const int64_t pt = ( flag & kInner ) ? i : ncell + i;
   if ( pt >= ncell && !( bndFlag[pt - ncell] & flag ) )
      return;
   v[pt] += value;
}

// v = 1/v on the flagged DoFs of a single-vector FP64 function (zeros stay)
__global__ void kInvertFlagged( int64_t ncell, int64_t nb, const uint8_t* __restrict__ bndFlag, int flag,
                                double* __restrict__ v )
{
   const int64_t i = int64_t( blockIdx.x ) * blockDim.x + threadIdx.x;
   const int64_t n = ( flag & kInner ? ncell : 0 ) + nb;
   if ( i >= n )
      return;
   const int64_t pt = ( flag & kInner ) ? i : ncell + i;
   if ( pt >= ncell && !( bndFlag[pt - ncell] & flag ) )
      return;
   if ( v[pt] != 0.0 )
      v[pt] = 1.0 / v[pt];
}

// u -= (u . n) n on the owned boundary DoFs whose type is in flag
// (P2ProjectNormalOperator::project, p1functionspace/freeslip/VertexDoFProjectNormal.hpp:43-120)
template < class T >
__global__ void kProjectNormal( int64_t nb, int64_t ncell, const uint8_t* __restrict__ bndFlag, int flag,
                                const double* __restrict__ nrm, T* __restrict__ u0, T* __restrict__ u1,
                                T* __restrict__ u2 )
{
   using R         = typename Acc< T >::type;
   const int64_t b = int64_t( blockIdx.x ) * blockDim.x + threadIdx.x;
   if ( b >= nb || !( bndFlag[b] & flag ) )
      return;
   const double* n    = nrm + 3 * b;
   const int64_t p    = ncell + b;
   const R       v[3] = { R( toAcc( u0[p] ) ), R( toAcc( u1[p] ) ), R( toAcc( u2[p] ) ) };
   const R       d    = R( n[0] ) * v[0] + R( n[1] ) * v[1] + R( n[2] ) * v[2];
   u0[p]              = fromAcc< T >( v[0] - d * R( n[0] ) );
   u1[p]              = fromAcc< T >( v[1] - d * R( n[1] ) );
   u2[p]              = fromAcc< T >( v[2] - d * R( n[2] ) );
}

struct StokesOperator : OperatorBase
{
   Storage*                                            st   = nullptr;
   int                                                 minL = 0, maxL = 0;
   double                                              c0 = 0.0, c1 = 0.0;
   std::map< int, DevBuf< P2CellGeom > >               tgeom;   // by P2 level
   std::map< int, DevBuf< P2CellGeomT< float > > >    tgeom32; // the same in FP32 (reduced-precision velocity block)
   std::map< int, std::array< DevBuf< double >, 3 > > invDiag; // velocity, lattice L+1
   std::map< int, DevBuf< double > >                   pspgInv, lumpedInv; // lattice L
};

namespace {

void checkVelocity( const StokesOperator& op, const Function& f, int L, int dtype = 0 )
{
   if ( f.st != op.st || f.off != 1 || f.lv != 0 || f.dtype != dtype )
      throw Error( HG_ERR_ARG, dtype == 0 ? "Stokes velocity components must be FP64 P2 functions on the operator's storage" :
                                            "the velocity components of a reduced-precision apply must share one type" );
   if ( L < op.minL || L > op.maxL || L < f.minL || L > f.maxL )
      throw Error( HG_ERR_ARG, "level outside the operator's or function's level range" );
}

void checkPressure( const StokesOperator& op, const Function& f, int L )
{
   if ( f.st != op.st || f.off != 0 || f.lv != 0 || f.dtype != 0 )
      throw Error( HG_ERR_ARG, "Stokes pressure must be an FP64 P1 function on the operator's storage" );
   if ( L < op.minL || L > op.maxL || L < f.minL || L > f.maxL )
      throw Error( HG_ERR_ARG, "level outside the operator's or function's level range" );
}

// pressure DoFs are all Inner (P2P1TaylorHoodFunction gives the pressure
// createAllInnerBC): a velocity flag selects every pressure DoF or none
int pressureFlag( int flag ) { return ( flag & kInner ) ? kAll : 0; }

template < class T >
void zeroTarget( Context* ctx, Storage& st, Lattice& lat, T* d, bool replaceAll )
{
   if ( replaceAll )
      kFillRange< T ><<< gridFor( lat.nc * lat.sc ), kBlock, 0, ctx->stream >>>( lat.nc * lat.sc, d, 0.0 );
   else if ( lat.haloPerCell() > 0 )
      kZeroHalos< T ><<< gridFor( lat.haloPerCell() * lat.nc ), kBlock, 0, ctx->stream >>>( BndGeom::of( st, lat ),
                                                                                         lat.nc, d );
   HG_CHECK_HIP( hipGetLastError() );
}

// the lists that the launches on a lattice read, built ahead of a timed region, whatever
// the mask: a launch captured after one of another mask cannot allocate its list
void stokesTileLists( Context* ctx, Lattice& l1, int64_t mm )
{
   const int64_t n = tilesPerCell( mm ) * l1.nc;
   for ( int mask = 0; mask <= 8; ++mask ) // 0: the velocity block in FP32
      if ( stokesForm( mask ? mask : 1, mask == 0, mm, n ) != kStokesLast )
         tileList( ctx, l1, mm, kTilesAll );
      else
         for ( int kind : { kTilesInterior, kTilesLast } )
            tileList( ctx, l1, mm, kind );
}

template < int MASK, class T >
void launchStokes( Context* ctx, StokesOperator& op, const P2CellGeomT< typename Acc< T >::type >* geom, int L, Lattice& l1,
                   Lattice& l0, T* const u[3], const T* p, T* const y[3], T* yp )
{
   using R          = typename Acc< T >::type;
   const int64_t mm = int64_t( 1 ) << L, T0 = tileEdges( mm );
   auto launch = [&]( auto which, int kind, int64_t ntiles ) {
      constexpr int FORM = decltype( which )::value, kTiles = stokesTiles( MASK, FORM );
      if ( ntiles < 1 )
         return;
      kStokesTileApply< MASK, T, FORM >
          <<< xcdGrid( ( ntiles + kTiles - 1 ) / kTiles ), FORM == kStokesLast ? 64 : kTiles * kTileThreads, 0, ctx->stream >>>(
          geom, R( op.c0 ), R( op.c1 ), mm, ntiles, l1.sc, l1.w, l0.sc, l0.w, u[0], u[1], u[2], p, y[0], y[1], y[2], yp,
          tileList( ctx, l1, mm, kind ) );
      HG_CHECK_HIP( hipGetLastError() );
   };
   using Wide   = std::integral_constant< int, kStokesWide >;
   using Shared = std::integral_constant< int, kStokesShared >;
   using Last   = std::integral_constant< int, kStokesLast >;
   const int64_t n = tilesPerCell( mm ) * l1.nc;
   switch ( stokesForm( MASK, std::is_same< R, float >::value, mm, n ) )
   {
   case kStokesShared: launch( Shared{}, kTilesAll, n ); break;
   case kStokesWide: launch( Wide{}, kTilesAll, n ); break;
   default:
      launch( Wide{}, kTilesInterior, tet( T0 - 1 ) * l1.nc );
      launch( Last{}, kTilesLast, T0 * ( T0 + 1 ) / 2 * l1.nc );
   }
}

// the velocity block alone on FP32 or FP16 velocity functions (FP32 arithmetic)
void stokesViscousLowPrecision( Context* ctx, StokesOperator& op, Function* const src[4], Function* const dst[4], int L,
                                int flag, int update )
{
   const int dtype = src[0]->dtype;
   for ( int c = 0; c < 3; ++c )
   {
      checkVelocity( op, *src[c], L, dtype );
      checkVelocity( op, *dst[c], L, dtype );
      for ( int k = 0; k < 3; ++k )
         if ( src[c] == dst[k] )
            throw Error( HG_ERR_ARG, "apply needs distinct src and dst functions" );
   }
   Storage&      st = *op.st;
   Lattice&      l1 = st.lattice( ctx, L + 1 );
   Lattice&      l0 = st.lattice( ctx, L );
   const int64_t mm = int64_t( 1 ) << L;
   if ( l1.w > 1024 )
      throw Error( HG_ERR_UNSUPPORT, "Stokes apply supports levels up to 8 (32-bit lattice offsets)" );
   stokesTileLists( ctx, l1, mm );
   dispatchType( dtype, [&]( auto tag ) {
      using T = decltype( tag );
      if constexpr ( std::is_same< T, double >::value )
         throw Error( HG_ERR_ARG, "FP64 velocity goes through the FP64 apply" );
      else
      {
         T* u[3];
         T* y[3];
         for ( int c = 0; c < 3; ++c )
         {
            u[c] = (T*) src[c]->ptr( L );
            pullHalos( ctx, st, l1, u[c], dtype );
            y[c] = (T*) dst[c]->ptr( L );
            zeroTarget( ctx, st, l1, y[c], update == HG_REPLACE && ( flag & kInner ) );
         }
         ctx->beginTiming();
         launchStokes< 1, T >( ctx, op, op.tgeom32.at( L ).p, L, l1, l0, u, nullptr, y, nullptr );
         ctx->endTiming();
         for ( int c = 0; c < 3; ++c )
            pushAdditive( ctx, st, l1, y[c], dtype, kAll ^ flag, update == HG_REPLACE );
      }
   } );
}

void stokesApply( Context* ctx, StokesOperator& op, Function* const src[4], Function* const dst[4], int L, int flag,
                  int mask, int update )
{
   if ( mask < 1 || mask > 8 )
      throw Error( HG_ERR_ARG, "block mask must be 1..7 (1: A u, 2: B^T p, 4: B u) or 8 (the 1/eta pressure mass)" );
   const bool needU = mask & 5, needP = mask & 10, outU = mask & 3, outP = mask & 12;
   for ( int c = 0; c < 4; ++c )
      if ( ( ( c < 3 ? needU : needP ) && !src[c] ) || ( ( c < 3 ? outU : outP ) && !dst[c] ) )
         throw Error( HG_ERR_ARG, "a function the block mask needs is missing" );
   if ( mask == 1 && src[0]->dtype != 0 )
   {
      stokesViscousLowPrecision( ctx, op, src, dst, L, flag, update );
      return;
   }
   for ( int c = 0; c < 3; ++c )
   {
      if ( needU )
         checkVelocity( op, *src[c], L );
      if ( outU )
         checkVelocity( op, *dst[c], L );
   }
   if ( needP )
      checkPressure( op, *src[3], L );
   if ( outP )
      checkPressure( op, *dst[3], L );
   for ( int c = 0; c < 4; ++c )
      for ( int k = 0; k < 4; ++k )
         if ( ( ( c < 3 && needU ) || ( c == 3 && needP ) ) && ( ( k < 3 && outU ) || ( k == 3 && outP ) ) &&
              src[c] == dst[k] )
            throw Error( HG_ERR_ARG, "apply needs distinct src and dst functions" );
   Storage&      st = *op.st;
   Lattice&      l1 = st.lattice( ctx, L + 1 );
   Lattice&      l0 = st.lattice( ctx, L );
   const int64_t mm = int64_t( 1 ) << L;
   if ( l1.w > 1024 )
      throw Error( HG_ERR_UNSUPPORT, "Stokes apply supports levels up to 8 (32-bit lattice offsets)" );
   double* u[3] = { nullptr, nullptr, nullptr };
   double* y[3] = { nullptr, nullptr, nullptr };
   double* p    = nullptr;
   double* yp   = nullptr;
   for ( int c = 0; c < 3; ++c )
   {
      if ( needU )
      {
         u[c] = (double*) src[c]->ptr( L );
         pullHalos( ctx, st, l1, u[c], 0 );
      }
      if ( outU )
      {
         y[c] = (double*) dst[c]->ptr( L );
         zeroTarget( ctx, st, l1, y[c], update == HG_REPLACE && ( flag & kInner ) );
      }
   }
   const int pflag = pressureFlag( flag );
   if ( needP )
   {
      p = (double*) src[3]->ptr( L );
      pullHalos( ctx, st, l0, p, 0 );
   }
   if ( outP )
   {
      yp = (double*) dst[3]->ptr( L );
      zeroTarget( ctx, st, l0, yp, update == HG_REPLACE && ( pflag & kInner ) );
   }
   stokesTileLists( ctx, l1, mm );
   ctx->beginTiming();
   switch ( mask )
   {
   case 1: launchStokes< 1, double >( ctx, op, op.tgeom.at( L ).p, L, l1, l0, u, p, y, yp ); break;
   case 2: launchStokes< 2, double >( ctx, op, op.tgeom.at( L ).p, L, l1, l0, u, p, y, yp ); break;
   case 3: launchStokes< 3, double >( ctx, op, op.tgeom.at( L ).p, L, l1, l0, u, p, y, yp ); break;
   case 4: launchStokes< 4, double >( ctx, op, op.tgeom.at( L ).p, L, l1, l0, u, p, y, yp ); break;
   case 5: launchStokes< 5, double >( ctx, op, op.tgeom.at( L ).p, L, l1, l0, u, p, y, yp ); break;
   case 6: launchStokes< 6, double >( ctx, op, op.tgeom.at( L ).p, L, l1, l0, u, p, y, yp ); break;
   case 7: launchStokes< 7, double >( ctx, op, op.tgeom.at( L ).p, L, l1, l0, u, p, y, yp ); break;
   default: launchStokes< 8, double >( ctx, op, op.tgeom.at( L ).p, L, l1, l0, u, p, y, yp ); break;
   }
   ctx->endTiming();
   if ( outU )
      for ( int c = 0; c < 3; ++c )
         pushAdditive( ctx, st, l1, y[c], 0, kAll ^ flag, update == HG_REPLACE );
   if ( outP )
      pushAdditive( ctx, st, l0, yp, 0, kAll ^ pflag, update == HG_REPLACE );
}

const std::array< DevBuf< double >, 3 >& velocityInverseDiagonal( Context* ctx, StokesOperator& op, int L )
{
   auto it = op.invDiag.find( L );
   if ( it != op.invDiag.end() )
      return it->second;
   Storage& st  = *op.st;
   Lattice& lat = st.lattice( ctx, L + 1 );
   auto&    b   = op.invDiag[L];
   for ( auto& d : b )
   {
      d.alloc( ctx, lat.nstore );
      kFillRange< double ><<< gridFor( lat.nstore ), kBlock, 0, ctx->stream >>>( lat.nstore, d.p, 0.0 );
   }
   const int64_t mm     = int64_t( 1 ) << L;
   const int64_t ntiles = tilesPerCell( mm ) * lat.nc;
   kStokesTileDiag<<< gridFor( ntiles, 1 ), kTileThreads, 0, ctx->stream >>>( op.tgeom.at( L ).p, op.c0, op.c1, mm, ntiles,
                                                                             lat.sc, lat.w, b[0].p, b[1].p, b[2].p );
   HG_CHECK_HIP( hipGetLastError() );
   for ( auto& d : b )
   {
      pushAdditive( ctx, st, lat, d.p, 0, 0, true );
      kInvertNonZero<<< gridFor( lat.nstore ), kBlock, 0, ctx->stream >>>( lat.nstore, d.p );
   }
   HG_CHECK_HIP( hipGetLastError() );
   return b;
}

const double* affineInverseDiagonal( Context* ctx, StokesOperator& op, int L, int kind )
{
   auto& m  = kind == 0 ? op.pspgInv : op.lumpedInv;
   auto  it = m.find( L );
   if ( it != m.end() )
      return it->second.p;
   Storage& st  = *op.st;
   Lattice& lat = st.lattice( ctx, L );
   auto&    b   = m[L];
   b.alloc( ctx, lat.nstore );
   kFillRange< double ><<< gridFor( lat.nstore ), kBlock, 0, ctx->stream >>>( lat.nstore, b.p, 0.0 );
   const int64_t mm     = int64_t( 1 ) << L;
   const int64_t ntiles = tilesPerCell( mm ) * lat.nc;
   kP1AffineDiag<<< gridFor( ntiles, 1 ), kTileThreads, 0, ctx->stream >>>( op.tgeom.at( L ).p, kind, mm, ntiles, lat.sc,
                                                                           lat.w, b.p );
   HG_CHECK_HIP( hipGetLastError() );
   pushAdditive( ctx, st, lat, b.p, 0, 0, true );
   kInvertNonZero<<< gridFor( lat.nstore ), kBlock, 0, ctx->stream >>>( lat.nstore, b.p );
   HG_CHECK_HIP( hipGetLastError() );
   return b.p;
}

// x/|x| of the owned boundary DoFs of a lattice: the outer normal of a sphere
// centred at the origin, which the shell map keeps (it only scales radii)
const double* boundaryNormals( Context* ctx, Storage& st, Lattice& lat )
{
   if ( lat.bndNormal.p )
      return lat.bndNormal.p;
   const Topology&       t  = st.topo;
   const int64_t         mm = lat.mm;
   std::vector< double > n( 3 * size_t( lat.nb ), 0.0 );
   std::vector< char >   done( size_t( lat.nb ), 0 );
   for ( int c = 0; c < t.nc; ++c )
   {
      const double* v[4];
      for ( int k = 0; k < 4; ++k )
         v[k] = &t.X[3 * t.cv[c][k]];
      for ( int64_t z = 0; z <= mm; ++z )
         for ( int64_t y = 0; y + z <= mm; ++y )
            for ( int64_t x = 0; x + y + z <= mm; x = ( y > 0 && z > 0 && x == 0 && mm - y - z > 0 ) ? mm - y - z : x + 1 )
            {
               const int64_t id = lat.num.locate( t, c, x, y, z );
               if ( id >= lat.nb || done[id] )
                  continue;
               done[id] = 1;
               double p[3], r = 0.0;
               for ( int d = 0; d < 3; ++d )
               {
                  p[d] = v[0][d] + ( double( x ) / double( mm ) ) * ( v[1][d] - v[0][d] ) +
                         ( double( y ) / double( mm ) ) * ( v[2][d] - v[0][d] ) +
                         ( double( z ) / double( mm ) ) * ( v[3][d] - v[0][d] );
                  r += p[d] * p[d];
               }
               r = std::sqrt( r );
               for ( int d = 0; d < 3; ++d )
                  n[3 * id + d] = p[d] / r;
            }
   }
   lat.bndNormal.upload( ctx, n );
   return lat.bndNormal.p;
}

void copyInto( Context* ctx, const double* src, Function& f, int L, size_t n )
{
   HG_CHECK_HIP( hipMemcpyAsync( f.ptr( L ), src, n * sizeof( double ), hipMemcpyDeviceToDevice, ctx->stream ) );
}

} // namespace
} // namespace hg

using namespace hg;

extern "C" {

int hg_stokes_create( hg_ctx* h, hg_handle s, int minLevel, int maxLevel, double viscC0, double viscC1, hg_handle* out )
{
   return hg_guard( h, [&]( Context* ctx ) {
      if ( !out || minLevel < 0 || maxLevel < minLevel || maxLevel > 9 || !std::isfinite( viscC0 ) ||
           !std::isfinite( viscC1 ) )
         throw Error( HG_ERR_ARG, "invalid Stokes operator parameters" );
      // uploaded once per process (several host threads may create operators at once)
      static std::once_flag quadOnce;
      std::call_once( quadOnce, [] {
         double q4[9][4], q4m[9][4];
         for ( int q = 0; q < 9; ++q )
            for ( int k = 0; k < 4; ++k )
            {
               q4[q][k]  = 4.0 * kSQP[q][k];
               q4m[q][k] = 4.0 * kSQP[q][k] - 1.0;
            }
         HG_CHECK_HIP( hipMemcpyToSymbol( HIP_SYMBOL( cSQ4 ), q4, sizeof( q4 ) ) );
         HG_CHECK_HIP( hipMemcpyToSymbol( HIP_SYMBOL( cSQ4m ), q4m, sizeof( q4m ) ) );
         HG_CHECK_HIP( hipMemcpyToSymbol( HIP_SYMBOL( cSQL ), kSQP, sizeof( kSQP ) ) );
         HG_CHECK_HIP( hipMemcpyToSymbol( HIP_SYMBOL( cSQW ), kSQW, sizeof( kSQW ) ) );
         float f4[9][4], f4m[9][4], fl[9][4], fw[9];
         for ( int q = 0; q < 9; ++q )
         {
            for ( int k = 0; k < 4; ++k )
            {
               f4[q][k]  = float( q4[q][k] );
               f4m[q][k] = float( q4m[q][k] );
               fl[q][k]  = float( kSQP[q][k] );
            }
            fw[q] = float( kSQW[q] );
         }
         HG_CHECK_HIP( hipMemcpyToSymbol( HIP_SYMBOL( cSQ4f ), f4, sizeof( f4 ) ) );
         HG_CHECK_HIP( hipMemcpyToSymbol( HIP_SYMBOL( cSQ4mf ), f4m, sizeof( f4m ) ) );
         HG_CHECK_HIP( hipMemcpyToSymbol( HIP_SYMBOL( cSQLf ), fl, sizeof( fl ) ) );
         HG_CHECK_HIP( hipMemcpyToSymbol( HIP_SYMBOL( cSQWf ), fw, sizeof( fw ) ) );
         const std::vector< int32_t > pairs = diagonalPairs(), boxp = diagonalBoxPoints();
         HG_CHECK_HIP( hipMemcpyToSymbol( HIP_SYMBOL( cDiagPairs ), pairs.data(), sizeof( int32_t ) * 64 ) );
         HG_CHECK_HIP( hipMemcpyToSymbol( HIP_SYMBOL( cDiagBox ), boxp.data(), sizeof( int32_t ) * kDiagBoxP ) );
      } );
      Storage& st = ctx->storage( s );
      auto     op = std::make_unique< StokesOperator >();
      op->st      = &st;
      op->minL    = minLevel;
      op->maxL    = maxLevel;
      op->c0      = viscC0;
      op->c1      = viscC1;
      const std::vector< P2CellGeom > tg = tileGeometry( st.topo );
      for ( int L = minLevel; L <= maxLevel; ++L )
      {
         std::vector< P2CellGeom > gl = tg;
         tileGeometryLevel( gl, int64_t( 1 ) << L, kSQP, 9 );
         op->tgeom[L].upload( ctx, gl );
         op->tgeom32[L].upload( ctx, toFloat( gl ) );
         st.lattice( ctx, L );
         st.lattice( ctx, L + 1 );
      }
      *out                  = ctx->nextHandle++;
      ctx->operators[*out] = std::move( op );
   } );
}

int hg_stokes_apply( hg_ctx* h, hg_handle op, const hg_handle* src, const hg_handle* dst, int level, int flag, int mask,
                     int update )
{
   return hg_guard( h, [&]( Context* ctx ) {
      if ( update != HG_REPLACE && update != HG_ADD )
         throw Error( HG_ERR_ARG, "invalid update type" );
      if ( !src || !dst )
         throw Error( HG_ERR_ARG, "null function list" );
      Function* s[4] = { nullptr, nullptr, nullptr, nullptr };
      Function* d[4] = { nullptr, nullptr, nullptr, nullptr };
      for ( int k = 0; k < 4; ++k )
      {
         const bool needS = k < 3 ? ( mask & 5 ) : ( mask & 10 );
         const bool needD = k < 3 ? ( mask & 3 ) : ( mask & 12 );
         if ( needS )
            s[k] = &ctx->function( src[k] );
         if ( needD )
            d[k] = &ctx->function( dst[k] );
      }
      stokesApply( ctx, ctx->op< StokesOperator >( op ), s, d, level, flag, mask, update );
   } );
}

int hg_stokes_velocity_inverse_diagonal( hg_ctx* h, hg_handle op, int level, const hg_handle* dst )
{
   return hg_guard( h, [&]( Context* ctx ) {
      StokesOperator& o = ctx->op< StokesOperator >( op );
      if ( !dst )
         throw Error( HG_ERR_ARG, "null function list" );
      const auto& inv = velocityInverseDiagonal( ctx, o, level );
      Lattice&    lat = o.st->lattice( ctx, level + 1 );
      for ( int c = 0; c < 3; ++c )
      {
         Function& f = ctx->function( dst[c] );
         checkVelocity( o, f, level );
         copyInto( ctx, inv[c].p, f, level, size_t( lat.nstore ) );
      }
   } );
}

int hg_stokes_pressure_diagonal( hg_ctx* h, hg_handle op, int level, int kind, hg_handle dst )
{
   return hg_guard( h, [&]( Context* ctx ) {
      StokesOperator& o = ctx->op< StokesOperator >( op );
      if ( kind != 0 && kind != 1 )
         throw Error( HG_ERR_ARG, "kind must be 0 (PSPG inverse diagonal) or 1 (inverse lumped mass)" );
      Function& f = ctx->function( dst );
      checkPressure( o, f, level );
      const double* inv = affineInverseDiagonal( ctx, o, level, kind );
      copyInto( ctx, inv, f, level, size_t( o.st->lattice( ctx, level ).nstore ) );
   } );
}

int hg_p2_project_normal( hg_ctx* h, const hg_handle* u, int level, int flag )
{
   return hg_guard( h, [&]( Context* ctx ) {
      if ( !u )
         throw Error( HG_ERR_ARG, "null function list" );
      // the normal is defined on boundary DoFs only (P2ProjectNormalOperator aborts on a non-boundary face)
      if ( flag & ( kInner | ~kAll ) )
         throw Error( HG_ERR_ARG, "normal projection flag must select boundary types only" );
      Function* f[3];
      for ( int c = 0; c < 3; ++c )
      {
         f[c] = &ctx->function( u[c] );
         if ( f[c]->off != 1 || f[c]->lv != 0 || f[c]->dtype != f[0]->dtype || f[c]->st != f[0]->st ||
              level < f[c]->minL || level > f[c]->maxL )
            throw Error( HG_ERR_ARG, "normal projection needs three P2 functions of one storage and one type" );
      }
      Storage& st  = *f[0]->st;
      Lattice& lat = st.lattice( ctx, level + 1 );
      if ( lat.nb == 0 )
         return;
      const double* nrm = boundaryNormals( ctx, st, lat );
      dispatchType( f[0]->dtype, [&]( auto tag ) {
         using T = decltype( tag );
         kProjectNormal< T ><<< gridFor( lat.nb ), kBlock, 0, ctx->stream >>>(
             lat.nb, lat.nc * lat.sc, lat.bndFlag.p, flag, nrm, (T*) f[0]->ptr( level ), (T*) f[1]->ptr( level ),
             (T*) f[2]->ptr( level ) );
      } );
      HG_CHECK_HIP( hipGetLastError() );
   } );
}

int hg_function_sum( hg_ctx* h, hg_handle fn, int level, int flag, double* out )
{
   return hg_guard( h, [&]( Context* ctx ) {
      Function& f = ctx->function( fn );
      if ( !out || f.lv != 0 || level < f.minL || level > f.maxL )
         throw Error( HG_ERR_ARG, "sum needs a single-vector function and a level in its range" );
      Lattice& lat = f.lat( ctx, level );
      if ( !lat.ones.p )
      {
         lat.ones.alloc( ctx, lat.nstore );
         kFillRange< double ><<< gridFor( lat.nstore ), kBlock, 0, ctx->stream >>>( lat.nstore, lat.ones.p, 1.0 );
         HG_CHECK_HIP( hipGetLastError() );
      }
      if ( f.dtype != 0 )
         throw Error( HG_ERR_UNSUPPORT, "sum supports FP64 functions" );
      *out = dotDevice( ctx, lat, f.ptr( level ), lat.ones.p, 0, flag );
   } );
}

int hg_function_add_const( hg_ctx* h, hg_handle fn, double value, int level, int flag )
{
   return hg_guard( h, [&]( Context* ctx ) {
      Function& f = ctx->function( fn );
      if ( f.lv != 0 || f.dtype != 0 || level < f.minL || level > f.maxL )
         throw Error( HG_ERR_ARG, "add of a constant needs a single-vector FP64 function and a level in its range" );
      Lattice&      l = f.lat( ctx, level );
      const int64_t n = ( flag & kInner ? l.nc * l.sc : 0 ) + l.nb;
      if ( n == 0 )
         return;
      kAddConst<<< gridFor( n ), kBlock, 0, ctx->stream >>>( l.nc * l.sc, l.nb, l.bndFlag.p, flag, value,
                                                             (double*) f.ptr( level ) );
      HG_CHECK_HIP( hipGetLastError() );
   } );
}

int hg_function_invert( hg_ctx* h, hg_handle fn, int level, int flag )
{
   return hg_guard( h, [&]( Context* ctx ) {
      Function& f = ctx->function( fn );
      if ( f.lv != 0 || f.dtype != 0 || level < f.minL || level > f.maxL )
         throw Error( HG_ERR_ARG, "invertElementwise needs a single-vector FP64 function and a level in its range" );
      Lattice&      l = f.lat( ctx, level );
      const int64_t n = ( flag & kInner ? l.nc * l.sc : 0 ) + l.nb;
      if ( n == 0 )
         return;
      kInvertFlagged<<< gridFor( n ), kBlock, 0, ctx->stream >>>( l.nc * l.sc, l.nb, l.bndFlag.p, flag,
                                                                  (double*) f.ptr( level ) );
      HG_CHECK_HIP( hipGetLastError() );
   } );
}

} // extern "C"

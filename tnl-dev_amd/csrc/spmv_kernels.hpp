// Row kernels of the sparse product over every segment format and the launch that picks one for a
// matrix, written for CDNA4 wavefront-64 execution; instantiated with the plain keeper by spmv.hip
// and with the solvers' fused keepers by krylov.hip.  SpMV is HBM-bound (about 0.14 flop per byte
// in FP64), so every kernel is organised around coalesced streaming of values and column
// indexes; x is gathered through L2 / MALL.
//
// Reference semantics: SparseMatrixView::vectorProduct (Matrices/SparseMatrixView.hpp:390-491):
// fetch = values[g] * x[columns[g]], padding (column -1) contributes nothing, keeper chosen
// from (alpha, beta).  Each format's Host traversal sums a row left to right in local
// order; the one-lane-per-row kernels here (CSR scalar, Ellpack, SlicedEllpack) keep that
// order and round each product and sum separately, so they reproduce the Host result bit
// for bit; the cooperative kernels reassociate the row sum.
//
// A kernel asks its keeper for everything beside the matrix: closed() (a plain product's gate), shut()
// (the gate of a fused product that has nothing to fold; the same for the whole grid), prefetch() and
// begin() (called by every thread before the first at(); begin: false, for the whole grid alike but for
// a gate that is being closed, when there is nothing to do), at( x, c ) (entry c of the operand),
// keep( row, sum ) (once per row, by one lane) and finish() (called by every thread after the rows).  The
// kernels of short rows call begin() behind the loads of their first elements, which do not depend on it.
#pragma once

#include "spmv.hpp"
#include "rowdist.hpp"

#include <type_traits>

namespace tnlhip {

template< bool EXACT, typename A >
__device__ __forceinline__ A madd( A acc, A a, A b )
{
   if constexpr( EXACT )
      return mulAddExact( acc, a, b );
   else
      return acc + a * b;
}

// closed(), prefetch() and begin() in one; the answer is the workgroup's, whose waves may see a gate that is just
// being closed differently and have barriers ahead of them
template< typename Keep >
__device__ __forceinline__ bool openKeeper( Keep& keep )
{
   if constexpr( Keep::kPlain )
      return ! keep.closed();
   else {
      if( keep.shut() )
         return false;
      keep.prefetch();
      return Keep::kStored || __syncthreads_and( keep.begin() );
   }
}

// Streaming loads of the matrix arrays bypass the caches' normal retention (non-temporal),
// so the 256 MiB MALL and the L2 keep x, which is gathered many times.
__device__ __forceinline__ int32_t ldnt( const int32_t* p ) { return __builtin_nontemporal_load( p ); }
__device__ __forceinline__ double ldnt( const double* p ) { return __builtin_nontemporal_load( p ); }
__device__ __forceinline__ float ldnt( const float* p ) { return __builtin_nontemporal_load( p ); }
__device__ __forceinline__ bf16 ldnt( const bf16* p )
{
   return __ushort_as_bfloat16( __builtin_nontemporal_load( reinterpret_cast< const unsigned short* >( p ) ) );
}

// Whether a kernel leaves out the loads of a chunk that lie beyond the end of its rows (by branches that
// whole waves or lane pairs take) instead of re-reading the last slot: from `least` value bytes on.  The
// branches keep narrow loads from being issued together.  us, re-read / left out, at 160^3 and 2000^2:
// staged CSR FP64 76.9 61.6 / 74.9 53.8, FP32 56.9 43.0 / 57.4 40.2, BF16 52.5 40.0 / 69.5 48.9;
// CSRAdaptive FP64 79.9 57.7 / 78.0 56.5, FP32 61.9 43.7 / 60.9 42.1 but on 40-entry rows 113 / 129, BF16
// 56.9 39.4 / 71.2 51.3; ChunkedEllpack FP64 71.1 59.6 / 68.5 54.0, FP32 46.3 38.4 / 50.3 38.4; BiEllpack FP64
// 77.1 68.7 / 72.1 56.3, FP32 48.9 47.1 / 46.5 41.3, BF16 42.3 42.6 / 58.6 49.1.
// An operand that is formed where it is gathered keeps the straight line (64^3 CG, SlicedEllpack: 14.8 us per iteration
// against 18.0).
template< typename V, typename Keep, int least >
constexpr bool kSkipSlots = Keep::kStored && (int) sizeof( V ) >= least;

__device__ __forceinline__ int64_t logicalBlock( int remap )
{
   return logicalBlockOf( blockIdx.x, gridDim.x, remap );
}

template< int P >
__device__ __forceinline__ RowSeq rowSequence( int64_t base, int64_t last, int64_t per, int dist )
{
   return rowSequenceAt< P >( base, last, per, dist, LaunchIndex{ blockIdx.x, gridDim.x, blockDim.x, threadIdx.x } );
}

// ------------------------------------------------------------------ CSR: G lanes per row

// G = 1: CSRScalar (one lane per row, exact Host order); G = 2..32: CSRLight / CSRHybrid;
// G = 64: CSRVector (a whole wavefront per row).  Groups of G lanes stride over the row
// with contiguous loads, then reduce across the group with cross-lane shuffles.  Every group
// keeps R rows in flight (rows r, r + stride, ...): their offsets, first chunk of columns /
// values and the gathers of x are issued together, so short rows do not serialize on the
// offsets -> columns -> x latency chain.  Each lane still sums its elements of a row in
// increasing order, so the result does not depend on R.
template< int G, int R, bool EXACT, typename V, typename A, typename Y, typename Keep >
__device__ __forceinline__ void csrGroupedRows( const int32_t* __restrict__ off,
                                                const int32_t* __restrict__ col,
                                                const V* __restrict__ val, const Y* __restrict__ x,
                                                Keep& keep, int32_t first, int32_t last )
{
   constexpr int GPB = 256 / G;
   const int gl = threadIdx.x % G;
   const int64_t stride = (int64_t) gridDim.x * GPB;
   if constexpr( R == 1 ) {
      for( int64_t r = first + (int64_t) blockIdx.x * GPB + threadIdx.x / G; r < last; r += stride ) {
         const int32_t b = off[ r ], e = off[ r + 1 ];
         A s = 0;
         for( int32_t k = b + gl; k < e; k += G ) {
            const int32_t c = col[ k ];
            if( c >= 0 )
               s = madd< EXACT >( s, toCompute( val[ k ], A() ), (A) keep.at( x, c ) );
         }
         if constexpr( G > 1 )
            s = groupSum< G >( s );
         if( gl == 0 )
            keep( r, s );
      }
      return;
   }
   for( int64_t r0 = first + (int64_t) blockIdx.x * GPB + threadIdx.x / G; r0 < last; r0 += stride * R ) {
      int32_t b[ R ], e[ R ];
#pragma unroll
      for( int j = 0; j < R; j++ ) {
         const int64_t r = r0 + j * stride;
         const bool valid = r < last;
         b[ j ] = valid ? off[ r ] : 0;
         e[ j ] = valid ? off[ r + 1 ] : 0;
      }
      int32_t c[ R ];
      V v[ R ];
#pragma unroll
      for( int j = 0; j < R; j++ ) {
         const int32_t k = b[ j ] + gl;
         const bool in = k < e[ j ];
         c[ j ] = in ? col[ k ] : -1;
         v[ j ] = in ? val[ k ] : V( 0 );
      }
      Y xv[ R ];
#pragma unroll
      for( int j = 0; j < R; j++ )
         xv[ j ] = keep.at( x, c[ j ] < 0 ? 0 : c[ j ] );
      A s[ R ];
#pragma unroll
      for( int j = 0; j < R; j++ ) {
         s[ j ] = 0;
         if( c[ j ] >= 0 )
            s[ j ] = madd< EXACT >( s[ j ], toCompute( v[ j ], A() ), (A) xv[ j ] );
         for( int32_t k = b[ j ] + gl + G; k < e[ j ]; k += G ) {
            const int32_t ck = col[ k ];
            if( ck >= 0 )
               s[ j ] = madd< EXACT >( s[ j ], toCompute( val[ k ], A() ), (A) keep.at( x, ck ) );
         }
      }
#pragma unroll
      for( int j = 0; j < R; j++ ) {
         A t = s[ j ];
         if constexpr( G > 1 )
            t = groupSum< G >( t );
         const int64_t r = r0 + j * stride;
         if( gl == 0 && r < last )
            keep( r, t );
      }
   }
}

template< int G, int R, bool EXACT, typename V, typename A, typename Y, typename Keep >
__global__ __launch_bounds__( 256 ) void csrGroupedKernel( const int32_t* __restrict__ off,
                                                           const int32_t* __restrict__ col,
                                                           const V* __restrict__ val, const Y* __restrict__ x,
                                                           Keep keep, int32_t first, int32_t last )
{
   if( ! openKeeper( keep ) )
      return;
   csrGroupedRows< G, R, EXACT, V, A, Y, Keep >( off, col, val, x, keep, first, last );
   keep.finish();
}

// ------------------------------------------------------------------ CSR scalar, staged

// CSRScalar (one lane per row, Kernels/CSRScalarKernel.hpp) with the elements staged through
// LDS.  Each wavefront owns 64 consecutive rows.  When their elements fit the wave's LDS slice
// (K x 64 of them: 512 FP64 or 1024 FP32 products), the wave loads them with coalesced loads,
// kStageLoads per lane in flight per round, stores each rounded product in LDS (a padding slot
// stores -0.0, the identity of IEEE addition, so adding it equals skipping it), and every lane
// then sums its own row left to right out of LDS: the Host traversal's result bit for bit, at
// streaming speed.  Waves whose rows hold more elements walk their rows in global memory, one
// lane per row, with the same arithmetic.  One wave per 64 rows and no grid-stride loop: at
// 160^3 FP64 neither a persistent grid that prefetches the next block's offsets (78-92 us by
// grid size) nor two 64-row blocks per wave (83 us; FP32 61.1 against 59.4 us) beat it (79 us).
constexpr int kStageLoads = 8;
constexpr int kShortRow = 8;  // mean row length up to which every CSR kernel takes the staged path

template< int K, typename V, typename A, typename Y, typename Keep >
__device__ __forceinline__ void csrScalarStagedRows( const int32_t* __restrict__ off,
                                                     const int32_t* __restrict__ col,
                                                     const V* __restrict__ val, const Y* __restrict__ x,
                                                     Keep& keep, int32_t first, int32_t last,
                                                     int remap )
{
   __shared__ A lds[ 4 ][ K * kWave ];
   const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
   const int64_t r0 = first + ( logicalBlock( remap ) * 4 + wave ) * kWave;
   const bool any = r0 < last;  // uniform over the wave
   if constexpr( Keep::kPlain ) {
      if( ! any )  // a plain product has no workgroup barrier
         return;
   }
   const int64_t r = r0 + lane;
   const int32_t used = any ? (int32_t) min( (int64_t) kWave, last - r0 ) : 0;  // rows of this wave
   const bool mine = lane < used;
   const int32_t rb = mine ? off[ r ] : 0;
   const int32_t re = mine ? off[ r + 1 ] : 0;
   const int32_t b = __shfl( rb, 0, kWave );
   // (a plain product's wave has rows)
   const int32_t size = __shfl( re, Keep::kPlain ? used - 1 : max( used, 1 ) - 1, kWave ) - b;
   auto loadRound = [ & ]( int32_t e0, int32_t ( &c )[ kStageLoads ], V ( &v )[ kStageLoads ] ) {
#pragma unroll
      for( int k = 0; k < kStageLoads; k++ ) {
         c[ k ] = -1;
         v[ k ] = V( 0.0f );
         if( ! kSkipSlots< V, Keep, 8 > || e0 + k * kWave < size ) {  // uniform over the wave
            const int32_t g = min( e0 + lane + k * kWave, size - 1 );
            c[ k ] = ldnt( col + b + g );
            v[ k ] = ldnt( val + b + g );
         }
      }
   };
   int32_t c0[ kStageLoads ];  // a fused product's first round, loaded before begin()
   V v0[ kStageLoads ];
   if constexpr( ! Keep::kPlain ) {
      if( size > 0 )
         loadRound( 0, c0, v0 );
      if( ! keep.begin() || ! any )
         return;
   }
   if( size <= 0 ) {
      if( mine )
         keep( r, (A) 0 );
      return;
   }
   if( size <= K * kWave ) {
      // rounds of kStageLoads loads per lane (one for FP64, up to two for FP32) keep the
      // registers, hence the waves per SIMD, of the one-round case
#pragma unroll
      for( int q = 0; q < K / kStageLoads; q++ ) {
         const int32_t e0 = q * kStageLoads * kWave;
         if( e0 >= size )  // uniform over the wave
            break;
         int32_t c[ kStageLoads ];
         V v[ kStageLoads ];
         if( Keep::kPlain || q > 0 )
            loadRound( e0, c, v );
         else {
#pragma unroll
            for( int k = 0; k < kStageLoads; k++ ) {
               c[ k ] = c0[ k ];
               v[ k ] = v0[ k ];
            }
         }
         Y xv[ kStageLoads ];
#pragma unroll
         for( int k = 0; k < kStageLoads; k++ )
            xv[ k ] = c[ k ] >= 0 ? keep.at( x, c[ k ] ) : Y( 0 );  // x may be empty when every slot is padding
#pragma unroll
         for( int k = 0; k < kStageLoads; k++ ) {
            const int32_t g = e0 + lane + k * kWave;
            if( g < size )
               lds[ wave ][ g ] = c[ k ] >= 0 ? toCompute( v[ k ], A() ) * (A) xv[ k ] : (A) -0.0;
         }
      }
      waveSync();
      if( mine ) {
         A s = 0;
         for( int32_t k = rb - b; k < re - b; k++ )
            s += lds[ wave ][ k ];
         keep( r, s );
      }
      return;
   }
   if( mine ) {
      A s = 0;
      for( int32_t k = rb; k < re; k++ ) {
         const int32_t ck = col[ k ];
         if( ck >= 0 )
            s = mulAddExact( s, toCompute( val[ k ], A() ), (A) keep.at( x, ck ) );
      }
      keep( r, s );
   }
}

template< int K, typename V, typename A, typename Y, typename Keep >
__global__ __launch_bounds__( 256 ) void csrScalarStagedKernel( const int32_t* __restrict__ off,
                                                                const int32_t* __restrict__ col,
                                                                const V* __restrict__ val, const Y* __restrict__ x,
                                                                Keep keep, int32_t first, int32_t last,
                                                                int remap )
{
   if constexpr( Keep::kPlain ) {
      if( keep.closed() )
         return;
   }
   else {
      if( keep.shut() )
         return;
      keep.prefetch();
   }
   csrScalarStagedRows< K, V, A, Y, Keep >( off, col, val, x, keep, first, last, remap );
   keep.finish();
}

// ------------------------------------------------------------------ CSR-Adaptive

// One wavefront per block descriptor (the scheme of Kernels/CSRAdaptiveKernelView.hpp:33-170,
// with wave64 budgets).  STREAM: the wave loads the elements of several short rows with fully
// coalesced loads (rounds of kStageLoads per lane in flight), keeps the products in
// its own LDS slice, then every lane sums whole rows out of LDS.  VECTOR: one row per wave.
// LONG: one row split over the waves left in the workgroup, partial sums combined in LDS in
// a fixed order.  One descriptor per wave and no grid-stride loop, so the single workgroup
// barrier (needed only by LONG rows) is uniform.
constexpr int kPreSets = 4;  // STREAM blocks: offsets of the first 4 x 64 rows are preloaded

template< int STREAM, typename V, typename A, typename Y, typename Keep >
__global__ __launch_bounds__( 256 ) void csrAdaptiveKernel( int32_t nblocks, const int4* __restrict__ desc,
                                                            const int32_t* __restrict__ off,
                                                            const int32_t* __restrict__ col,
                                                            const V* __restrict__ val, const Y* __restrict__ x,
                                                            Keep keep, int remap )
{
   if( ! openKeeper( keep ) )
      return;
   constexpr int K = STREAM / kWave;
   __shared__ A lds[ 4 ][ STREAM ];
   __shared__ A longPart[ 4 ];
   const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
   // remap: XCD x (blockIdx % 8) takes the x-th eighth of the descriptors, in order
   const int64_t lb = remap ? logicalBlock( 1 ) : blockIdx.x;
   const int64_t di = lb * 4 + wave;
   const bool active = di < nblocks;
   const int4 d = active ? desc[ di ] : make_int4( BLOCK_VECTOR, 0, 0, 0 );
   const int type = d.x & 0xff;
   const int32_t firstRow = d.y;
   const int32_t b = active ? off[ firstRow ] : 0;
   A vsum = 0;
   if( active && type == BLOCK_STREAM && d.z == 0 ) {
      for( int32_t r = lane; r < d.w; r += kWave )  // a block of empty rows
         keep( firstRow + r, (A) 0 );
   }
   else if( active && type == BLOCK_STREAM ) {
      const int32_t size = d.z;
      // offsets of the first kPreRows rows of the block, fetched alongside the element stream
      int32_t rbPre[ kPreSets ];
#pragma unroll
      for( int q = 0; q < kPreSets; q++ ) {
         const int32_t r = lane + q * kWave;
         rbPre[ q ] = r <= d.w ? off[ firstRow + r ] : 0;
      }
      // rounds of kStageLoads loads per lane (one for FP64, up to two for FP32 blocks of 1024
      // elements): the FP32 kernel keeps the FP64 kernel's registers and waves per SIMD
#pragma unroll
      for( int q = 0; q < K / kStageLoads; q++ ) {
         const int32_t e0 = q * kStageLoads * kWave;
         if( e0 >= size )  // uniform over the wave
            break;
         int32_t c[ kStageLoads ];
         V v[ kStageLoads ];
#pragma unroll
         for( int k = 0; k < kStageLoads; k++ ) {
            c[ k ] = -1;
            v[ k ] = V( 0.0f );
            if( ! kSkipSlots< V, Keep, 8 > || e0 + k * kWave < size ) {  // uniform over the wave
               const int32_t e = min( e0 + lane + k * kWave, size - 1 );
               c[ k ] = ldnt( col + b + e );
               v[ k ] = ldnt( val + b + e );
            }
         }
         Y xv[ kStageLoads ];
#pragma unroll
         for( int k = 0; k < kStageLoads; k++ ) {
            xv[ k ] = Y( 0 );
            if( ! kSkipSlots< V, Keep, 8 > || e0 + k * kWave < size )
               xv[ k ] = keep.at( x, c[ k ] < 0 ? 0 : c[ k ] );
         }
#pragma unroll
         for( int k = 0; k < kStageLoads; k++ ) {
            const int32_t e = e0 + lane + k * kWave;
            if( e < size )
               lds[ wave ][ e ] = c[ k ] >= 0 ? toCompute( v[ k ], A() ) * (A) xv[ k ] : (A) 0;
         }
      }
      waveSync();
#pragma unroll
      for( int q = 0; q < kPreSets; q++ ) {
         // row r = lane + 64 q ends where row r + 1 starts: the next lane's offset, or the
         // first of the next set for lane 63
         const int32_t nextLane = __shfl( rbPre[ q ], ( lane + 1 ) % kWave, kWave );
         const int32_t nextSet = q + 1 < kPreSets ? __shfl( rbPre[ q + 1 < kPreSets ? q + 1 : q ], 0, kWave ) : 0;
         const int32_t r = lane + q * kWave;
         if( r < d.w ) {
            const int32_t rb = rbPre[ q ] - b;
            const int32_t re = ( lane + 1 < kWave ? nextLane : q + 1 < kPreSets ? nextSet : off[ firstRow + r + 1 ] ) - b;
            A s = 0;
            for( int32_t k = rb; k < re; k++ )
               s += lds[ wave ][ k ];
            keep( firstRow + r, s );
         }
      }
      for( int32_t r = lane + kPreSets * kWave; r < d.w; r += kWave ) {
         const int32_t rb = off[ firstRow + r ] - b;
         const int32_t re = off[ firstRow + r + 1 ] - b;
         A s = 0;
         for( int32_t k = rb; k < re; k++ )
            s += lds[ wave ][ k ];
         keep( firstRow + r, s );
      }
   }
   else if( active ) {
      const int32_t e = off[ firstRow + 1 ];
      const int32_t widx = type == BLOCK_LONG ? ( d.x >> 8 ) & 0xff : 0;
      const int32_t wcnt = type == BLOCK_LONG ? ( d.x >> 16 ) & 0xff : 1;
      A p = 0;
      for( int32_t k = b + widx * kWave + lane; k < e; k += kWave * wcnt ) {
         const int32_t c = ldnt( col + k );
         if( c >= 0 )
            p += toCompute( ldnt( val + k ), A() ) * (A) keep.at( x, c );
      }
      vsum = groupSum< kWave >( p );
      if( type == BLOCK_VECTOR && lane == 0 )
         keep( firstRow, vsum );
      if( type == BLOCK_LONG && lane == 0 )
         longPart[ wave ] = vsum;
   }
   __syncthreads();
   if( active && type == BLOCK_LONG && ( ( d.x >> 8 ) & 0xff ) == 0 && lane == 0 ) {
      const int32_t wcnt = ( d.x >> 16 ) & 0xff;
      A s = 0;
      for( int32_t w = 0; w < wcnt; w++ )
         s += longPart[ wave + w ];
      keep( firstRow, s );
   }
   keep.finish();
}

// ------------------------------------------------------------------ Ellpack / SlicedEllpack

// One or two adjacent rows per lane, column-major storage: consecutive lanes read consecutive
// addresses for every local index (EllpackView.hpp:361-378, SlicedEllpackView.hpp:248-290).  The
// slots of a row are read eight at a time, their loads in flight together (24 with the gathers of
// x); the sum still runs left to right over the non-padding slots only, which is the Host result
// bit for bit.  What becomes of a chunk's slots beyond the row's end: paddedRows.  Each workgroup
// owns `rowsPerBlock` consecutive rows.
constexpr int kChunk = 8;
constexpr int kRowsInFlight = 2;  // rows per lane per iteration of the padded kernels

// Two vertically adjacent slots (rows r, r+1 at one local index) are one aligned 8-byte
// index load and one 2-element value load.
typedef double double2v __attribute__( ( ext_vector_type( 2 ) ) );
typedef float float2v __attribute__( ( ext_vector_type( 2 ) ) );
template< typename V >
struct Pair;
template<>
struct Pair< double >
{
   using T = double2v;
};
template<>
struct Pair< float >
{
   using T = float2v;
};
template<>
struct Pair< bf16 >
{
   using T = unsigned int;
};
__device__ __forceinline__ void split( double2v p, double& a, double& b )
{
   a = p.x;
   b = p.y;
}
__device__ __forceinline__ void split( float2v p, float& a, float& b )
{
   a = p.x;
   b = p.y;
}
__device__ __forceinline__ void split( unsigned int p, bf16& a, bf16& b )
{
   a = __ushort_as_bfloat16( (unsigned short) ( p & 0xffff ) );
   b = __ushort_as_bfloat16( (unsigned short) ( p >> 16 ) );
}
template< typename V >
__device__ __forceinline__ typename Pair< V >::T ldnt2( const V* p )
{
   using P = typename Pair< V >::T;
   return __builtin_nontemporal_load( reinterpret_cast< const P* >( p ) );
}
__device__ __forceinline__ int2 ldnt2( const int32_t* p )
{
   const long long v = __builtin_nontemporal_load( reinterpret_cast< const long long* >( p ) );
   return make_int2( (int32_t) ( v & 0xffffffff ), (int32_t) ( v >> 32 ) );
}

// One or two (PAIR) rows per lane.  Slot index of row r at local index l: base( r ) + step * l.
// With SKIP a lane pair neither loads nor gathers a chunk's slots beyond the row's width (whole waves skip
// them): re-reading the last slot instead costs a 5-wide row 3 of 8 loads (FP64 SlicedEllpack 160^3
// 77.1 -> 69.6 us, 128^3 41.2 -> 37.0, 2000^2 69.9 -> 51.6).  The branches cost registers (72 -> 96 in FP64, 7
// -> 5 waves per SIMD), so rows of more than kSkipSlotsUpTo slots on average, whose chunks are mostly full,
// re-read (FP64 SlicedEllpack, re-read / left out: 27 slots 49.5 / 45.6 us, 30 75.6 / 76.3, 34 103.3 / 108.8,
// 73 173.9 / 182.8).  One row per lane re-reads x[ 0 ] for such slots, and its last row the last slot.
constexpr int kSkipSlotsUpTo = 32;
template< bool PAIR, bool SKIP, typename V, typename A, typename Y, typename Keep, typename Slots >
__device__ __forceinline__ void paddedRows( const Slots& slots, const int32_t* __restrict__ col,
                                            const V* __restrict__ val, const Y* __restrict__ x, Keep& keep,
                                            int32_t first, RowSeq seq )
{
   if constexpr( ! PAIR ) {
      // kRowsInFlight rows of the sequence per lane (r, r + step, ...), their loads issued
      // together; each row keeps its own left-to-right sum
      constexpr int Q = kRowsInFlight;
      const int64_t step = slots.step();
      int64_t r = seq.start;
      for( ; r + ( Q - 1 ) * seq.step < seq.end; r += Q * seq.step ) {
         int64_t b[ Q ];
         int32_t w[ Q ];
         int32_t wmax = 0;
#pragma unroll
         for( int q = 0; q < Q; q++ ) {
            b[ q ] = slots.base( r + q * seq.step );
            w[ q ] = slots.width( r + q * seq.step );
            wmax = max( wmax, w[ q ] );
         }
         A s[ Q ];
#pragma unroll
         for( int q = 0; q < Q; q++ )
            s[ q ] = 0;
         for( int32_t l0 = 0; l0 < wmax; l0 += kChunk ) {
            int32_t c[ Q ][ kChunk ];
            V v[ Q ][ kChunk ];
#pragma unroll
            for( int q = 0; q < Q; q++ )
#pragma unroll
               for( int j = 0; j < kChunk; j++ ) {
                  const bool in = l0 + j < w[ q ];
                  const int64_t g = b[ q ] + step * ( l0 + j );
                  c[ q ][ j ] = in ? ldnt( col + g ) : -1;
                  v[ q ][ j ] = in ? ldnt( val + g ) : V( 0 );
               }
            Y xv[ Q ][ kChunk ];
#pragma unroll
            for( int q = 0; q < Q; q++ )
#pragma unroll
               for( int j = 0; j < kChunk; j++ )
                  xv[ q ][ j ] = keep.at( x, c[ q ][ j ] < 0 ? 0 : c[ q ][ j ] );
#pragma unroll
            for( int q = 0; q < Q; q++ )
#pragma unroll
               for( int j = 0; j < kChunk; j++ )
                  if( c[ q ][ j ] >= 0 )
                     s[ q ] = mulAddExact( s[ q ], toCompute( v[ q ][ j ], A() ), (A) xv[ q ][ j ] );
         }
#pragma unroll
         for( int q = 0; q < Q; q++ )
            if( r + q * seq.step >= first )
               keep( r + q * seq.step, s[ q ] );
      }
      seq.start = r;  // the rows left over run one per iteration below
   }
   // a fused product's first chunk is loaded before begin()
   constexpr bool kAhead = PAIR && ! Keep::kPlain;
   constexpr bool kSkip = SKIP && kSkipSlots< V, Keep, 1 >;
   int2 c[ kChunk ];
   typename Pair< V >::T v[ kChunk ];
   auto loadChunk = [ & ]( int64_t b, int32_t l0, int32_t width, int64_t step ) {
#pragma unroll
      for( int j = 0; j < kChunk; j++ ) {
         c[ j ] = make_int2( -1, -1 );
         v[ j ] = typename Pair< V >::T{};
         if( ! kSkip || l0 + j < width ) {
            const int64_t g = b + step * ( kSkip ? l0 + j : min( l0 + j, width - 1 ) );
            c[ j ] = ldnt2( col + g );
            v[ j ] = ldnt2( val + g );
         }
      }
   };
   bool ahead = false;
   if constexpr( kAhead ) {
      if( seq.start < seq.end && slots.width( seq.start ) > 0 ) {
         loadChunk( slots.base( seq.start ), 0, slots.width( seq.start ), slots.step() );
         ahead = true;
      }
      if( ! keep.begin() )
         return;
   }
   for( int64_t r = seq.start; r < seq.end; r += seq.step ) {
      const int64_t b = slots.base( r );
      const int32_t width = slots.width( r );
      const int64_t step = slots.step();
      A s0 = 0, s1 = 0;
      for( int32_t l0 = 0; l0 < width; l0 += kChunk ) {
         if constexpr( PAIR && ! kSkip && ! kAhead ) {
            int2 c[ kChunk ];
            typename Pair< V >::T v[ kChunk ];
#pragma unroll
            for( int j = 0; j < kChunk; j++ ) {
               const int64_t g = b + step * min( l0 + j, width - 1 );
               c[ j ] = ldnt2( col + g );
               v[ j ] = ldnt2( val + g );
            }
            Y x0[ kChunk ], x1[ kChunk ];
#pragma unroll
            for( int j = 0; j < kChunk; j++ ) {
               x0[ j ] = keep.at( x, c[ j ].x < 0 ? 0 : c[ j ].x );
               x1[ j ] = keep.at( x, c[ j ].y < 0 ? 0 : c[ j ].y );
            }
#pragma unroll
            for( int j = 0; j < kChunk; j++ ) {
               V a, bb;
               split( v[ j ], a, bb );
               if( l0 + j < width && c[ j ].x >= 0 )
                  s0 = mulAddExact( s0, toCompute( a, A() ), (A) x0[ j ] );
               if( l0 + j < width && c[ j ].y >= 0 )
                  s1 = mulAddExact( s1, toCompute( bb, A() ), (A) x1[ j ] );
            }
         }
         else if constexpr( PAIR ) {
            if( ! kAhead || ! ahead )
               loadChunk( b, l0, width, step );
            ahead = false;
            Y x0[ kChunk ], x1[ kChunk ];
#pragma unroll
            for( int j = 0; j < kChunk; j++ ) {
               x0[ j ] = x1[ j ] = Y( 0 );
               if( ! kSkip || l0 + j < width ) {
                  x0[ j ] = keep.at( x, c[ j ].x < 0 ? 0 : c[ j ].x );
                  x1[ j ] = keep.at( x, c[ j ].y < 0 ? 0 : c[ j ].y );
               }
            }
#pragma unroll
            for( int j = 0; j < kChunk; j++ ) {
               V a, bb;
               split( v[ j ], a, bb );
               if( ( kSkip || l0 + j < width ) && c[ j ].x >= 0 )
                  s0 = mulAddExact( s0, toCompute( a, A() ), (A) x0[ j ] );
               if( ( kSkip || l0 + j < width ) && c[ j ].y >= 0 )
                  s1 = mulAddExact( s1, toCompute( bb, A() ), (A) x1[ j ] );
            }
         }
         else {
            int32_t c[ kChunk ];
            V v[ kChunk ];
#pragma unroll
            for( int j = 0; j < kChunk; j++ ) {
               const int64_t g = b + step * min( l0 + j, width - 1 );
               c[ j ] = ldnt( col + g );
               v[ j ] = ldnt( val + g );
            }
            Y xv[ kChunk ];
#pragma unroll
            for( int j = 0; j < kChunk; j++ )
               xv[ j ] = keep.at( x, c[ j ] < 0 ? 0 : c[ j ] );
#pragma unroll
            for( int j = 0; j < kChunk; j++ )
               if( l0 + j < width && c[ j ] >= 0 )
                  s0 = mulAddExact( s0, toCompute( v[ j ], A() ), (A) xv[ j ] );
         }
      }
      if( r >= first )
         keep( r, s0 );
      if( PAIR && r + 1 < seq.end )
         keep( r + 1, s1 );
   }
}

struct EllpackSlots
{
   int32_t segmentSize, aligned;
   __device__ int64_t base( int64_t r ) const { return r; }
   __device__ int32_t width( int64_t ) const { return segmentSize; }
   __device__ int64_t step() const { return aligned; }
};

struct SlicedSlots
{
   const int32_t* sliceOffsets;
   const int32_t* sliceSizes;
   int32_t logSlice;  // log2 of the slice size (TNL's SliceSize, 32 by default)
   __device__ int64_t base( int64_t r ) const
   {
      return sliceOffsets[ r >> logSlice ] + ( r & ( ( 1 << logSlice ) - 1 ) );
   }
   __device__ int32_t width( int64_t r ) const { return sliceSizes[ r >> logSlice ]; }
   __device__ int64_t step() const { return (int64_t) 1 << logSlice; }
};

template< bool PAIR, typename V, typename A, typename Y, typename Keep >
__global__ __launch_bounds__( 256 ) void ellpackKernel( EllpackSlots slots, const int32_t* __restrict__ col,
                                                        const V* __restrict__ val, const Y* __restrict__ x,
                                                        Keep keep, int32_t first, int32_t last,
                                                        int32_t rowsPerBlock, int dist )
{
   if constexpr( PAIR && ! Keep::kPlain ) {
      if( keep.shut() )
         return;
      keep.prefetch();  // begin() follows the first loads
   }
   else if( ! openKeeper( keep ) )
      return;
   const int64_t base = PAIR ? ( first & ~1 ) : first;
   paddedRows< PAIR, true, V, A >( slots, col, val, x, keep, first, rowSequence< PAIR ? 2 : 1 >( base, last, rowsPerBlock, dist ) );
   keep.finish();
}

template< bool PAIR, bool SKIP, typename V, typename A, typename Y, typename Keep >
__global__ __launch_bounds__( 256 ) void slicedKernel( SlicedSlots slots, const int32_t* __restrict__ col,
                                                       const V* __restrict__ val, const Y* __restrict__ x,
                                                       Keep keep, int32_t first, int32_t last,
                                                       int32_t rowsPerBlock, int dist )
{
   if constexpr( PAIR && ! Keep::kPlain ) {
      if( keep.shut() )
         return;
      keep.prefetch();  // begin() follows the first loads
   }
   else if( ! openKeeper( keep ) )
      return;
   const int64_t base = PAIR ? ( first & ~1 ) : first;
   paddedRows< PAIR, SKIP, V, A >( slots, col, val, x, keep, first, rowSequence< PAIR ? 2 : 1 >( base, last, rowsPerBlock, dist ) );
   keep.finish();
}

// ------------------------------------------------------------------ ChunkedEllpack

// One 256-lane workgroup per slice, one lane per chunk (the format is built around 256
// chunks per slice): chunk c's elements sit at pointer + c + 256*k, coalesced across the
// workgroup.  Chunk sums meet in LDS and each row adds up its chunk range
// (rowToChunkMapping is an inclusive per-slice prefix of chunk counts).  A chunk's padding
// follows its elements, so with `stopAtPadding` a wavefront stops reading once every lane's
// chunk has reached padding: a slice's chunk size is set by its longest row, and short rows
// beside long ones would otherwise stream their padding in full.
template< typename V, typename A, typename Y, typename Keep >
__global__ __launch_bounds__( 256 ) void chunkedKernel( int32_t nslices, const int4* __restrict__ slices,
                                                        const int32_t* __restrict__ rowToChunk,
                                                        const int32_t* __restrict__ col,
                                                        const V* __restrict__ val, const Y* __restrict__ x,
                                                        Keep keep, int32_t first, int32_t last,
                                                        int stopAtPadding, int remap )
{
   if( ! openKeeper( keep ) )
      return;
   __shared__ A part[ kChunksInSlice ];
   const int t = threadIdx.x;
   // remap: XCD x (blockIdx % 8) takes the x-th eighth of the slices, in order
   for( int64_t sl = logicalBlock( remap ); sl < nslices; sl += gridDim.x ) {
      const int4 s = slices[ sl ];  // size, chunkSize, firstSegment, pointer
      if( s.z >= last || s.z + s.x <= first )
         continue;  // uniform over the workgroup
      // every row owns exactly one chunk when the slice uses as many chunks as it has rows
      const bool onePerRow = s.x > 0 && rowToChunk[ s.z + s.x - 1 ] == s.x;
      A p = 0;
      for( int32_t k0 = 0; k0 < s.y; k0 += kChunk ) {
         int32_t c[ kChunk ];
         if constexpr( kSkipSlots< V, Keep, 8 > ) {
            // `full`: every slot of the round exists, and its loads go out without a branch between them (FP64,
            // lognormal rows of 6 entries on average, 1 million of them: 307 us with the branches in every round, 264
            // with re-read slots, 240; 150^3 Laplacian 58.3 / 59.4 / 56.5)
            auto round = [ & ]( auto full ) {
               constexpr bool kFull = decltype( full )::value;
               V v[ kChunk ];
               Y xv[ kChunk ];
#pragma unroll
               for( int j = 0; j < kChunk; j++ ) {
                  c[ j ] = -1;
                  v[ j ] = V( 0.0f );
                  if( kFull || k0 + j < s.y ) {  // uniform over the workgroup
                     const int64_t g = (int64_t) s.w + t + (int64_t) kChunksInSlice * ( k0 + j );
                     c[ j ] = ldnt( col + g );
                     v[ j ] = ldnt( val + g );
                  }
               }
#pragma unroll
               for( int j = 0; j < kChunk; j++ ) {
                  xv[ j ] = Y( 0 );
                  if( kFull || k0 + j < s.y )
                     xv[ j ] = keep.at( x, c[ j ] < 0 ? 0 : c[ j ] );
               }
#pragma unroll
               for( int j = 0; j < kChunk; j++ )
                  if( c[ j ] >= 0 )
                     p += toCompute( v[ j ], A() ) * (A) xv[ j ];
            };
            if( k0 + kChunk <= s.y )
               round( std::true_type() );
            else
               round( std::false_type() );
         }
         else {
            V v[ kChunk ];
#pragma unroll
            for( int j = 0; j < kChunk; j++ ) {
               const int64_t g = (int64_t) s.w + t + (int64_t) kChunksInSlice * min( k0 + j, s.y - 1 );
               c[ j ] = ldnt( col + g );
               v[ j ] = ldnt( val + g );
            }
            Y xv[ kChunk ];
#pragma unroll
            for( int j = 0; j < kChunk; j++ )
               xv[ j ] = keep.at( x, c[ j ] < 0 ? 0 : c[ j ] );
#pragma unroll
            for( int j = 0; j < kChunk; j++ )
               if( k0 + j < s.y && c[ j ] >= 0 )
                  p += toCompute( v[ j ], A() ) * (A) xv[ j ];
         }
         // the last slot read is padding: so is the rest of this lane's chunk
         if( stopAtPadding && __all( c[ kChunk - 1 ] < 0 ) )
            break;  // wave-uniform; the loop holds no barrier
      }
      if( onePerRow ) {  // uniform: chunk t is row s.z + t, no exchange through LDS
         const int32_t row = s.z + t;
         if( t < s.x && row >= first && row < last )
            keep( row, (A) 0 + p );
         continue;
      }
      part[ t ] = p;
      __syncthreads();
      if( t < s.x ) {
         const int32_t row = s.z + t;
         if( row >= first && row < last ) {
            const int32_t cb = t == 0 ? 0 : rowToChunk[ row - 1 ], ce = rowToChunk[ row ];
            A acc = 0;
            for( int32_t c = cb; c < ce; c++ )
               acc += part[ c ];
            keep( row, acc );
         }
      }
      __syncthreads();
   }
   keep.finish();
}

// ------------------------------------------------------------------ BiEllpack

// A wavefront takes two strips of 32 rows, one per half-wave.  Group g of a strip is a
// dense height x width block (height 32 >> g) stored column-major, i.e. contiguous: lane l
// streams elements l, l+32, ... which all belong to rank l % height, then lanes with equal
// l % height are folded with xor-shuffles.  Lane l < height keeps rank l's running sum; at
// the end each lane fetches the sum of its own row's rank and stores it, so y is written
// coalesced.  The rank comes from a one-byte copy of rowPermArray[row] - 32 * strip (4 MB
// instead of 16 MB at 160^3).
constexpr int kBiUnroll = 8;

template< typename V, typename A, typename Y, typename Keep >
__global__ __launch_bounds__( 256 ) void biellpackKernel( int32_t n, int32_t strips, const uint8_t* __restrict__ rowRank,
                                                          const int32_t* __restrict__ groupPointers,
                                                          const int32_t* __restrict__ col,
                                                          const V* __restrict__ val, const Y* __restrict__ x,
                                                          Keep keep, int32_t first, int32_t last )
{
   if( ! openKeeper( keep ) )
      return;
   const int lane = threadIdx.x % kWave, half = lane / 32, l = lane % 32;
   const int32_t wave = ( blockIdx.x * blockDim.x + threadIdx.x ) / kWave;
   const int32_t waves = gridDim.x * ( blockDim.x / kWave );
   // group pointers of the half-wave's strip are fetched one iteration ahead
   int32_t gp[ kLogStrip + 1 ];
   auto fetch = [ & ]( int32_t strip, int32_t( &g )[ kLogStrip + 1 ] ) {
#pragma unroll
      for( int k = 0; k <= kLogStrip; k++ )
         g[ k ] = strip < strips ? groupPointers[ (int64_t) strip * kGroupsPerStrip + k ] : 0;
   };
   fetch( 2 * wave + half, gp );
   for( int32_t pair = wave; 2 * pair < strips; pair += waves ) {
      const int32_t strip = 2 * pair + half;
      const bool valid = strip < strips;
      const int64_t row = (int64_t) strip * kStrip + l;
      const bool mine = valid && row < n;
      const int rank = mine ? rowRank[ row ] : 0;
      int32_t gpNext[ kLogStrip + 1 ];
      fetch( 2 * ( pair + waves ) + half, gpNext );
      A acc = 0;
      if( valid ) {
         // group 5 (height 1) is always empty: the widths are taken at ranks 15, 7, 3, 1, 0
#pragma unroll
         for( int grp = 0; grp < kLogStrip; grp++ ) {
            const int32_t base = gp[ grp ], size = gp[ grp + 1 ] - base;
            const int h = kStrip >> grp;
            A p = 0;
            // 8 elements per lane in flight: a 32-row group up to 8 wide is one round trip
            for( int32_t e0 = l; e0 < size; e0 += kBiUnroll * kStrip ) {
               int32_t c[ kBiUnroll ];
               V v[ kBiUnroll ];
#pragma unroll
               for( int j = 0; j < kBiUnroll; j++ ) {
                  c[ j ] = -1;
                  v[ j ] = V( 0.0f );
                  if( ! kSkipSlots< V, Keep, 4 > || e0 + j * kStrip < size ) {
                     const int32_t e = kSkipSlots< V, Keep, 4 > ? e0 + j * kStrip : min( e0 + j * kStrip, size - 1 );
                     c[ j ] = ldnt( col + base + e );
                     v[ j ] = ldnt( val + base + e );
                  }
               }
               Y xv[ kBiUnroll ];
#pragma unroll
               for( int j = 0; j < kBiUnroll; j++ ) {
                  xv[ j ] = Y( 0 );
                  if( ! kSkipSlots< V, Keep, 4 > || e0 + j * kStrip < size )
                     xv[ j ] = keep.at( x, c[ j ] < 0 ? 0 : c[ j ] );
               }
#pragma unroll
               for( int j = 0; j < kBiUnroll; j++ )
                  if( ( kSkipSlots< V, Keep, 4 > || e0 + j * kStrip < size ) && c[ j ] >= 0 )
                     p += toCompute( v[ j ], A() ) * (A) xv[ j ];
            }
            for( int o = h; o < kStrip; o <<= 1 )
               p += __shfl_xor( p, o, kWave );
            if( l < h )
               acc += p;
         }
      }
      const A v = __shfl( acc, half * 32 + rank, kWave );
      if( mine && row >= first && row < last )
         keep( row, v );
#pragma unroll
      for( int k = 0; k <= kLogStrip; k++ )
         gp[ k ] = gpNext[ k ];
   }
   keep.finish();
}

// Rows without any stored element: y = keep( 0 ).
template< typename A, typename Keep >
__global__ __launch_bounds__( 256 ) void zeroRowsKernel( Keep keep, int32_t first, int32_t last )
{
   if( keep.closed() )
      return;
   const int64_t stride = (int64_t) gridDim.x * blockDim.x;
   for( int64_t r = first + (int64_t) blockIdx.x * blockDim.x + threadIdx.x; r < last; r += stride )
      keep( r, (A) 0 );
}

// ------------------------------------------------------------------ launch

// Lanes per row of the cooperative CSR kernel; 0 where the rows take the staged one
inline int lanesPerRow( const Matrix& M )
{
   if( M.format == TNLHIP_CSR_SCALAR || ( ! M.lanesExplicit && M.meta.allocated <= (int64_t) kShortRow * M.rows ) )
      return 0;
   return M.format == TNLHIP_CSR_VECTOR && ! M.lanesExplicit ? kWave : M.lanes;
}

// Whether M's rows take the staged CSR kernel with every wave's elements in LDS, none walking its rows one lane each
template< typename A >
bool stagedThroughout( const Matrix& M )
{
   return kindOf( M.format ) == KIND_CSR && lanesPerRow( M ) == 0 && M.meta.allocated <= (int64_t) kShortRow * M.rows &&
          M.meta.waveMost <= kAdaptiveStreamBytesPerWave / (int) sizeof( A );
}

// Launches the row kernel of M's format over rows [first, last) and returns its grid, or with `dry`
// only returns the grid; 0 when no row kernel runs (no rows, no columns, a striped plan, no storage).
template< typename V, typename A, typename Y, typename Keep >
unsigned launchProduct( const Matrix& M, const Y* x, Keep keep, int32_t first, int32_t last, hipStream_t st,
                        bool dry = false )
{
   const V* val = reinterpret_cast< const V* >( M.values.ptr );
   const int32_t* col = M.columns.ptr;
   const int64_t rows = last - first;
   unsigned used = 0;
   if( rows <= 0 )
      return used;
   // `used` stays 0 where the kernel that runs is not one of the row kernels above
   auto run = [ & ]( auto kernel, unsigned grid, auto... args ) {
      used = grid;
      if( ! dry )
         kernel<<< grid, 256, 0, st >>>( args... );
   };
   auto zeroRows = [ & ] {
      if constexpr( Keep::kPlain )
         zeroRowsKernel< A, Keep ><<< gridFor( rows, 256 ), 256, 0, st >>>( keep, first, last );
   };
   auto launchStaged = [ & ] {
      constexpr int K = kAdaptiveStreamBytesPerWave / sizeof( A ) / kWave;
      unsigned grid = (unsigned) ( ( rows + 255 ) / 256 );
      if( M.xcdRemap )
         grid = ( grid + kXcds - 1 ) / kXcds * kXcds;  // logicalBlock needs a multiple of 8
      run( csrScalarStagedKernel< K, V, A, Y, Keep >, grid, M.offsets.ptr, col, val, x, keep, first, last,
           M.xcdRemap ? 1 : 0 );
   };
   if constexpr( Keep::kPlain )
      if( M.streamY >= 0 )
         keep.streamY = M.streamY != 0;
   if( M.cols == 0 ) {
      // every stored slot is padding and x is empty: the kernels below gather x[0] for padding
      // slots, so a matrix without columns takes the all-zero product without touching x
      zeroRows();
      TNLHIP_CHECK( hipGetLastError() );
      return 0;
   }
   if( M.stripes && kindOf( M.format ) == KIND_CSR ) {
      if constexpr( std::is_same_v< Keep, Keeper< A, Y > > )
         stripeLaunch< V, A, Y >( M, x, keep, first, last, st );
      return 0;
   }
   switch( M.format ) {
      case TNLHIP_CSR_SCALAR:
         launchStaged();
         break;
      case TNLHIP_CSR_VECTOR:
      case TNLHIP_CSR_LIGHT:
      case TNLHIP_CSR_HYBRID:
      case TNLHIP_CSR_ADAPTIVE: {
         // a fused product of short rows takes the staged kernel, which hides the fold, unless some of its waves would
         // walk their rows (us per CG iteration with a row of 20000 elements among 200000 of 3: 5180 staged, 82 here; per BiCGStab
         // iteration with 1 million lognormal rows of 6: 764, 177)
         if( M.format == TNLHIP_CSR_ADAPTIVE && first == 0 && last == M.rows && M.adaptiveBlocks > 0 &&
             ( Keep::kPlain || ! stagedThroughout< A >( M ) ) ) {
            constexpr int STREAM = kAdaptiveStreamBytesPerWave / sizeof( A );
            // y through L2 on request (STREAM blocks end rows anywhere in a cache line of y, so
            // non-temporal stores write some lines twice); non-temporal by default, which measured
            // 79-80 us at 160^3 FP64 against 81-83 us through L2
            if constexpr( Keep::kPlain )
               keep.streamY = M.streamY != 0;
            unsigned groups = ( M.adaptiveBlocks + 3 ) / 4;
            if( M.xcdRemap )
               groups = ( groups + kXcds - 1 ) / kXcds * kXcds;  // logicalBlock needs a multiple of 8
            run( csrAdaptiveKernel< STREAM, V, A, Y, Keep >, groups, M.adaptiveBlocks,
                 reinterpret_cast< const int4* >( M.adaptive.ptr ), M.offsets.ptr, col, val, x, keep,
                 M.xcdRemap ? 1 : 0 );
            break;
         }
         // rows of at most kShortRow stored elements on average: most lanes of a cooperative row
         // group would idle (a wavefront per 7-element row uses 7 of 64), so unless lanes_per_row
         // was set the rows take CSRScalar's staged kernel (the Host result bit for bit)
         const int G = lanesPerRow( M );
         if( G == 0 ) {
            launchStaged();
            break;
         }
         const int gpb = 256 / G;
         const unsigned grid = gridFor( rows, gpb );
         switch( G ) {
            case 1:
               run( csrGroupedKernel< 1, 1, false, V, A, Y, Keep >, grid, M.offsets.ptr, col, val, x, keep, first,
                    last );
               break;
            case 2:
               run( csrGroupedKernel< 2, 4, false, V, A, Y, Keep >, grid, M.offsets.ptr, col, val, x, keep, first,
                    last );
               break;
            case 4:
               run( csrGroupedKernel< 4, 4, false, V, A, Y, Keep >, grid, M.offsets.ptr, col, val, x, keep, first,
                    last );
               break;
            case 8:
               run( csrGroupedKernel< 8, 4, false, V, A, Y, Keep >, grid, M.offsets.ptr, col, val, x, keep, first,
                    last );
               break;
            case 16:
               run( csrGroupedKernel< 16, 2, false, V, A, Y, Keep >, grid, M.offsets.ptr, col, val, x, keep, first,
                    last );
               break;
            case 32:
               run( csrGroupedKernel< 32, 2, false, V, A, Y, Keep >, grid, M.offsets.ptr, col, val, x, keep, first,
                    last );
               break;
            default:
               run( csrGroupedKernel< 64, 1, false, V, A, Y, Keep >, grid, M.offsets.ptr, col, val, x, keep, first,
                    last );
               break;
         }
         break;
      }
      case TNLHIP_ELLPACK:
      case TNLHIP_SLICED_ELLPACK: {
         // grid a multiple of the XCD count; contiguous row blocks when dist != 0
         // a row pair is one 8- / 16-byte load of two vertically adjacent slots: SlicedEllpack
         // with slice size 1 has no such neighbours (row r + 1 lies in the next slice), so it
         // takes one row per lane whatever pair_rows says
         const bool pair = M.pairRows != 0 && ( M.format == TNLHIP_ELLPACK || M.meta.sliceSize >= 2 );
         // a fused product takes the rows in the order of the passes around it, which read and write the same
         // vectors: 64^3 CG 14.8 us per iteration against 17.1 in XCD order
         const int dist = Keep::kPlain ? M.xcdRemap : 0;
         if( ! knownDistribution( dist ) )
            throw Error( TNLHIP_ERROR_INVALID_ARGUMENT, "unknown row distribution" );
         const PaddedLaunch pl = paddedLaunch( first, last, pair, M.blocksPerCu, deviceProps().cus );
         const unsigned grid = (unsigned) pl.grid;
         const int64_t per = pl.per;
         const EllpackSlots es{ M.meta.segmentSize, M.meta.alignedSize };
         const SlicedSlots ss{ M.sliceOffsets.ptr, M.sliceSizes.ptr, log2Exact( M.meta.sliceSize ) };
         if( M.format == TNLHIP_ELLPACK ) {
            if( pair )
               run( ellpackKernel< true, V, A, Y, Keep >, grid, es, col, val, x, keep, first, last, (int32_t) per,
                    dist );
            else
               run( ellpackKernel< false, V, A, Y, Keep >, grid, es, col, val, x, keep, first, last, (int32_t) per,
                    dist );
         }
         else {
            // (a fused product's rows take the registers either way)
            bool skip = true;
            if constexpr( Keep::kPlain ) {
               skip = M.meta.allocated <= (int64_t) kSkipSlotsUpTo * M.rows;
               if( pair && ! skip )
                  run( slicedKernel< true, false, V, A, Y, Keep >, grid, ss, col, val, x, keep, first, last, (int32_t) per,
                       dist );
            }
            if( pair && skip )
               run( slicedKernel< true, true, V, A, Y, Keep >, grid, ss, col, val, x, keep, first, last, (int32_t) per,
                    dist );
            if( ! pair )
               run( slicedKernel< false, true, V, A, Y, Keep >, grid, ss, col, val, x, keep, first, last, (int32_t) per,
                    dist );
         }
         break;
      }
      case TNLHIP_CHUNKED_ELLPACK:
         if( M.meta.numberOfSlices > 0 )
            // one workgroup per slice: at 160^3 70.6 us, against 78.1 / 72.7 us for grids of 8 / 32
            // workgroups per CU striding over the slices
            run( chunkedKernel< V, A, Y, Keep >,
                 M.xcdRemap ? ( M.meta.numberOfSlices + kXcds - 1 ) / kXcds * kXcds : M.meta.numberOfSlices,
                 M.meta.numberOfSlices, reinterpret_cast< const int4* >( M.slices.ptr ), M.rowToChunk.ptr, col,
                 val, x, keep, first, last, M.trailingPadding ? 1 : 0, M.xcdRemap ? 1 : 0 );
         break;
      case TNLHIP_BIELLPACK: {
         const int32_t strips = M.meta.virtualRows / kStrip;
         const int32_t pairs = ( strips + 1 ) / 2;
         if( strips > 0 && M.meta.allocated > 0 )
            // 32 workgroups per CU (two strip pairs per wave at 160^3): 79.8 us, against 83.0 us
            // at 8 and 84.3 us with one workgroup per 4 pairs
            run( biellpackKernel< V, A, Y, Keep >, gridFor( pairs, 4, 32 ), M.rows, strips, M.biRank.ptr,
                 M.groupPointers.ptr, col, val, x, keep, first, last );
         else
            // no stored element at all (TNL's Host path returns without touching y here,
            // BiEllpackView.hpp:248-249); every row of A x is zero
            zeroRows();
         break;
      }
      default: throw Error( TNLHIP_ERROR_INVALID_ARGUMENT, "unknown format" );
   }
   TNLHIP_CHECK( hipGetLastError() );
   return used;
}

}  // namespace tnlhip

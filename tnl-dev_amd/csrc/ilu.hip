// ILU(0) preconditioner: Preconditioners/ILU0.hpp:17-137 (Host) and
// Utils/TriangularSolve.h:25-111, on the device.
//
// Symbolic part (host, once per matrix): row i of A is read in storage order (stored zeros
// included); TNL's counting rule gives nl entries with column < i and nu with column in [i, N),
// padding skipped, and the first nl stored entries become row i of L, the next nu row i of U
// (ILU0.hpp:36-90).  Rows whose split does not put every L column in [0, i) and every U column
// in [i, N), or whose U row is empty (no U_ii to divide by), are refused.
//
// Numeric factorization and the two triangular solves run on the device in level order: row i
// depends on the rows named by its L columns (factorization and forward solve) or by its U
// columns above the diagonal (backward solve), so all rows of one level are independent.  Every
// row is processed by one lane with TNL's operation order -- L_ik = L_ik / U_kk, then
// L_ij -= L_ik U_kj and U_ij -= L_ik U_kj (U_kj = 0 when row k of U has no column j); forward
// x_i = b_i - sum L_ij x_j; backward x_i = (x_i - sum_{c >= 1} U_ij x_j) / U_i[0] -- each
// product rounded before the subtraction, so the factors and the solves equal TNL's Host results
// bit for bit.
//
// The triangular solves work on a copy of the factor in level order (Sweep): the rows of a level,
// longest first, take consecutive positions from an even one on, and vectors are permuted to
// positions before the first level and back after the last one.  A level with more than
// kNarrowLevel rows, or more than kFarLevel of them that reach far back, is one launch over the
// device; runs of consecutive smaller levels are one launch of a single workgroup, as large as the
// largest of them needs (up to 1024 lanes), which takes two adjacent positions per lane at a time (a step).
//
// 64^3 7-point convection-diffusion in FP64 (190 levels a sweep): BiCGStab to 1e-10, 58 iterations.
// One launch per level above 1024 rows and a workgroup for the others, each row reading its row
// pointers, entries and solution entries in turn from memory: 240 ms; as above: 60 ms, 212 / 250 us
// a lower / upper sweep (about 1000 before), of which 80 us are the chain and the arithmetic and the
// rest the loads of the run's one CU.
#include "ilu.hpp"

#include <algorithm>

namespace tnlhip {

namespace {

constexpr int kIluBlock = 256;
constexpr int kRunBlock = 1024;         // one workgroup of 16 waves for runs of small levels
constexpr int32_t kSliceRows = 2 * kWave;
constexpr int32_t kNarrowLevel = 4096;  // levels of at most this many rows are taken in runs
constexpr int32_t kFarLevel = 1024;     // and these where some entry is older than the ring
constexpr int32_t kNarrowFactor = 1024; // likewise in the factorization
constexpr int32_t kRing = 16384;        // solution entries kept in LDS by a run (128 KiB in FP64)
static_assert( kRing >= 2 * kNarrowLevel && ( kRing & ( kRing - 1 ) ) == 0 && kRing < 65536,
               "the ring holds a level and the one before it, and its slots are 16-bit numbers" );

// Step flags: the step is the last one of its level; its entries are all in the rest arrays (some
// entry is not in the ring, or the level is wide); some row has more than W entries
constexpr int32_t kLastOfLevel = 1, kAllInRest = 2, kLongRow = 4;

template< typename T >
struct IluView
{
   const int32_t* Lrp;
   const int32_t* Lc;
   T* Lv;
   const int32_t* Urp;
   const int32_t* Uc;
   T* Uv;
};

// U.getElement( k, j ): the first stored entry of row k with column j, or 0
template< typename T >
__device__ __forceinline__ T uElement( const IluView< T >& f, int32_t k, int32_t j )
{
   for( int32_t c = f.Urp[ k ]; c < f.Urp[ k + 1 ]; c++ )
      if( f.Uc[ c ] == j )
         return f.Uv[ c ];
   return (T) 0;
}

template< typename T >
__device__ __forceinline__ void factorRow( const IluView< T >& f, int32_t i )
{
   const int32_t le = f.Lrp[ i + 1 ];
   for( int32_t ck = f.Lrp[ i ]; ck < le; ck++ ) {
      const int32_t k = f.Lc[ ck ];
      const T lik = f.Lv[ ck ] / uElement( f, k, k );
      f.Lv[ ck ] = lik;
      for( int32_t cj = ck + 1; cj < le; cj++ )
         f.Lv[ cj ] = mulSubExact( f.Lv[ cj ], lik, uElement( f, k, f.Lc[ cj ] ) );
      for( int32_t cj = f.Urp[ i ]; cj < f.Urp[ i + 1 ]; cj++ )
         f.Uv[ cj ] = mulSubExact( f.Uv[ cj ], lik, uElement( f, k, f.Uc[ cj ] ) );
   }
}

// factorization: one level over the whole device
template< typename T >
__global__ __launch_bounds__( kIluBlock ) void factorLevelKernel( IluView< T > f, const int32_t* __restrict__ order,
                                                                  int32_t begin, int32_t end )
{
   for( int32_t k = begin + blockIdx.x * kIluBlock + threadIdx.x; k < end; k += gridDim.x * kIluBlock )
      factorRow( f, order[ k ] );
}

// factorization: consecutive small levels in one workgroup; the barrier makes each level's results
// visible to the next (same CU)
template< typename T >
__global__ __launch_bounds__( kRunBlock ) void factorRunKernel( IluView< T > f, const int32_t* __restrict__ order,
                                                                const int32_t* __restrict__ levels, int32_t first,
                                                                int32_t last )
{
   for( int32_t lv = first; lv < last; lv++ ) {
      const int32_t end = levels[ lv + 1 ];
      for( int32_t k = levels[ lv ] + threadIdx.x; k < end; k += kRunBlock )
         factorRow( f, order[ k ] );
      __syncthreads();
   }
}

// ------------------------------------------------------------------ triangular sweeps

template< typename T >
struct PairOf;
template<>
struct PairOf< double >
{
   typedef double type __attribute__( ( ext_vector_type( 2 ) ) );
};
template<>
struct PairOf< float >
{
   typedef float type __attribute__( ( ext_vector_type( 2 ) ) );
};

// 16-byte words of ring slots per pair of rows: one for W <= 4 (four slots a row), else one a row
constexpr int slotWords( int W )
{
   return W <= 4 ? 1 : 2;
}

// The pair of positions 2 t, 2 t + 1 past a step's first position is word first / 2 + t of vectors;
// its slots are words C * first / 2 + j * pairs + t (j < C = slotWords( W )) and its entries l < W
// are words W * first / 2 + l * pairs + t, so that every load of a wave is contiguous and 16 bytes
// wide in FP64.  (A CU takes about 16 clocks per load instruction of a wave, whatever its width:
// 37, 74 and 140 GB/s at 4, 8 and 16 bytes a lane.)
template< typename T >
struct SweepView
{
   using Pair = typename PairOf< T >::type;
   const int4* steps;         // {first position, pairs, first slice, flags}
   const uint4* slots;        // ring slots, kRing for an absent entry
   const Pair* val;
   const T* diag;             // U: the diagonal of the row at each position
   const int32_t* len;        // entries of the row at each position (U: without the diagonal)
   // entries in the rest arrays: of the even, then of the odd positions of each slice, by entry,
   // then position, without padding -- the rows still active at entry l are the first ones
   const int32_t* sliceRest;  // two starts per slice
   const int32_t* restCol;    // ring slot s, or position q as ~q
   const T* restVal;
};

template< typename T >
SweepView< T > sweepView( const Ilu0::Sweep& s )
{
   return SweepView< T >{ reinterpret_cast< const int4* >( s.steps.ptr ), reinterpret_cast< const uint4* >( s.slots.ptr ),
                          reinterpret_cast< const typename PairOf< T >::type* >( s.val.ptr ),
                          reinterpret_cast< const T* >( s.diag.ptr ), s.len.ptr, s.sliceRest.ptr, s.restCol.ptr,
                          reinterpret_cast< const T* >( s.restVal.ptr ) };
}

// Copies a factor into its sweep layout: one wavefront per slice.  An absent entry is 0 times the
// ring's slot kRing, which holds +0: subtracting +0 leaves every value as it is.
template< typename T >
__global__ __launch_bounds__( kIluBlock ) void packKernel( int32_t nslices, int32_t W, const int4* __restrict__ slices,
                                                           const int32_t* __restrict__ order,
                                                           const int32_t* __restrict__ position,
                                                           const int32_t* __restrict__ rp,
                                                           const int32_t* __restrict__ c, const T* __restrict__ v,
                                                           int skipDiagonal, const int32_t* __restrict__ len,
                                                           const int4* __restrict__ steps,
                                                           const int32_t* __restrict__ sliceRest, uint16_t* slots, T* val,
                                                           T* diag, int32_t* restCol, T* restVal )
{
   const int lane = threadIdx.x % kWave;
   const int32_t s = ( blockIdx.x * kIluBlock + threadIdx.x ) / kWave;
   if( s >= nslices )
      return;
   const int4 d = slices[ s ];  // first position, step, oldest position in the ring, first position of the level
   const int4 st = steps[ d.y ];
   for( int odd = 0; odd < 2; odd++ ) {
      const int32_t p = d.x + 2 * lane + odd;
      const int64_t t = ( p - st.x ) / 2;
      const bool mine = t < st.y;
      const int32_t n = mine ? len[ p ] : 0;
      const int32_t src = mine ? rp[ order[ p ] ] + skipDiagonal : 0;
      if( mine && skipDiagonal )
         diag[ p ] = v[ src - 1 ];
      const bool packed = ! ( st.w & kAllInRest );
      if( mine && packed )
         for( int32_t l = 0; l < W; l++ ) {
            const int64_t word = slotWords( W ) == 1 ? st.x / 2 + t : 2 * (int64_t) ( st.x / 2 ) + (int64_t) odd * st.y + t;
            slots[ 8 * word + ( slotWords( W ) == 1 ? 4 * odd : 0 ) + l ] =
               (uint16_t) ( l < n ? position[ c[ src + l ] ] & ( kRing - 1 ) : kRing );
            val[ 2 * ( W * (int64_t) ( st.x / 2 ) + (int64_t) l * st.y + t ) + odd ] = l < n ? v[ src + l ] : (T) 0;
         }
      int32_t e = sliceRest[ 2 * s + odd ];
      for( int32_t l = packed ? W : 0;; l++ ) {
         const unsigned long long on = __ballot( l < n );
         if( ! on )
            break;
         if( l < n ) {
            const int32_t q = position[ c[ src + l ] ];
            restCol[ e + lane ] = q >= d.z && q < d.w ? q & ( kRing - 1 ) : ~q;
            restVal[ e + lane ] = v[ src + l ];
         }
         e += __popcll( on );
      }
   }
}

// dst[ k ] = src[ index[ k ] ]: a vector into level order, between the two level orders, or back
template< typename T >
__global__ __launch_bounds__( kIluBlock ) void permuteKernel( int32_t n, const int32_t* __restrict__ index,
                                                              const T* __restrict__ src, T* __restrict__ dst,
                                                              Gate gate )
{
   if( ! gate.open() )
      return;
   for( int32_t k = blockIdx.x * kIluBlock + threadIdx.x; k < n; k += gridDim.x * kIluBlock )
      dst[ k ] = src[ index[ k ] ];
}

// Subtracts the entries of a row from entry `from` on, which are in the rest arrays, from acc, left to
// right; `start` is the start of the row's half of its slice, solved( column ) a solution entry.  The
// loads of U entries go out together: one by one each took two trips to memory (27-point 60^3, BiCGStab:
// 14.3 -> 8.2 ms an iteration).
template< int U, typename T, typename F >
__device__ __forceinline__ void restOfRow( const SweepView< T >& f, int32_t start, int32_t from, int32_t n, T& acc,
                                           F&& solved )
{
   const int lane = threadIdx.x % kWave;
   int32_t e = start;
   for( int32_t l = from; __any( l < n ); l += U ) {
      int32_t c[ U ];
      T v[ U ], xv[ U ];
#pragma unroll
      for( int u = 0; u < U; u++ ) {
         // a lane without the entry reads the first one of the half slice
         const int32_t at = l + u < n ? e + lane : start;
         c[ u ] = f.restCol[ at ];
         v[ u ] = f.restVal[ at ];
         e += __popcll( __ballot( l + u < n ) );
      }
#pragma unroll
      for( int u = 0; u < U; u++ )
         xv[ u ] = solved( c[ u ] );
#pragma unroll
      for( int u = 0; u < U; u++ )
         acc = l + u < n ? mulSubExact( acc, v[ u ], xv[ u ] ) : acc;
   }
}

// x (on entry the right-hand side, in level order) of one level, over the whole device; a wide
// level is no part of a run, so every entry is in the rest arrays, as a position
template< bool UPPER, typename T >
__global__ __launch_bounds__( kIluBlock ) void sweepLevelKernel( SweepView< T > f, int32_t firstSlice, int32_t slices,
                                                                 int32_t begin, int32_t end, T* x, Gate gate )
{
   if( ! gate.open() )
      return;
   const int lane = threadIdx.x % kWave;
   for( int32_t h = ( blockIdx.x * kIluBlock + threadIdx.x ) / kWave; h < 2 * slices; h += gridDim.x * ( kIluBlock / kWave ) ) {
      const int32_t p = begin + h / 2 * kSliceRows + 2 * lane + h % 2;
      const bool mine = p < end;
      T acc = mine ? x[ p ] : (T) 0;
      restOfRow< 8 >( f, f.sliceRest[ 2 * firstSlice + h ], 0, mine ? f.len[ p ] : 0, acc,
                      [ & ]( int32_t c ) { return x[ ~c ]; } );
      if( mine )
         x[ p ] = UPPER ? acc / f.diag[ p ] : acc;
   }
}

// LDS traffic of the workgroup only: global loads in flight stay in flight across it
__device__ __forceinline__ void ldsBarrier()
{
   __builtin_amdgcn_fence( __ATOMIC_RELEASE, "workgroup", "local" );
   __builtin_amdgcn_s_barrier();
   __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "workgroup", "local" );
}

// A run of small levels in one workgroup.  What bounds it is the chain of levels and, for levels of
// thousands of rows, the load instructions of one CU, so a level waits only for the level before:
// the solution entries of the last kRing positions are read from LDS, and everything else of a step
// (its rows' first W entries, right-hand sides and diagonals) is fetched D steps ahead, across
// barriers that wait for LDS only.  Step descriptors come 64 at a time into the lanes of each wave,
// so a step's addresses are scalars plus the lane's offset.  count is a multiple of D.
template< bool UPPER, int W, int D, typename T >
__global__ __launch_bounds__( kRunBlock ) void sweepRunKernel( SweepView< T > f, int32_t firstStep, int32_t count, T* x,
                                                               Gate gate )
{
   static_assert( kWave % D == 0, "a table of descriptors ends with a round of D steps" );
   using Pair = typename SweepView< T >::Pair;
   constexpr int C = slotWords( W );
   if( ! gate.open() )
      return;
   __shared__ __align__( 16 ) T ring[ kRing + 2 ];
   const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
   const int32_t tid = threadIdx.x;
   if( tid == 0 )
      ring[ kRing ] = 0;
   f.steps += firstStep;
   Pair* xp = reinterpret_cast< Pair* >( x );
   const Pair* diag = reinterpret_cast< const Pair* >( f.diag );
   auto loadTable = [ & ]( int32_t from ) { return f.steps[ min( from + lane, count - 1 ) ]; };
   // The first loads and, once in 64 steps, a table are waited for where they are issued: left in
   // flight into the loop, they would make the waits of every step cover all that the wave has in
   // flight.  (vmcnt 0, the other counters untouched)
   auto arrived = [] { __builtin_amdgcn_s_waitcnt( 0x0f70 ); };
   struct Entries
   {
      int32_t first, pairs, slice, flags;  // of the step: uniform
      uint4 slots[ C ];
      Pair val[ W ];
      Pair rhs, diag;
   };
   // the step in lane k of `table`; lanes past its pairs re-read its last one (a step without rows:
   // its first position's)
   auto fetch = [ & ]( const int4& table, int k, Entries& q ) {
      q.first = __builtin_amdgcn_readlane( table.x, k );
      q.pairs = __builtin_amdgcn_readlane( table.y, k );
      q.slice = __builtin_amdgcn_readlane( table.z, k );
      q.flags = __builtin_amdgcn_readlane( table.w, k );
      const uint32_t at = (uint32_t) min( tid, max( q.pairs - 1, 0 ) );
      const int64_t pair = q.first / 2;
      const uint4* c = f.slots + C * pair;
      const Pair* v = f.val + W * pair;
#pragma unroll
      for( int j = 0; j < C; j++, c += q.pairs )
         q.slots[ j ] = c[ at ];
#pragma unroll
      for( int l = 0; l < W; l++, v += q.pairs )
         q.val[ l ] = v[ at ];
      q.rhs = ( xp + pair )[ at ];
      if constexpr( UPPER )
         q.diag = ( diag + pair )[ at ];
   };
   auto slotOf = [ & ]( const Entries& q, int odd, int l ) -> uint32_t {
      const int k = ( C == 1 ? 4 * odd : 0 ) + l;  // of the word's eight slots
      const uint4& w = q.slots[ C == 1 ? 0 : odd ];
      const uint32_t two = k / 2 == 0 ? w.x : k / 2 == 1 ? w.y : k / 2 == 2 ? w.z : w.w;
      return k % 2 ? two >> 16 : two & 0xffffu;
   };
   auto solveStep = [ & ]( const Entries& q ) {
      const bool mine = tid < q.pairs;
      Pair acc = q.rhs;
      if( ! ( q.flags & kAllInRest ) ) {
         T xv[ 2 ][ W ];
#pragma unroll
         for( int odd = 0; odd < 2; odd++ )
#pragma unroll
            for( int l = 0; l < W; l++ )
               xv[ odd ][ l ] = ring[ slotOf( q, odd, l ) ];
#pragma unroll
         for( int odd = 0; odd < 2; odd++ )
#pragma unroll
            for( int l = 0; l < W; l++ )
               acc[ odd ] = mulSubExact( (T) acc[ odd ], (T) q.val[ l ][ odd ], xv[ odd ][ l ] );
      }
      if( q.flags & ( kAllInRest | kLongRow ) ) {
         __syncthreads();  // uniform: every earlier level's entries are in memory after it
         if( wave * kWave < q.pairs ) {
            for( int odd = 0; odd < 2; odd++ ) {
               T a = odd ? acc[ 1 ] : acc[ 0 ];
               restOfRow< W <= 4 ? 4 : 8 >( f, f.sliceRest[ 2 * ( q.slice + wave ) + odd ], q.flags & kAllInRest ? 0 : W,
                          mine ? f.len[ q.first + 2 * tid + odd ] : 0, a,
                          [ & ]( int32_t c ) { return c >= 0 ? ring[ c ] : x[ ~c ]; } );
               if( odd )
                  acc[ 1 ] = a;
               else
                  acc[ 0 ] = a;
            }
         }
      }
      if constexpr( UPPER ) {
         acc[ 0 ] = acc[ 0 ] / q.diag[ 0 ];
         acc[ 1 ] = acc[ 1 ] / q.diag[ 1 ];
      }
      if( mine ) {
         *reinterpret_cast< Pair* >( &ring[ ( q.first + 2 * tid ) & ( kRing - 1 ) ] ) = acc;
         ( xp + q.first / 2 )[ (uint32_t) tid ] = acc;
      }
   };
   int4 table = loadTable( 0 ), tableNext = loadTable( kWave );
   arrived();
   Entries entries[ D ];
#pragma unroll
   for( int u = 0; u < D; u++ )
      fetch( table, u, entries[ u ] );
   arrived();
   __syncthreads();  // ring[ kRing ]
   for( int32_t t0 = 0; t0 < count; t0 += D ) {
      // the steps fetched in this round: t0 + D .. t0 + 2 D - 1, past the last one re-read
      const int k0 = ( t0 + D ) % kWave;
      if( k0 == 0 ) {
         table = tableNext;
         tableNext = loadTable( t0 + D + kWave );
         arrived();
      }
#pragma unroll
      for( int u = 0; u < D; u++ ) {
         solveStep( entries[ u ] );
         const bool last = entries[ u ].flags & kLastOfLevel;
         fetch( table, k0 + u, entries[ u ] );
         if( last )
            ldsBarrier();
      }
   }
}

// Entries of a row fetched ahead (W), and how many steps ahead (D): 3 entries cover the lower and the
// upper half of a 7-point stencil; D is what the 128 registers of a lane hold.  Factors of more than 3
// entries a row take 7 two steps ahead (ms per iteration of BiCGStab, 3 four ahead / 7 two ahead: 9-point
// 300^2 9.2 / 3.0, 27-point 60^3 10.8 / 8.2, 120^3 54.6 / 36.3).
constexpr int kShortW = 3, kShortD = 4, kLongW = 7, kLongD = 2;

// Rows grouped by level, in a level the rows with the most entries first (`length`, without U's
// diagonal; stable in the row index), every level from an even position on (a position left over
// takes row 0, without entries), and the launches, steps and slices that cover the levels.
// columns( i ): the first of row i's `length[ i ]` column indexes.
template< typename Columns >
void buildSchedule( Ilu0::Sweep& s, const std::vector< int32_t >& level, const std::vector< int32_t >& length,
                    Columns&& columns, std::vector< int32_t >& order, std::vector< int32_t >& position, hipStream_t st )
{
   const int32_t n = (int32_t) level.size();
   int32_t nl = 0, longest = 0;
   int64_t total = 0;
   for( int32_t i = 0; i < n; i++ ) {
      nl = std::max( nl, level[ i ] + 1 );
      longest = std::max( longest, length[ i ] );
      total += length[ i ];
   }
   s.longRows = total > (int64_t) kShortW * n;
   const int32_t W = s.longRows ? kLongW : kShortW, D = s.longRows ? kLongD : kShortD;
   // two stable counting sorts: by length, longest first, then by level
   std::vector< int32_t > fill( (size_t) longest + 2, 0 ), byLength( n );
   for( int32_t i = 0; i < n; i++ )
      fill[ longest - length[ i ] + 1 ]++;
   for( int32_t k = 0; k <= longest; k++ )
      fill[ k + 1 ] += fill[ k ];
   for( int32_t i = 0; i < n; i++ )
      byLength[ fill[ longest - length[ i ] ]++ ] = i;
   s.levels.assign( (size_t) nl + 1, 0 );
   for( int32_t l : level )
      s.levels[ l + 1 ]++;
   int64_t positions = 0;
   for( int32_t l = 0; l < nl; l++ ) {
      positions += ( s.levels[ l + 1 ] + 1 ) / 2 * 2;
      TNLHIP_REQUIRE( positions <= INT32_MAX, "ILU(0): too many rows" );
      s.levels[ l + 1 ] = (int32_t) positions;
   }
   s.positions = (int32_t) positions;
   fill.assign( s.levels.begin(), s.levels.end() - 1 );
   order.assign( s.positions, 0 );
   position.resize( n );
   std::vector< int32_t > len( s.positions, 0 ), sliceRest, slices, steps;
   for( int32_t i : byLength ) {
      position[ i ] = fill[ level[ i ] ]++;
      order[ position[ i ] ] = i;
      len[ position[ i ] ] = length[ i ];
   }
   s.rest = 0;
   s.launches.clear();
   auto rowsOf = [ & ]( int32_t l ) { return s.levels[ l + 1 ] - s.levels[ l ]; };
   // The positions a step of level l finds in the ring of a run that starts at position runFirst: solved by the
   // run in an earlier level, and no more than kRing positions before this level's end.  (A second entry of U
   // at the row's own column takes the value from before the row is solved: not in the ring.)
   auto ringFrom = [ & ]( int32_t l, int32_t runFirst ) { return std::max( runFirst, s.levels[ l + 1 ] - kRing ); };
   // whether some of the first W entries of rows [ p, last ) of level l are not in that ring
   auto outside = [ & ]( int32_t l, int32_t p, int32_t last, int32_t runFirst ) {
      const int32_t begin = s.levels[ l ], oldest = ringFrom( l, runFirst );
      for( int32_t k = p; k < last; k++ ) {
         const int32_t* c = len[ k ] > 0 ? columns( order[ k ] ) : nullptr;
         for( int32_t j = 0; j < std::min( len[ k ], W ); j++ )
            if( position[ c[ j ] ] < oldest || position[ c[ j ] ] >= begin )
               return true;
      }
      return false;
   };
   // the steps and slices of levels [ l, e ); flags: of each step, nullptr where every entry is in the rest arrays
   auto addLaunch = [ & ]( int32_t l, int32_t e, int32_t block, const int32_t* flags ) {
      const int32_t runFirst = s.levels[ l ], firstStep = (int32_t) steps.size() / 4, firstSlice = (int32_t) slices.size() / 4;
      for( int32_t lv = l; lv < e; lv++ ) {
         const int32_t begin = s.levels[ lv ], end = s.levels[ lv + 1 ];
         const int32_t oldest = flags ? ringFrom( lv, runFirst ) : s.positions;
         for( int32_t p = begin; p < end; p += 2 * block ) {
            const int32_t last = std::min( end, p + 2 * block );
            const int32_t flag = flags ? *flags++ : kAllInRest;
            const int32_t from = flag & kAllInRest ? 0 : W, step = (int32_t) steps.size() / 4;
            steps.insert( steps.end(), { p, ( last - p ) / 2, (int32_t) slices.size() / 4, flag } );
            for( int32_t q = p; q < last; q += kSliceRows ) {
               slices.insert( slices.end(), { q, step, oldest, begin } );
               for( int odd = 0; odd < 2; odd++ ) {
                  sliceRest.push_back( s.rest );
                  for( int32_t k = q + odd; k < std::min( q + kSliceRows, last ); k += 2 )
                     s.rest += std::max( len[ k ] - from, 0 );
               }
            }
         }
      }
      // a run takes its steps in rounds of D: steps without rows fill the last one
      while( flags && ( (int32_t) ( steps.size() / 4 ) - firstStep ) % D )
         steps.insert( steps.end(), { runFirst, 0, firstSlice, 0 } );
      s.launches.push_back( { l, e, firstStep, (int32_t) ( steps.size() / 4 ) - firstStep, firstSlice,
                              (int32_t) ( slices.size() / 4 ) - firstSlice, block, ! flags } );
   };
   // A level that is a launch of its own: more rows than a run takes, or more than kFarLevel of them with an
   // entry older than the ring, which a run's one CU would fetch from memory.  us per iteration of BiCGStab (four
   // sweeps), 40 levels that draw on all before them, in the run / as launches: 4000 rows of 3 entries 1759 / 1103, 2500 of
   // 13 3607 / 1406, 1100 of 13 1312 / 1095; at 900 rows of 13, in the run 1050.
   auto wide = [ & ]( int32_t l ) {
      return rowsOf( l ) > kNarrowLevel ||
             ( rowsOf( l ) > kFarLevel && outside( l, s.levels[ l ], s.levels[ l + 1 ], 0 ) );
   };
   for( int32_t l = 0; l < nl; ) {
      int32_t e = l, rows = 0;
      for( ; e < nl && ! wide( e ); e++ )
         rows = std::max( rows, rowsOf( e ) );
      if( e > l ) {
         // a workgroup for the largest level of the run, two rows per lane: every wave of it issues the loads of
         // every step, rows or not, and a CU issues them one after another (tridiagonal matrix of 20000 rows,
         // BiCGStab: 129 ms an iteration with 16 waves, 48 ms)
         const int32_t block = std::min( kRunBlock, ( rows + kSliceRows - 1 ) / kSliceRows * kWave );
         std::vector< int32_t > flags;
         for( int32_t lv = l; lv < e; lv++ ) {
            // wide() has seen that the ring holds what its rows need, if it began that early
            const bool inside = rowsOf( lv ) > kFarLevel && ringFrom( lv, s.levels[ l ] ) == ringFrom( lv, 0 );
            for( int32_t p = s.levels[ lv ]; p < s.levels[ lv + 1 ]; p += 2 * block ) {
               const int32_t last = std::min( s.levels[ lv + 1 ], p + 2 * block );
               flags.push_back( ( last == s.levels[ lv + 1 ] ? kLastOfLevel : 0 ) |
                                ( ! inside && outside( lv, p, last, s.levels[ l ] ) ? kAllInRest : 0 ) |
                                ( len[ p ] > W ? kLongRow : 0 ) );  // the longest row is the first one
            }
         }
         addLaunch( l, e, block, flags.data() );
      }
      if( e < nl )
         addLaunch( e, e + 1, kRunBlock, nullptr );
      l = e + 1;
   }
   s.nslices = (int32_t) slices.size() / 4;
   s.order.upload( order, st );
   s.position.upload( position, st );
   s.levelsDevice.upload( s.levels, st );
   s.len.upload( len, st );
   s.sliceRest.upload( sliceRest, st );
   s.slices.upload( slices, st );
   s.steps.upload( steps, st );
   TNLHIP_CHECK( hipStreamSynchronize( st ) );  // the host vectors are local
}

template< typename T >
void factorize( const Ilu0::Sweep& s, const IluView< T >& f, hipStream_t st )
{
   const int32_t nl = (int32_t) s.levels.size() - 1;
   auto rows = [ & ]( int32_t l ) { return s.levels[ l + 1 ] - s.levels[ l ]; };
   for( int32_t l = 0; l < nl; ) {
      int32_t e = l + 1;
      if( rows( l ) > kNarrowFactor )
         factorLevelKernel< T ><<< gridFor( rows( l ), kIluBlock ), kIluBlock, 0, st >>>( f, s.order.ptr, s.levels[ l ],
                                                                                         s.levels[ e ] );
      else {
         while( e < nl && rows( e ) <= kNarrowFactor )
            e++;
         factorRunKernel< T ><<< 1, kRunBlock, 0, st >>>( f, s.order.ptr, s.levelsDevice.ptr, l, e );
      }
      l = e;
   }
   TNLHIP_CHECK( hipGetLastError() );
}

template< typename T >
void packSweep( Ilu0::Sweep& s, const int32_t* rp, const int32_t* c, const T* v, bool upper, hipStream_t st )
{
   const int32_t W = s.longRows ? kLongW : kShortW;
   s.slots.resize( (int64_t) slotWords( W ) * ( s.positions / 2 ) * 4 );
   s.val.resize( (int64_t) W * s.positions * (int64_t) sizeof( T ) );
   s.restCol.resize( s.rest );
   s.restVal.resize( (int64_t) s.rest * (int64_t) sizeof( T ) );
   if( upper )
      s.diag.resize( (int64_t) s.positions * (int64_t) sizeof( T ) );
   const unsigned grid = (unsigned) ( ( s.nslices + kIluBlock / kWave - 1 ) / ( kIluBlock / kWave ) );
   packKernel< T ><<< grid, kIluBlock, 0, st >>>(
      s.nslices, W, reinterpret_cast< const int4* >( s.slices.ptr ), s.order.ptr, s.position.ptr, rp, c, v, upper ? 1 : 0,
      s.len.ptr, reinterpret_cast< const int4* >( s.steps.ptr ), s.sliceRest.ptr,
      reinterpret_cast< uint16_t* >( s.slots.ptr ), reinterpret_cast< T* >( s.val.ptr ),
      reinterpret_cast< T* >( s.diag.ptr ), s.restCol.ptr, reinterpret_cast< T* >( s.restVal.ptr ) );
   TNLHIP_CHECK( hipGetLastError() );
}

template< bool UPPER, int W, int D, typename T >
void runSweep( const Ilu0::Sweep& s, T* x, Gate gate, hipStream_t st )
{
   const SweepView< T > f = sweepView< T >( s );
   for( const auto& L : s.launches ) {
      if( L.wide )
         sweepLevelKernel< UPPER, T ><<< gridFor( 2 * L.slices, kIluBlock / kWave ), kIluBlock, 0, st >>>(
            f, L.firstSlice, L.slices, s.levels[ L.firstLevel ], s.levels[ L.lastLevel ], x, gate );
      else
         sweepRunKernel< UPPER, W, D, T ><<< 1, L.block, 0, st >>>( f, L.firstStep, L.steps, x, gate );
   }
   TNLHIP_CHECK( hipGetLastError() );
}

template< bool UPPER, typename T >
void runSweep( const Ilu0::Sweep& s, T* x, Gate gate, hipStream_t st )
{
   if( s.longRows )
      runSweep< UPPER, kLongW, kLongD >( s, x, gate, st );
   else
      runSweep< UPPER, kShortW, kShortD >( s, x, gate, st );
}

template< typename T >
void permute( const DeviceArray< int32_t >& index, const T* src, T* dst, Gate gate, hipStream_t st )
{
   const int32_t n = (int32_t) index.size;
   permuteKernel< T ><<< gridFor( n, kIluBlock ), kIluBlock, 0, st >>>( n, index.ptr, src, dst, gate );
   TNLHIP_CHECK( hipGetLastError() );
}

template< typename T >
IluView< T > viewOf( const Ilu0& M )
{
   return IluView< T >{ M.Lrp.ptr, M.Lc.ptr, reinterpret_cast< T* >( M.Lv.ptr ),
                        M.Urp.ptr, M.Uc.ptr, reinterpret_cast< T* >( M.Uv.ptr ) };
}

template< typename T >
void factorizeAndPack( Ilu0& M, hipStream_t st )
{
   const IluView< T > f = viewOf< T >( M );
   factorize< T >( M.lower, f, st );
   packSweep< T >( M.lower, f.Lrp, f.Lc, f.Lv, false, st );
   packSweep< T >( M.upper, f.Urp, f.Uc, f.Uv, true, st );
   M.work.resize( ( (int64_t) M.lower.positions + M.upper.positions ) * (int64_t) sizeof( T ) );
}

template< typename T >
void solveSweeps( const Ilu0& M, const T* b, T* x, Gate gate, hipStream_t st )
{
   T* xl = reinterpret_cast< T* >( M.work.ptr );
   T* xu = xl + M.lower.positions;  // an even number of entries
   permute( M.lower.order, b, xl, gate, st );
   runSweep< false >( M.lower, xl, gate, st );
   permute( M.between, (const T*) xl, xu, gate, st );
   runSweep< true >( M.upper, xu, gate, st );
   permute( M.upper.position, (const T*) xu, x, gate, st );
}

template< typename T >
void uploadValues( DeviceArray< uint8_t >& dst, const std::vector< double >& v, hipStream_t st )
{
   std::vector< T > t( v.begin(), v.end() );
   dst.resize( (int64_t) t.size() * (int64_t) sizeof( T ) );
   if( ! t.empty() ) {
      TNLHIP_CHECK( hipMemcpyAsync( dst.ptr, t.data(), t.size() * sizeof( T ), hipMemcpyHostToDevice, st ) );
      TNLHIP_CHECK( hipStreamSynchronize( st ) );  // t lives on this frame
   }
}

}  // namespace

void Ilu0::build( const Matrix& A, int vectorDtype, hipStream_t st )
{
   TNLHIP_REQUIRE( A.rows == A.cols, "ILU(0) needs a square matrix" );
   if( A.symmetric )
      throw Error( TNLHIP_ERROR_UNSUPPORTED, "ILU(0) of a symmetric matrix (lower triangle stored) is not supported" );
   TNLHIP_REQUIRE( vectorDtype == TNLHIP_F64 || vectorDtype == TNLHIP_F32, "ILU(0) computes in double or float" );
   n = A.rows;
   dtype = vectorDtype;
   // the rows of A in storage order, stored zeros included
   std::vector< int32_t > rp( (size_t) n + 1, 0 ), cols;
   std::vector< double > vals;
   if( n > 0 ) {
      DeviceArray< int32_t > dcaps( n );
      capacitiesOf( A, dcaps.ptr, st );
      const std::vector< int32_t > caps = dcaps.download( st );
      for( int32_t i = 0; i < n; i++ )
         rp[ i + 1 ] = rp[ i ] + caps[ i ];
      DeviceArray< int32_t > drp, dcol( rp[ n ] );
      DeviceArray< double > dval( rp[ n ] );
      drp.upload( rp, st );
      gatherToCsr( A, drp.ptr, dcol.ptr, dval.ptr, st, true );
      cols = dcol.download( st );
      vals = dval.download( st );
   }
   // L / U split with TNL's counting rule (ILU0.hpp:36-50) and copy of the first entries
   std::vector< int32_t > lrp( (size_t) n + 1, 0 ), urp( (size_t) n + 1, 0 ), lc, uc;
   std::vector< double > lv, uv;
   for( int32_t i = 0; i < n; i++ ) {
      int32_t nl = 0, nu = 0;
      for( int32_t g = rp[ i ]; g < rp[ i + 1 ]; g++ ) {
         const int32_t c = cols[ g ];
         if( c < 0 )
            continue;
         if( c < i )
            nl++;
         else if( c < n )
            nu++;
         else
            break;
      }
      int32_t g = rp[ i ];
      while( g < rp[ i + 1 ] && cols[ g ] < 0 )
         g++;
      for( int32_t k = 0; k < nl; k++, g++ ) {
         if( cols[ g ] < 0 || cols[ g ] >= i )
            throw Error( TNLHIP_ERROR_UNSUPPORTED, "ILU(0): row " + std::to_string( i ) +
                                                      " does not store its columns below the diagonal first" );
         lc.push_back( cols[ g ] );
         lv.push_back( vals[ g ] );
      }
      for( int32_t k = 0; k < nu; k++, g++ ) {
         if( cols[ g ] < i || cols[ g ] >= n )
            throw Error( TNLHIP_ERROR_UNSUPPORTED, "ILU(0): row " + std::to_string( i ) +
                                                      " does not store its columns below the diagonal first" );
         uc.push_back( cols[ g ] );
         uv.push_back( vals[ g ] );
      }
      if( nu == 0 )
         throw Error( TNLHIP_ERROR_INVALID_ARGUMENT,
                      "ILU(0): row " + std::to_string( i ) + " has no entry on or above the diagonal" );
      lrp[ i + 1 ] = (int32_t) lc.size();
      urp[ i + 1 ] = (int32_t) uc.size();
   }
   // levels: forward / factorization over the L columns, backward over the U columns above i
   std::vector< int32_t > lo( n, 0 ), up( n, 0 );
   for( int32_t i = 0; i < n; i++ )
      for( int32_t c = lrp[ i ]; c < lrp[ i + 1 ]; c++ )
         lo[ i ] = std::max( lo[ i ], lo[ lc[ c ] ] + 1 );
   for( int32_t i = n - 1; i >= 0; i-- )
      for( int32_t c = urp[ i ]; c < urp[ i + 1 ]; c++ )
         if( uc[ c ] > i )
            up[ i ] = std::max( up[ i ], up[ uc[ c ] ] + 1 );
   std::vector< int32_t > ll( n ), ul( n ), orderL, orderU, positionL, positionU;
   for( int32_t i = 0; i < n; i++ ) {
      ll[ i ] = lrp[ i + 1 ] - lrp[ i ];
      ul[ i ] = urp[ i + 1 ] - urp[ i ] - 1;
   }
   buildSchedule( lower, lo, ll, [ & ]( int32_t i ) { return &lc[ lrp[ i ] ]; }, orderL, positionL, st );
   buildSchedule( upper, up, ul, [ & ]( int32_t i ) { return &uc[ urp[ i ] + 1 ]; }, orderU, positionU, st );
   std::vector< int32_t > mid( upper.positions );
   for( int32_t k = 0; k < upper.positions; k++ )
      mid[ k ] = positionL[ orderU[ k ] ];
   between.upload( mid, st );
   Lrp.upload( lrp, st );
   Urp.upload( urp, st );
   Lc.upload( lc, st );
   Uc.upload( uc, st );
   if( dtype == TNLHIP_F64 ) {
      uploadValues< double >( Lv, lv, st );
      uploadValues< double >( Uv, uv, st );
      if( n > 0 )
         factorizeAndPack< double >( *this, st );
   }
   else {
      uploadValues< float >( Lv, lv, st );
      uploadValues< float >( Uv, uv, st );
      if( n > 0 )
         factorizeAndPack< float >( *this, st );
   }
   TNLHIP_CHECK( hipStreamSynchronize( st ) );  // the host vectors are local
   // the solves read the packed copies only
   for( DeviceArray< int32_t >* a : { &Lrp, &Urp, &Lc, &Uc, &lower.slices, &upper.slices } )
      a->release();
   Lv.release();
   Uv.release();
}

void Ilu0::solve( const void* b, void* x, Gate gate, hipStream_t st ) const
{
   if( n == 0 )
      return;
   if( dtype == TNLHIP_F64 )
      solveSweeps( *this, (const double*) b, (double*) x, gate, st );
   else
      solveSweeps( *this, (const float*) b, (float*) x, gate, st );
}

}  // namespace tnlhip

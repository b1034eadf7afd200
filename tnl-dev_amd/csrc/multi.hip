// Product with several right-hand sides at once: Y = alpha A X + beta Y for k <= 64 columns.
//
// SparseMatrixView::vectorProduct (Matrices/SparseMatrixView.hpp:390-491) takes one vector; a
// caller with k of them (block Krylov methods, many time levels, the solve server's requests)
// would read the matrix k times.  Here the matrix is read once: X and Y are row-major (entry
// row * k + j), a row is taken by KP / VW lanes (KP = k rounded up to a power of two), each lane
// keeping VW adjacent right-hand sides.  multiProductKernel: VW is two FP64 or four FP32 columns, one
// 16-byte load and store, when k is a multiple of it and X, Y are 16-byte aligned, and 1 otherwise; the
// lanes of a row load the same stored element (one transaction) while their gathers of x at that column
// are contiguous, and each lane keeps 8 slots' loads in flight.  multiShortKernel, for matrices whose
// every row has at most 8 slots: several columns a lane whatever k and the alignment, slots shared through
// LDS, the next rows' loads under way (launchShort's rule).  Each column is summed left to right
// over the row's slots, rounding each product (TNL's Host order: CSRScalarKernel.hpp:70-107 and
// the padded formats' per-segment loops), so column j of Y equals TNL's product of column j of X
// bit for bit; padding slots (column -1) are skipped.  Keepers as SparseMatrixView.hpp:447-471.
#include "rowdist.hpp"
#include "spmv.hpp"

#include <algorithm>
#include <type_traits>

namespace tnlhip {

namespace {

constexpr int kMultiChunk = 8;  // slots of a row whose loads are in flight together
constexpr int64_t kMultiManyTiles = 100000;  // tiles from which a wave of the short-row kernel walks 8 of them

// Row blocks an XCD takes in a row before the next XCD's share begins.  A block gathers the X rows
// within the matrix's reach of it; where an XCD sweeps a contiguous eighth of the rows, two reaches of X
// rows pass through its L2 before one is read again.  A share of an eighth of the reach puts rows r - reach,
// r and r + reach on the same XCD with an eighth of that in between.  128^3 Laplacian, k = 16 in
// FP64 (reach 16384 rows, 2 MB of X): 239 us contiguous, 227 us in shares; where the window fits anyway
// (3 reaches within a MiB) and where the reach is that of the matrix, contiguous eighths stay.
int64_t multiChunk( const Matrix& M, int64_t blocks, int64_t rowsPerBlock, int64_t rowBytes )
{
   const int64_t whole = std::max< int64_t >( 1, ( blocks + kXcds - 1 ) / kXcds );
   // (ChunkedEllpack's and BiEllpack's kernels are bound by their index maps: 328 us contiguous against 342)
   const int kind = kindOf( M.format );
   if( kind == KIND_CHUNKED || kind == KIND_BIELLPACK || M.reach <= 0 || 3 * (int64_t) M.reach * rowBytes <= ( 1 << 20 ) )
      return whole;
   return std::min( whole, std::max< int64_t >( 1, ( M.reach / kXcds + rowsPerBlock - 1 ) / rowsPerBlock ) );
}

// The row block of this workgroup: in shares of `chunk` blocks, or, chunk 0, in contiguous eighths.  (A wave lives
// for a row or two: with the division for both FP32 k = 8 on the 1400^2 Laplacian took 45.1 us instead of 43.0.)
__device__ __forceinline__ int64_t multiBlock( int32_t chunk )
{
   const uint32_t xcd = blockIdx.x % kXcds, pos = blockIdx.x / kXcds;
   if( chunk == 0 )
      return (int64_t) xcd * ( gridDim.x / kXcds ) + pos;
   const uint32_t share = pos / (uint32_t) chunk;
   return (int64_t) ( share * kXcds + xcd ) * chunk + ( pos - share * (uint32_t) chunk );
}

// VW-wide vector of the compute type (VW = 1: the scalar itself)
template< typename A, int VW >
struct Lanes
{
   typedef A type __attribute__( ( ext_vector_type( VW ) ) );
};
template< typename A >
struct Lanes< A, 1 >
{
   typedef A type;
};

template< typename A, typename T >
__device__ __forceinline__ A lane( const T& v, int i )
{
   if constexpr( sizeof( T ) == sizeof( A ) )
      return v;
   else
      return v[ i ];
}

// A row is taken by L = KP / VW lanes; lane jq holds columns VW jq .. VW jq + VW - 1 of X and Y,
// loaded and stored VW at a time (VW > 1 only when k % VW == 0 and X, Y are 16-byte aligned).
// Workgroup b works on logical row block multiBlock( chunk ): the rows go to the XCDs in shares of `chunk`
// blocks, so that the x rows a block gathers stay in its XCD's L2 (the grid is a multiple of 8 shares;
// blocks past the last row exit).
template< int KP, int VW, typename V, typename A, typename Y, typename View >
__global__ __launch_bounds__( 256 ) void multiProductKernel( View view, const int32_t* __restrict__ col,
                                                             const V* __restrict__ val, int32_t k,
                                                             const Y* __restrict__ X, Y* __restrict__ Yout, A alpha,
                                                             A beta, int mode, int32_t first, int32_t last,
                                                             int32_t ncols, int32_t chunk )
{
   constexpr int L = KP / VW;
   constexpr int kRowsPerBlock = 256 / L;
   using VA = typename Lanes< A, VW >::type;
   using VY = typename Lanes< Y, VW >::type;
   const int jq = threadIdx.x % L;
   const int64_t r = first + multiBlock( chunk ) * kRowsPerBlock + threadIdx.x / L;
   if( r >= last )
      return;
   // no columns: every slot is padding and X may be empty
   const int32_t len = ncols > 0 ? view.size( (int32_t) r ) : 0;
   const int j0 = VW * jq;
   const bool mine = j0 < k;
   const Y* xs = X + ( mine ? j0 : 0 );
   VA sum = (VA) 0;
   for( int32_t l0 = 0; l0 < len; l0 += kMultiChunk ) {
      // the chunk's loads go out together: slots past the row re-read its last slot, padding and
      // lanes past k read row 0 of X; then the slots are summed left to right, each column on its own
      int32_t c[ kMultiChunk ];
      A a[ kMultiChunk ];
      VY xv[ kMultiChunk ];
#pragma unroll
      for( int u = 0; u < kMultiChunk; u++ ) {
         const int64_t g = view.global( (int32_t) r, min( l0 + u, len - 1 ) );
         c[ u ] = l0 + u < len ? col[ g ] : -1;
         a[ u ] = toCompute( val[ g ], A() );
      }
#pragma unroll
      for( int u = 0; u < kMultiChunk; u++ )
         xv[ u ] = *reinterpret_cast< const VY* >( xs + (int64_t) ( c[ u ] >= 0 ? c[ u ] : 0 ) * k );
#pragma unroll
      for( int u = 0; u < kMultiChunk; u++ )
         if( c[ u ] >= 0 ) {  // padding skipped
            if constexpr( VW == 1 )
               sum = mulAddExact( sum, a[ u ], (A) xv[ u ] );
            else
#pragma unroll
               for( int i = 0; i < VW; i++ )
                  sum[ i ] = mulAddExact( lane< A >( sum, i ), a[ u ], (A) lane< Y >( xv[ u ], i ) );
         }
   }
   if( ! mine )
      return;
   Y* out = Yout + r * k + j0;
   VY o;
   if constexpr( VW == 1 )
      o = mode >= 2 ? *out : (Y) 0;
   else
      o = mode >= 2 ? *reinterpret_cast< const VY* >( out ) : (VY) 0;
#pragma unroll
   for( int i = 0; i < VW; i++ ) {
      const A sv = lane< A >( sum, i );
      A v;
      switch( mode ) {
         case 0: v = sv; break;
         case 1: v = alpha * sv; break;
         case 2: v = beta * (A) lane< Y >( o, i ) + sv; break;
         default: v = beta * (A) lane< Y >( o, i ) + alpha * sv; break;
      }
      if constexpr( VW == 1 )
         o = (Y) v;
      else
         o[ i ] = (Y) v;
   }
   if constexpr( VW == 1 )
      *out = o;
   else
      *reinterpret_cast< VY* >( out ) = o;
}

template< int KP, int VW, typename V, typename A, typename Y >
void launchMultiW( const Matrix& M, int32_t k, const Y* X, Y* Yv, double alpha, double beta, int32_t first,
                   int32_t last, hipStream_t st )
{
   int mode;
   if( beta == 0.0 )
      mode = alpha == 1.0 ? 0 : 1;
   else
      mode = alpha == 1.0 ? 2 : 3;
   constexpr int kRowsPerBlock = 256 / ( KP / VW );
   const int64_t rows = last - first;
   int64_t blocks = ( rows + kRowsPerBlock - 1 ) / kRowsPerBlock;
   const int64_t chunk = multiChunk( M, blocks, kRowsPerBlock, (int64_t) k * sizeof( Y ) );
   blocks = ( blocks + kXcds * chunk - 1 ) / ( kXcds * chunk ) * ( kXcds * chunk );
   TNLHIP_REQUIRE( blocks < ( 1ll << 31 ), "too many rows for one launch" );
   withView( M, [ & ]( auto view ) {
      multiProductKernel< KP, VW, V, A, Y ><<< (unsigned) blocks, 256, 0, st >>>(
         view, M.columns.ptr, reinterpret_cast< const V* >( M.values.ptr ), k, X, Yv, (A) alpha, (A) beta, mode, first,
         last, M.cols, blocks == kXcds * chunk ? 0 : (int32_t) chunk );
   } );
   TNLHIP_CHECK( hipGetLastError() );
}

// ------------------------------------------------------------------ short rows

// The words a lane loads to address the slots of one row, for the formats whose rows are one run of
// equal steps (CSR, Ellpack, SlicedEllpack).  They are kept as loaded and combined where they are used:
// arithmetic on them at the load would wait for it, and with it for every load under way.
struct RowRun
{
   int32_t a = 0, b = 0;
};
__device__ __forceinline__ RowRun rowRun( const CsrView& v, int32_t r )
{
   return RowRun{ v.offsets[ r ], v.offsets[ r + 1 ] };
}
__device__ __forceinline__ RowRun rowRun( const EllpackView& v, int32_t ) { return RowRun{ 0, v.segmentSize }; }
__device__ __forceinline__ RowRun rowRun( const SlicedView& v, int32_t r )
{
   return RowRun{ v.sliceOffsets[ r >> v.logSlice ], v.sliceSizes[ r >> v.logSlice ] };
}
__device__ __forceinline__ int32_t runSize( const CsrView&, RowRun m ) { return m.b - m.a; }
__device__ __forceinline__ int32_t runSize( const EllpackView&, RowRun m ) { return m.b; }
__device__ __forceinline__ int32_t runSize( const SlicedView&, RowRun m ) { return m.b; }
__device__ __forceinline__ int64_t runStart( const CsrView&, RowRun m, int64_t ) { return m.a; }
__device__ __forceinline__ int64_t runStart( const EllpackView&, RowRun, int64_t r ) { return r; }
__device__ __forceinline__ int64_t runStart( const SlicedView& v, RowRun m, int64_t r )
{
   return m.a + ( r & ( ( 1 << v.logSlice ) - 1 ) );
}
__device__ __forceinline__ int64_t runStep( const CsrView& ) { return 1; }
__device__ __forceinline__ int64_t runStep( const EllpackView& v ) { return v.alignedSize; }
__device__ __forceinline__ int64_t runStep( const SlicedView& v ) { return (int64_t) 1 << v.logSlice; }

template< typename View >
constexpr bool kRunView = std::is_same_v< View, CsrView > || std::is_same_v< View, EllpackView > ||
                          std::is_same_v< View, SlicedView >;

// VW adjacent entries wherever they start (global loads need only element alignment)
template< typename Y, int VW >
struct Packed
{
   typedef Y type __attribute__( ( ext_vector_type( VW ), aligned( sizeof( Y ) ) ) );
};

// The product where no row has more than kMultiChunk slots.  Bound by latency before it is bound by bytes: in multiProductKernel a wave lives
// for one row per L lanes, through three dependent trips to memory (row, slots, X).  Here a
// wave walks `tiles` tiles of 64 / L rows with the next tile's slots and the one after's row
// loaded ahead, and X of the next tile under way while it sums this one.  A tile's slots are
// loaded once, one lane each, and shared through wave-local LDS; the L lanes of a row read them
// there.  Lane jq of a row takes columns j0 .. j0 + VW - 1, j0 = VW jq; when VW does not divide k the last
// lane starts early enough to end at column k - 1 and stores only its own columns.  Every column is
// summed left to right in the Host order, as in multiProductKernel.
// 128^3 Laplacian, SlicedEllpack FP64, k = 16: 239 -> 209 us
template< int L, int VW, typename V, typename A, typename Y, typename View >
__global__ __launch_bounds__( 256 ) void multiShortKernel( View view, const int32_t* __restrict__ col,
                                                           const V* __restrict__ val, int32_t k,
                                                           const Y* __restrict__ X, Y* __restrict__ Yout, A alpha,
                                                           A beta, int mode, int32_t first, int32_t last,
                                                           int32_t ncols, int32_t chunk, int32_t tiles )
{
   constexpr int RW = kWave / L;  // rows of a tile
   constexpr int S = kMultiChunk;
   constexpr int PL = L >= S ? 1 : S / L;  // slots a lane loads
   constexpr int kWaves = 256 / kWave;
   using VY = typename Packed< Y, VW >::type;
   __shared__ __align__( 16 ) int32_t sc[ kWaves ][ 2 ][ RW * S ];
   __shared__ __align__( 16 ) A sv[ kWaves ][ 2 ][ RW * S ];
   const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
   const int loadRow = lane % RW, loadSlot = lane / RW;  // as a loader: slots loadSlot, loadSlot + L, ...
   const int myRow = lane / L, jq = lane % L;            // as a summer
   const bool mine = VW * jq < k;
   const int j0 = mine ? min( VW * jq, k - VW ) : 0;
   const int64_t step = runStep( view );
   // a workgroup takes `tiles` consecutive blocks of kWaves tiles, in the order of multiBlock
   int64_t block = multiBlock( chunk ) * tiles;
   auto nextBase = [ & ] {  // first row of the wave's next tile (past the last one: no rows)
      const int64_t base = first + ( block * kWaves + wave ) * RW;
      block++;
      return base;
   };
   auto loadRun = [ & ]( int64_t base ) {
      const int64_t r = base + loadRow;
      RowRun m;
      if( r < last )
         m = rowRun( view, (int32_t) r );
      return m;
   };
   struct Slots
   {
      int32_t c[ PL ];
      V v[ PL ];
   };
   auto loadSlots = [ & ]( RowRun m, int64_t base ) {
      Slots s;
      const int32_t size = base + loadRow < last ? runSize( view, m ) : 0;
      const int64_t start = runStart( view, m, base + loadRow );
#pragma unroll
      for( int j = 0; j < PL; j++ ) {
         const int l = loadSlot + j * L;
         s.c[ j ] = -1;
         s.v[ j ] = V( 0.0f );
         if( l < S && l < size ) {
            const int64_t g = start + step * l;
            s.c[ j ] = __builtin_nontemporal_load( col + g );
            s.v[ j ] = val[ g ];
         }
      }
      return s;
   };
   auto share = [ & ]( int buf, const Slots& s ) {
      waveSync();
#pragma unroll
      for( int j = 0; j < PL; j++ ) {
         const int l = loadSlot + j * L;
         if( l < S ) {
            sc[ wave ][ buf ][ loadRow * S + l ] = s.c[ j ];
            sv[ wave ][ buf ][ loadRow * S + l ] = toCompute( s.v[ j ], A() );
         }
      }
      waveSync();
   };
   struct Gathered
   {
      VY x[ S ];
      VY y;
   };
   const Y* xs = X + j0;
   auto gather = [ & ]( int buf, int64_t base, Gathered& g ) {
      const int64_t r = min( base + myRow, (int64_t) last - 1 );
      const int32_t spare = (int32_t) min( r, (int64_t) ncols - 1 );  // padding reads a row that is read anyway
#pragma unroll
      for( int u = 0; u < S; u++ ) {
         const int32_t c = sc[ wave ][ buf ][ myRow * S + u ];
         g.x[ u ] = *reinterpret_cast< const VY* >( xs + (int64_t) ( c >= 0 ? c : spare ) * k );
      }
      if( mode >= 2 )
         g.y = *reinterpret_cast< const VY* >( Yout + r * k + j0 );
   };
   auto finish = [ & ]( int buf, int64_t base, const Gathered& g ) {
      const int64_t r = base + myRow;
      A sum[ VW ] = {};
#pragma unroll
      for( int u = 0; u < S; u++ ) {
         const int32_t c = sc[ wave ][ buf ][ myRow * S + u ];
         const A a = sv[ wave ][ buf ][ myRow * S + u ];
#pragma unroll
         for( int i = 0; i < VW; i++ )
            sum[ i ] = c >= 0 ? mulAddExact( sum[ i ], a, (A) g.x[ u ][ i ] ) : sum[ i ];
      }
      if( ! mine || r >= last )
         return;
      VY o;
#pragma unroll
      for( int i = 0; i < VW; i++ ) {
         A v;
         switch( mode ) {
            case 0: v = sum[ i ]; break;
            case 1: v = alpha * sum[ i ]; break;
            case 2: v = beta * (A) g.y[ i ] + sum[ i ]; break;
            default: v = beta * (A) g.y[ i ] + alpha * sum[ i ]; break;
         }
         o[ i ] = (Y) v;
      }
      Y* out = Yout + r * k + j0;
      if( j0 == VW * jq )
         *reinterpret_cast< VY* >( out ) = o;
      else {
#pragma unroll
         for( int i = 0; i < VW; i++ )
            if( j0 + i >= VW * jq )
               out[ i ] = o[ i ];
      }
   };
   // while a tile (base b0) is summed, X of the next (b1) is under way, the slots of the one after (b2)
   // and the row starts of the one after that (b3) are loading
   int64_t b0 = nextBase(), b1 = nextBase(), b2 = nextBase(), b3;
   RowRun m = loadRun( b0 );
   Slots s = loadSlots( m, b0 );
   m = loadRun( b1 );
   Gathered g0, g1;
   share( 0, s );
   s = loadSlots( m, b1 );
   m = loadRun( b2 );
   gather( 0, b0, g0 );
   for( int t = 0; t < tiles; t += 2 ) {
      b3 = nextBase();
      share( 1, s );
      s = loadSlots( m, b2 );
      m = loadRun( b3 );
      gather( 1, b1, g1 );
      finish( 0, b0, g0 );
      b0 = nextBase();
      share( 0, s );
      s = loadSlots( m, b3 );
      m = loadRun( b0 );
      gather( 0, b2, g0 );
      finish( 1, b1, g1 );
      b1 = b3;
      const int64_t b4 = b0;
      b0 = b2;
      b2 = b4;
   }
}

template< int L, int VW, typename V, typename A, typename Y, typename View >
void launchMultiShort( const Matrix& M, const View& view, int32_t k, const Y* X, Y* Yv, double alpha, double beta,
                       int32_t first, int32_t last, hipStream_t st )
{
   const int mode = beta == 0.0 ? ( alpha == 1.0 ? 0 : 1 ) : ( alpha == 1.0 ? 2 : 3 );
   constexpr int RW = kWave / L;
   constexpr int kWaves = 256 / kWave;
   const int64_t all = ( (int64_t) last - first + RW - 1 ) / RW;
   // X of one tile past a wave's last is gathered for nothing: many tiles a wave where there are enough
   const int64_t tiles = all >= kMultiManyTiles ? 8 : 2;
   const int64_t perBlock = tiles * kWaves;
   int64_t blocks = ( all + perBlock - 1 ) / perBlock;
   const int64_t chunk = multiChunk( M, blocks, perBlock * RW, (int64_t) k * sizeof( Y ) );
   blocks = ( blocks + kXcds * chunk - 1 ) / ( kXcds * chunk ) * ( kXcds * chunk );
   TNLHIP_REQUIRE( blocks < ( 1ll << 31 ), "too many rows for one launch" );
   multiShortKernel< L, VW, V, A, Y ><<< (unsigned) blocks, 256, 0, st >>>(
      view, M.columns.ptr, reinterpret_cast< const V* >( M.values.ptr ), k, X, Yv, (A) alpha, (A) beta, mode, first,
      last, M.cols, blocks == kXcds * chunk ? 0 : (int32_t) chunk, (int32_t) tiles );
   TNLHIP_CHECK( hipGetLastError() );
}

// Takes the product of short rows where it is the faster one; false: it is the other kernel's.  us, other kernel /
// this one, SlicedEllpack: FP64 on the 128^3 Laplacian k = 3 97 / 62, 4 67 / 63, 7 196 / 114, 8 127 / 115,
// 12 227 / 177, 16 239 / 209, 32 474 / 403; on the 1400^2 one k = 4 40 / 57, 8 114 / 101, 16 221 / 179; on
// the 64^3 one k = 7 22.5 / 18.8, 8 14.3 / 18.7, 16 23.5 / 25.8.  FP32 128^3 k = 7 111 / 62, 8 41 / 58,
// 16 110 / 110; CSRScalar FP64 k = 3 on 127 x 150 x 93 67 / 69, FP32 k = 3 on 128^3 43 / 61.  So it
// takes the widths that 16-byte lanes do not divide (k = 3 only where FP64 slots lie slice by slice, from a
// million rows on), and from four lanes a row (two FP64 columns each) on where there are rows enough to
// walk.  Rows beyond kMultiChunk slots would hold up a wave's whole walk: finished in a loop of their own here, one
// row of 20000 slots among 300000 of 3 cost 6343 us instead of 1736 (k = 7), lognormal rows of 6 on average 702
// instead of 271.
template< int KP, typename V, typename A, typename Y >
bool launchShort( const Matrix& M, int32_t k, const Y* X, Y* Yv, double alpha, double beta, int32_t first, int32_t last,
                  bool wide, hipStream_t st )
{
   constexpr int VW = KP <= 2 ? 2 : std::min( 16 / (int) sizeof( Y ), KP / 2 );
   constexpr int L = KP / VW;
   const int64_t rows = (int64_t) last - first;
   if( wide && ( sizeof( Y ) != 8 || L < 4 || rows * L / kWave < kMultiManyTiles ) )
      return false;
   if( rows < 200000 )  // FP32 k = 7, CSR: 132000 rows 9.5 / 10.5, 262000 rows 16.5 / 13.6
      return false;
   if( KP == 4 && ( sizeof( Y ) != 8 || kindOf( M.format ) == KIND_CSR || rows < 1000000 ) )
      return false;
   if constexpr( L >= 2 ) {
      if( M.cols == 0 || M.meta.rowMost > kMultiChunk )
         return false;
      bool taken = false;
      withView( M, [ & ]( auto view ) {
         if constexpr( kRunView< decltype( view ) > ) {
            launchMultiShort< L, VW, V, A, Y >( M, view, k, X, Yv, alpha, beta, first, last, st );
            taken = true;
         }
      } );
      return taken;
   }
   return false;
}

// 16-byte lanes (two FP64 or four FP32 columns) when k allows them and X, Y are 16-byte aligned
template< int KP, typename V, typename A, typename Y >
void launchMulti( const Matrix& M, int32_t k, const Y* X, Y* Yv, double alpha, double beta, int32_t first,
                  int32_t last, hipStream_t st )
{
   constexpr int VW = 16 / (int) sizeof( Y ) < KP ? 16 / (int) sizeof( Y ) : KP;
   const bool aligned = ( ( reinterpret_cast< uintptr_t >( X ) | reinterpret_cast< uintptr_t >( Yv ) ) % 16 ) == 0;
   const bool wide = VW > 1 && k % VW == 0 && aligned;
   if( launchShort< KP, V, A, Y >( M, k, X, Yv, alpha, beta, first, last, wide, st ) )
      return;
   if constexpr( VW > 1 ) {
      if( wide ) {
         launchMultiW< KP, VW, V, A, Y >( M, k, X, Yv, alpha, beta, first, last, st );
         return;
      }
   }
   launchMultiW< KP, 1, V, A, Y >( M, k, X, Yv, alpha, beta, first, last, st );
}

template< typename V, typename A, typename Y >
void dispatchK( const Matrix& M, int32_t k, const Y* X, Y* Yv, double alpha, double beta, int32_t first, int32_t last,
                hipStream_t st )
{
   if( k <= 1 )
      launchMulti< 1, V, A, Y >( M, k, X, Yv, alpha, beta, first, last, st );
   else if( k <= 2 )
      launchMulti< 2, V, A, Y >( M, k, X, Yv, alpha, beta, first, last, st );
   else if( k <= 4 )
      launchMulti< 4, V, A, Y >( M, k, X, Yv, alpha, beta, first, last, st );
   else if( k <= 8 )
      launchMulti< 8, V, A, Y >( M, k, X, Yv, alpha, beta, first, last, st );
   else if( k <= 16 )
      launchMulti< 16, V, A, Y >( M, k, X, Yv, alpha, beta, first, last, st );
   else if( k <= 32 )
      launchMulti< 32, V, A, Y >( M, k, X, Yv, alpha, beta, first, last, st );
   else
      launchMulti< 64, V, A, Y >( M, k, X, Yv, alpha, beta, first, last, st );
}

}  // namespace

void spmvMultiLaunch( const Matrix& M, int32_t k, const void* X, void* Yv, double alpha, double beta, int32_t first,
                      int32_t last, hipStream_t st )
{
   if( M.symmetric || M.dtype == TNLHIP_BINARY )
      throw Error( TNLHIP_ERROR_UNSUPPORTED, "products with several right-hand sides take general real-valued matrices" );
   TNLHIP_REQUIRE( k >= 1 && k <= kMaxMultiRhs, "the number of right-hand sides must be in [1, 64]" );
   if( last <= first )
      return;
   switch( M.dtype ) {
      case TNLHIP_F64:
         dispatchK< double, double, double >( M, k, (const double*) X, (double*) Yv, alpha, beta, first, last, st );
         break;
      case TNLHIP_F32:
         dispatchK< float, float, float >( M, k, (const float*) X, (float*) Yv, alpha, beta, first, last, st );
         break;
      default:
         dispatchK< bf16, float, float >( M, k, (const float*) X, (float*) Yv, alpha, beta, first, last, st );
         break;
   }
}

}  // namespace tnlhip

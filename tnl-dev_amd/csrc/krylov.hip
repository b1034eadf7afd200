// Products fused with the vector passes around them (krylov.hpp): the row kernels of
// spmv_kernels.hpp with a keeper that divides by the Jacobi diagonal, stores the entry and adds up the
// operand's sums, and operands that are formed where they are gathered.
#include "krylov.hpp"
#include "spmv_kernels.hpp"

namespace tnlhip {

namespace {

template< typename A, typename Y, typename Op >
struct FusedKeeper
{
   static constexpr bool kPlain = false;
   static constexpr bool kStored = Op::kStored;
   Op op;
   const Y* diag;
   Y* y;
   ReduceSlot out;
   Gate gate;
   double acc[ Op::kSums ] = {};
   __device__ __forceinline__ bool shut() const
   {
      if constexpr( Op::kStored )
         return Op::shut( gate );
      return false;
   }
   __device__ __forceinline__ void prefetch() { op.prefetch( gate ); }
   __device__ __forceinline__ bool begin() { return op.begin(); }
   __device__ __forceinline__ Y at( const Y* x, int64_t c ) const { return op.at( x, c ); }
   __device__ __forceinline__ void operator()( int64_t row, A v )
   {
      const Y o = diag ? (Y) ( v / (A) diag[ row ] ) : (Y) v;
      y[ row ] = o;
      op.row( row, o, acc );
   }
   __device__ __forceinline__ void finish() const { storeBlockPartials< Op::kSums >( acc, out ); }
};

}  // namespace

int fusedGrid( const Matrix& A, bool twoProducts )
{
   if( A.symmetric || ( A.dtype != TNLHIP_F64 && A.dtype != TNLHIP_F32 ) || A.meta.allocated == 0 )
      return 0;
   // With 32 or 64 lanes a row one lane in so many adds up a wave's dots, behind the row's sum; launches saved pay for
   // it only where they count.  us per iteration, separate passes / fused, 27-point box, CSRLight (32 lanes) FP64: CG
   // 40^3 25.5 / 24.4, 52^3 34.4 / 34.5, 90^3 86.1 / 95.5; BiCGStab 52^3 70.6 / 58.5, 90^3 168 / 172; CSRVector (64
   // lanes) CG 52^3 47.3 / 49.8, 90^3 176 / 197, BiCGStab 500000 rows of 40 entries 365 / 366, 90^3 343 / 364.
   if( kindOf( A.format ) == KIND_CSR && A.format != TNLHIP_CSR_ADAPTIVE && lanesPerRow( A ) >= 32 &&
       A.rows > ( twoProducts ? 500000 : 100000 ) )
      return 0;
   unsigned grid;
   if( A.dtype == TNLHIP_F64 )
      grid = launchProduct< double, double, double >( A, nullptr, FusedKeeper< double, double, DotOperand< double > >{}, 0,
                                                      A.rows, nullptr, true );
   else
      grid = launchProduct< float, float, float >( A, nullptr, FusedKeeper< float, float, DotOperand< float > >{}, 0,
                                                   A.rows, nullptr, true );
   // one workgroup takes 256 short CSR rows: the workgroup barrier of the sums costs FP32 rows more than
   // the dot's pass did beyond a million of them (128^3 CG 59.7 against 56.1 us per iteration; FP64 78.1
   // against 80.5)
   const unsigned most = A.dtype == TNLHIP_F32 && kindOf( A.format ) == KIND_CSR ? kMaxFusedPartials / 2
                                                                                 : kMaxFusedPartials;
   return grid <= most ? (int) grid : 0;
}

// Forming the operand in the product saves a launch and its pass (about 2 us) and costs a gather of
// each of its vectors per stored element instead of one.  us per iteration, operand formed in the
// product / in a pass of its own: CG 2D 256^2 11.2 / 13.3 (SlicedEllpack), 11.9 / 13.2 (CSRScalar);
// 64^3 14.9 / 16.5, 18.9 / 18.8; 80^3 26.4 / 26.8, 30.6 / 30.2; 100^3 42.3 / 41.1, 48.2 / 42.3.
// BiCGStab (three vectors) 256^2 20.0 / 23.0, 20.6 / 22.3; 64^3 28.5 / 29.2, 34.9 / 35.3; 80^3
// 49.8 / 46.9, 62.7 / 53.1.  So it pays while the launches count: up to 300000 short rows, in CSR only where no
// lane walks a row (200000 rows of 3 with one of 20000, CG: 5645 / 4739) and no lane group shares one (65^3, 8 and 64
// lanes, CG: 34.5 / 32.3 and 84.6 / 76.7).
bool fuseOperand( const Matrix& A )
{
   if( A.meta.allocated > (int64_t) kShortRow * A.rows || A.rows > 300000 )
      return false;
   if( kindOf( A.format ) != KIND_CSR )
      return true;
   return A.dtype == TNLHIP_F64 ? stagedThroughout< double >( A ) : stagedThroughout< float >( A );
}

template< typename T, typename Op >
void fusedProduct( const Matrix& A, const Op& op, const T* x, const T* diag, T* y, ReduceSlot out, Gate gate,
                   hipStream_t stream )
{
   launchProduct< T, T, T >( A, x, FusedKeeper< T, T, Op >{ op, diag, y, out, gate }, 0, A.rows, stream );
}

#define TNLHIP_FUSED( T, OP )                                                                                      \
   template void fusedProduct< T, OP< T > >( const Matrix&, const OP< T >&, const T*, const T*, T*, ReduceSlot, Gate, \
                                             hipStream_t );
#define TNLHIP_FUSED_ALL( T )           \
   TNLHIP_FUSED( T, CgDirectionOperand ) \
   TNLHIP_FUSED( T, DotOperand )        \
   TNLHIP_FUSED( T, DotSquareOperand )  \
   TNLHIP_FUSED( T, BiDirectionOperand ) \
   TNLHIP_FUSED( T, BiSOperand )
TNLHIP_FUSED_ALL( double )
TNLHIP_FUSED_ALL( float )

}  // namespace tnlhip

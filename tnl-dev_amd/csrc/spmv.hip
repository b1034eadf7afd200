// Sparse matrix-vector product y = alpha * A x + beta * y over every segment format: the keeper of a
// product and the dispatch on the value type.  The row kernels are in spmv_kernels.hpp.
#include "spmv_kernels.hpp"

namespace tnlhip {

// ------------------------------------------------------------------ dispatch

namespace {

template< typename V, typename A, typename Y >
void launchTyped( const Matrix& M, const Y* x, Y* y, double alpha, double beta, int32_t first, int32_t last,
                  const Y* diag, const int32_t* gate, int gateMode, hipStream_t st, const Y* rhs = nullptr,
                  const Y* prev = nullptr )
{
   Keeper< A, Y > keep{ y, (A) alpha, (A) beta, diag, 0, gate, gate ? gateMode : 0 };
   if( rhs ) {
      keep.mode = 5;
      keep.rhs = rhs;
      keep.prev = prev;
   }
   else if( diag )
      keep.mode = 4;
   else if( beta == 0.0 )
      keep.mode = alpha == 1.0 ? 0 : 1;
   else
      keep.mode = alpha == 1.0 ? 2 : 3;
   launchProduct< V, A, Y >( M, x, keep, first, last, st );
}

}  // namespace

void spmvLaunchGated( const Matrix& A, const void* x, void* y, double alpha, double beta, const void* diag,
                      const int32_t* gate, int gateMode, hipStream_t stream, int32_t first, int32_t last )
{
   if( last < 0 )
      last = A.rows;
   if( A.dtype == TNLHIP_BINARY ) {
      if( A.symmetric || diag )
         throw Error( TNLHIP_ERROR_UNSUPPORTED, "symmetric binary matrices and preconditioned binary products" );
      spmvBinary( A, x, y, alpha, beta, first, last, Gate{ gate, gate ? gateMode : 0 }, stream );
      return;
   }
   if( A.symmetric ) {
      spmvSymmetric( A, x, y, alpha, beta, first, last, diag, Gate{ gate, gate ? gateMode : 0 }, stream );
      return;
   }
   switch( A.dtype ) {
      case TNLHIP_F64:
         launchTyped< double, double, double >( A, (const double*) x, (double*) y, alpha, beta, first, last,
                                                (const double*) diag, gate, gateMode, stream );
         break;
      case TNLHIP_F32:
         launchTyped< float, float, float >( A, (const float*) x, (float*) y, alpha, beta, first, last,
                                             (const float*) diag, gate, gateMode, stream );
         break;
      case TNLHIP_BF16:
         launchTyped< bf16, float, float >( A, (const float*) x, (float*) y, alpha, beta, first, last,
                                            (const float*) diag, gate, gateMode, stream );
         break;
      default: throw Error( TNLHIP_ERROR_INVALID_ARGUMENT, "unknown value type" );
   }
}

void spmvJacobiStepGated( const Matrix& P, const void* z, void* znew, const void* rhs, const void* diag,
                          const int32_t* gate, int gateMode, hipStream_t stream )
{
   if( P.dtype == TNLHIP_BINARY || P.symmetric )
      throw Error( TNLHIP_ERROR_UNSUPPORTED, "the Jacobi-polynomial preconditioner needs a general real-valued matrix" );
   TNLHIP_REQUIRE( z != znew && rhs != znew, "a Jacobi step writes a vector of its own" );
   switch( P.dtype ) {
      case TNLHIP_F64:
         launchTyped< double, double, double >( P, (const double*) z, (double*) znew, 1.0, 0.0, 0, P.rows,
                                                (const double*) diag, gate, gateMode, stream, (const double*) rhs,
                                                (const double*) z );
         break;
      case TNLHIP_F32:
         launchTyped< float, float, float >( P, (const float*) z, (float*) znew, 1.0, 0.0, 0, P.rows,
                                             (const float*) diag, gate, gateMode, stream, (const float*) rhs,
                                             (const float*) z );
         break;
      default:
         launchTyped< bf16, float, float >( P, (const float*) z, (float*) znew, 1.0, 0.0, 0, P.rows,
                                            (const float*) diag, gate, gateMode, stream, (const float*) rhs,
                                            (const float*) z );
         break;
   }
}

bool quotientProduct( const Matrix& A )
{
   return A.dtype != TNLHIP_BINARY && ! A.symmetric && ! A.stripes;
}

void spmvQuotientGated( const Matrix& A, const void* x, void* y, void* quotient, const void* diag,
                        const int32_t* gate, int gateMode, hipStream_t stream )
{
   if( ! quotientProduct( A ) )
      throw Error( TNLHIP_ERROR_UNSUPPORTED, "products with a quotient take general real-valued matrices without a "
                                             "striped plan" );
   TNLHIP_REQUIRE( y != quotient, "the product and its quotient are two vectors" );
   auto launch = [ & ]( auto* tagV, auto* tagY ) {
      using V = std::remove_pointer_t< decltype( tagV ) >;
      using Y = std::remove_pointer_t< decltype( tagY ) >;
      const QuotientKeeper< Y, Y > keep{ { (Y*) y, (Y) 1, (Y) 0, (const Y*) diag, 0, gate, gate ? gateMode : 0 },
                                         (Y*) quotient };
      launchProduct< V, Y, Y >( A, (const Y*) x, keep, 0, A.rows, stream );
   };
   switch( A.dtype ) {
      case TNLHIP_F64: launch( (double*) nullptr, (double*) nullptr ); break;
      case TNLHIP_F32: launch( (float*) nullptr, (float*) nullptr ); break;
      default: launch( (bf16*) nullptr, (float*) nullptr ); break;
   }
}

void spmvLaunch( const Matrix& A, const void* x, void* y, double alpha, double beta, int32_t first, int32_t last,
                 const void* diag, hipStream_t stream )
{
   spmvLaunchGated( A, x, y, alpha, beta, diag, nullptr, 0, stream, first, last );
}

}  // namespace tnlhip

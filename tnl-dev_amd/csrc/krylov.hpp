// Device state of a Krylov solve and the products that CG and BiCGStab fuse with the vector passes
// around them (krylov.hip).
//
// One product of a Krylov step is followed by a dot product with its result, and preceded by the
// vector update that makes its operand.  Both fit into the row kernels: each workgroup adds up its
// rows' share of the dot and stores one partial, and the operand can be formed where it is
// gathered (p[c] = z[c] + beta p_old[c]), each row's own entry being stored for the passes that
// follow.  The scalars come from the partials of the launch before, summed by every workgroup in
// the same order (Fold), so there are no launches for them either.  A CG iteration is then two
// launches and a BiCGStab iteration three.
#pragma once

#include "blas.hpp"
#include "matrix.hpp"

#include <algorithm>

namespace tnlhip {

// ------------------------------------------------------------------ device state

struct State
{
   double normb, residue, s1, s2, alpha, beta, omega, rho, rho_old, r_ast_sqnorm, normw, tmp, beta_gm;
   double pad_;
   int32_t it;
   int32_t flags[ 2 ];  // [0] done (stop this solve / this GMRES cycle), [1] auxiliary gate
   int32_t histLen;
   int32_t o_steps;
   int32_t breakdown;
   int32_t stop;  // solve finished (GMRES: the outer loop must not continue)
   int32_t started;  // fused BiCGStab: 0 before the first direction, 2 after a restart, else 1
};

struct Stop
{
   int32_t maxIt, minIt;
   double conv, div;
};

// IterativeSolver::checkNextIteration (IterativeSolver.hpp:116-124)
__device__ __forceinline__ bool checkNext( const State& s, const Stop& p )
{
   const double r = s.residue;
   return ! ( isnan( r ) || s.it > p.maxIt || ( r > p.div && s.it >= p.minIt ) || ( r < p.conv && s.it >= p.minIt ) );
}

// IterativeSolver::setResidue with the residual history (IterativeSolver.hpp:189-200): each call
// records (residue, the iteration count at that moment), the two fields of a history-file line
__device__ __forceinline__ void setResidue( State& s, double r, double* hist, int64_t cap )
{
   s.residue = r;
   if( s.histLen < cap ) {
      hist[ 2 * (int64_t) s.histLen ] = r;
      hist[ 2 * (int64_t) s.histLen + 1 ] = (double) s.it;
   }
   s.histLen++;
}

// setResidue, checkNext and the count of the next iteration by a lane that holds the state's
// counters already: stores only, where the separate calls are a chain of loads and stores
__device__ __forceinline__ void recordStep( State& s, double r, int32_t it, int32_t histLen, double* hist,
                                            int64_t cap, const Stop& p )
{
   s.residue = r;
   if( histLen < cap ) {
      hist[ 2 * (int64_t) histLen ] = r;
      hist[ 2 * (int64_t) histLen + 1 ] = (double) it;
   }
   s.histLen = histLen + 1;
   if( isnan( r ) || it > p.maxIt || ( r > p.div && it >= p.minIt ) || ( r < p.conv && it >= p.minIt ) )
      s.flags[ 0 ] = 1;
   s.it = it + 1;
}

// ------------------------------------------------------------------ folded sums

// The sum a reduction's final kernel would form, formed instead by every workgroup of the next
// kernel from the same partials in the same order (sumPartials), so each workgroup holds the
// same bits; the next kernel's workgroup 0 then does the final kernel's state update.  It saves
// the final kernel's launch; no workgroup may read a state field that workgroup 0 of the same
// launch writes.
__device__ __forceinline__ double foldPartials1( ReduceSlot slot, int grid )
{
   __shared__ double tot[ 1 ];
   sumPartials< 1 >( slot, grid, tot );
   return tot[ 0 ];
}

__device__ __forceinline__ void foldPartials2( ReduceSlot slot, int grid, double ( &v )[ 2 ] )
{
   __shared__ double tot[ 2 ];
   sumPartials< 2 >( slot, grid, tot );
   v[ 0 ] = tot[ 0 ];
   v[ 1 ] = tot[ 1 ];
}

__device__ __forceinline__ bool leadLane()
{
   return blockIdx.x == 0 && threadIdx.x == 0;
}

// A fold in two halves, so that the loads of a launch's first rows go out between them: prefetch()
// issues the loads of the gate and of the first kFoldAhead partials per lane (all there are for up to
// 1024), begin() adds them up.  Nothing waits in prefetch(): the gate is looked at after the sum, since
// a launch that finds it closed has no time to lose.
// The gate's flag is the one state field that workgroup 0 may set while other workgroups of the launch still
// read it.  A launch that sets it may therefore be carried out by some of its workgroups only, and nothing it
// made may be used afterwards: the launches queued behind it find the gate closed, and a restart starts from x.
// The waves of one workgroup may see it differently, so whoever has a barrier ahead asks all of them (openKeeper)
// or reaches it either way (the kernels that call begin() between their loads; a pass with sums is in no launch that
// sets the flag without every workgroup returning).
constexpr int kFoldAhead = 4;

template< int W >
struct Fold
{
   ReduceSlot slot;
   int grid;
   double a[ W ][ kFoldAhead ];
   int32_t done;
   __device__ __forceinline__ void prefetch( Gate gate )
   {
      done = __builtin_nontemporal_load( gate.flags );
#pragma unroll
      for( int k = 0; k < W; k++ )
#pragma unroll
         for( int u = 0; u < kFoldAhead; u++ ) {
            const int j = (int) threadIdx.x + u * kReduceBlock;
            a[ k ][ u ] = j < grid ? slot.partials[ (int64_t) k * grid + j ] : 0.0;
         }
   }
   // false: the gate is closed
   __device__ __forceinline__ bool begin( double ( &v )[ W ] )
   {
      __shared__ double lds[ W ][ kReduceBlock / kWave ];
      const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
#pragma unroll
      for( int k = 0; k < W; k++ ) {
         for( int j = (int) threadIdx.x + kFoldAhead * kReduceBlock; j < grid; j += kFoldAhead * kReduceBlock )
#pragma unroll
            for( int u = 0; u < kFoldAhead; u++ )
               if( j + u * kReduceBlock < grid )
                  a[ k ][ u ] += slot.partials[ (int64_t) k * grid + j + u * kReduceBlock ];
         const double t = groupSum< kWave >( ( a[ k ][ 0 ] + a[ k ][ 1 ] ) + ( a[ k ][ 2 ] + a[ k ][ 3 ] ) );
         if( lane == 0 )
            lds[ k ][ wave ] = t;
      }
      __syncthreads();
#pragma unroll
      for( int k = 0; k < W; k++ )
         v[ k ] = ( lds[ k ][ 0 ] + lds[ k ][ 1 ] ) + ( lds[ k ][ 2 ] + lds[ k ][ 3 ] );
      return done == 0;
   }
};

// ------------------------------------------------------------------ operands

// An operand of a fused product or a fused pass: prefetch() and begin() are called by every thread of
// a workgroup (behind shut(), where it has one), with the launch's first loads between them (begin: false, in every workgroup alike,
// when there is nothing to do); at( x, c ) gives entry c as every row that gathers it sees it;
// row( r, v, acc ) takes the product's (stored) entry of row r.  Entries that are formed on the way are
// formed by explicit fused multiply-adds, so that every gather of an entry and its stored copy have
// the same bits.  The state fields a workgroup needs are loaded in prefetch(), and workgroup 0
// writes only fields that no other workgroup of the same launch uses, but for the stop flag (Fold).

// CG's scalars for the iteration that begins (FinCgBeta) from the (r, z) partials
struct CgNext
{
   State* st;
   double* hist;
   int64_t cap;
   Stop stop;
   Fold< 1 > upd;
   double rhoOld, normb;
   int32_t it, histLen;
   __device__ __forceinline__ void prefetch( Gate gate )
   {
      upd.prefetch( gate );
      rhoOld = st->rho_old;
      normb = st->normb;
      it = st->it;
      histLen = st->histLen;
   }
   __device__ __forceinline__ bool begin( double& beta )
   {
      double v[ 1 ];
      if( ! upd.begin( v ) )
         return false;
      const double rho = v[ 0 ];
      beta = rhoOld == 0.0 ? 0.0 : rho / rhoOld;
      if( leadLane() ) {
         State& s = *st;
         s.s2 = rhoOld;
         s.s1 = rho;
         s.beta = beta;
         recordStep( s, sqrt( rho ) / normb, it, histLen, hist, cap, stop );
      }
      return true;
   }
};

// alpha = rho / (p, Ap) from the partials (FinCgAlpha); the previous rho moves to rho_old for CgNext
struct CgAlpha
{
   State* st;
   double* hist;
   int64_t cap;
   Fold< 1 > dot;
   double rho;
   __device__ __forceinline__ void prefetch( Gate gate )
   {
      dot.prefetch( gate );
      rho = st->s1;
   }
   __device__ __forceinline__ bool begin( double& alpha )
   {
      double v[ 1 ];
      if( ! dot.begin( v ) )
         return false;
      const bool skip = v[ 0 ] == 0.0;
      alpha = skip ? 0.0 : rho / v[ 0 ];
      if( leadLane() ) {
         State& s = *st;
         s.s2 = v[ 0 ];
         s.rho_old = rho;
         if( skip ) {
            // p = 0 => r = 0: the solution has been reached (CG.hpp:64-67)
            setResidue( s, 0.0, hist, cap );
            s.flags[ 0 ] = 1;
         }
         else
            s.alpha = alpha;
      }
      return ! skip;
   }
};

// Scalars of a BiCGStab direction from the {(r, r_ast), (r, r)} partials (FinBiRho): the restart
// test (BICGStab.hpp:88-95), beta, the residue and the stopping rule.  On a restart the state is
// left as it was but for the flags, which stop the queued launches until the host has made the
// new residual.
struct BiNext
{
   State* st;
   double* hist;
   int64_t cap;
   Stop stop;
   double eps2;
   Fold< 2 > upd;
   double rhoOld, omega, alpha, normb, sqnorm;
   int32_t it, histLen, started;
   __device__ __forceinline__ void prefetch( Gate gate )
   {
      upd.prefetch( gate );
      rhoOld = st->rho;
      omega = st->omega;
      alpha = st->alpha;
      normb = st->normb;
      sqnorm = st->r_ast_sqnorm;
      it = st->it;
      histLen = st->histLen;
      started = st->started;
   }
   __device__ __forceinline__ bool begin( double& beta, double& bo )
   {
      double v[ 2 ];
      if( ! upd.begin( v ) )
         return false;
      const double rho = v[ 0 ];
      if( started == 1 && fabs( rho ) < eps2 * sqnorm ) {
         if( leadLane() ) {
            st->flags[ 1 ] = 1;
            st->flags[ 0 ] = 1;
         }
         return false;
      }
      beta = started == 0 ? 0.0 : ( rho / rhoOld ) * ( alpha / omega );
      bo = started == 0 ? 0.0 : beta * omega;
      if( leadLane() ) {
         State& s = *st;
         s.s1 = rho;
         if( started != 1 )  // nobody tests it in this launch
            s.r_ast_sqnorm = rho;
         s.beta = beta;
         recordStep( s, sqrt( v[ 1 ] ) / normb, it, histLen, hist, cap, stop );
      }
      return true;
   }
};

// alpha = rho / (Ap, r_ast) from the partials; workgroup 0 stores it and makes rho the old one
struct BiAlpha
{
   State* st;
   Fold< 1 > dot;
   double rho;
   __device__ __forceinline__ void prefetch( Gate gate )
   {
      dot.prefetch( gate );
      rho = st->s1;
   }
   __device__ __forceinline__ bool begin( double& alpha )
   {
      double v[ 1 ];
      if( ! dot.begin( v ) )
         return false;
      alpha = rho / v[ 0 ];
      if( leadLane() ) {
         st->alpha = alpha;
         st->rho = rho;
         st->started = 1;
      }
      return true;
   }
};

// omega = (As, s) / (As, As) from the partials
struct BiOmega
{
   State* st;
   Fold< 2 > om;
   double alpha;
   __device__ __forceinline__ void prefetch( Gate gate )
   {
      om.prefetch( gate );
      alpha = st->alpha;
   }
   __device__ __forceinline__ bool begin( double& omega )
   {
      double v[ 2 ];
      if( ! om.begin( v ) )
         return false;
      omega = v[ 0 ] / v[ 1 ];
      if( leadLane() )
         st->omega = omega;
      return true;
   }
};

// p = z + beta p_old (z = r without a preconditioner); acc = (Ap, p)
template< typename T >
struct CgDirectionOperand
{
   static constexpr int kSums = 1;
   static constexpr bool kStored = false;
   const T* z;
   const T* pOld;
   T* p;
   CgNext next;
   double beta = 0;
   __device__ __forceinline__ void prefetch( Gate gate ) { next.prefetch( gate ); }
   __device__ __forceinline__ bool begin() { return next.begin( beta ); }
   __device__ __forceinline__ T at( const T*, int64_t c ) const
   {
      return (T) __builtin_fma( beta, (double) pOld[ c ], (double) z[ c ] );
   }
   __device__ __forceinline__ void row( int64_t r, T v, double ( &acc )[ 1 ] ) const
   {
      const T pr = at( nullptr, r );
      p[ r ] = pr;
      acc[ 0 ] = __builtin_fma( (double) v, (double) pr, acc[ 0 ] );
   }
};

// The gate of an operand that folds nothing: no launch of one writes the flag, and there is no sum to hide loads
// behind, so it is looked at first and a closed launch loads nothing (128^3 product: 27 us with its first rows under
// way).
struct OpenGate
{
   __device__ __forceinline__ static bool shut( Gate gate ) { return __builtin_nontemporal_load( gate.flags ) != 0; }
   __device__ __forceinline__ void prefetch( Gate ) {}
   __device__ __forceinline__ bool begin() const { return true; }
};

// a stored operand x; acc = (Ax, w)
template< typename T >
struct DotOperand : OpenGate
{
   static constexpr int kSums = 1;
   static constexpr bool kStored = true;
   const T* w;
   __device__ __forceinline__ T at( const T* x, int64_t c ) const { return x[ c ]; }
   __device__ __forceinline__ void row( int64_t r, T v, double ( &acc )[ 1 ] ) const
   {
      acc[ 0 ] = __builtin_fma( (double) v, (double) w[ r ], acc[ 0 ] );
   }
};

// a stored operand s; acc = { (As, s), (As, As) }
template< typename T >
struct DotSquareOperand : OpenGate
{
   static constexpr int kSums = 2;
   static constexpr bool kStored = true;
   const T* s;
   __device__ __forceinline__ T at( const T* x, int64_t c ) const { return x[ c ]; }
   __device__ __forceinline__ void row( int64_t r, T v, double ( &acc )[ 2 ] ) const
   {
      acc[ 0 ] = __builtin_fma( (double) v, (double) s[ r ], acc[ 0 ] );
      acc[ 1 ] = __builtin_fma( (double) v, (double) v, acc[ 1 ] );
   }
};

// p = r + beta p_old - (beta omega) Ap_old; acc = (Ap, r_ast)
template< typename T >
struct BiDirectionOperand
{
   static constexpr int kSums = 1;
   static constexpr bool kStored = false;
   const T* r;
   const T* pOld;
   const T* ApOld;
   T* p;
   const T* rast;
   BiNext next;
   double beta = 0, bo = 0;
   __device__ __forceinline__ void prefetch( Gate gate ) { next.prefetch( gate ); }
   __device__ __forceinline__ bool begin() { return next.begin( beta, bo ); }
   __device__ __forceinline__ T at( const T*, int64_t c ) const
   {
      const double t = __builtin_fma( beta, (double) pOld[ c ], (double) r[ c ] );
      return (T) __builtin_fma( -bo, (double) ApOld[ c ], t );
   }
   __device__ __forceinline__ void row( int64_t i, T v, double ( &acc )[ 1 ] ) const
   {
      p[ i ] = at( nullptr, i );
      acc[ 0 ] = __builtin_fma( (double) v, (double) rast[ i ], acc[ 0 ] );
   }
};

// s = r - alpha Ap; acc = { (As, s), (As, As) }
template< typename T >
struct BiSOperand
{
   static constexpr int kSums = 2;
   static constexpr bool kStored = false;
   const T* r;
   const T* Ap;
   T* s;
   BiAlpha a;
   double alpha = 0;
   __device__ __forceinline__ void prefetch( Gate gate ) { a.prefetch( gate ); }
   __device__ __forceinline__ bool begin() { return a.begin( alpha ); }
   __device__ __forceinline__ T at( const T*, int64_t c ) const
   {
      return (T) __builtin_fma( -alpha, (double) Ap[ c ], (double) r[ c ] );
   }
   __device__ __forceinline__ void row( int64_t i, T v, double ( &acc )[ 2 ] ) const
   {
      const T si = at( nullptr, i );
      s[ i ] = si;
      acc[ 0 ] = __builtin_fma( (double) v, (double) si, acc[ 0 ] );
      acc[ 1 ] = __builtin_fma( (double) v, (double) v, acc[ 1 ] );
   }
};

// ------------------------------------------------------------------ vector passes

// kVec< T > adjacent entries: 16 bytes, one load or store where all of them exist and the vector is
// 16-byte aligned (`wide`; the solver's own vectors are, the caller's x need not be)
template< typename T >
constexpr int kVec = 16 / (int) sizeof( T );

template< typename T >
struct Lane16
{
   T e[ kVec< T > ];
};

template< typename T >
__device__ __forceinline__ Lane16< T > load16( const T* p, int64_t i, int64_t n, bool wide = true )
{
   typedef T V __attribute__( ( ext_vector_type( 16 / sizeof( T ) ) ) );
   Lane16< T > r;
   if( wide && i + kVec< T > <= n ) {
      const V v = *reinterpret_cast< const V* >( p + i );
#pragma unroll
      for( int u = 0; u < kVec< T >; u++ )
         r.e[ u ] = v[ u ];
   }
   else {
#pragma unroll
      for( int u = 0; u < kVec< T >; u++ )
         r.e[ u ] = i + u < n ? p[ i + u ] : T( 0 );
   }
   return r;
}

template< typename T >
__device__ __forceinline__ void store16( T* p, int64_t i, int64_t n, const Lane16< T >& r, bool wide = true )
{
   typedef T V __attribute__( ( ext_vector_type( 16 / sizeof( T ) ) ) );
   if( wide && i + kVec< T > <= n ) {
      V v;
#pragma unroll
      for( int u = 0; u < kVec< T >; u++ )
         v[ u ] = r.e[ u ];
      *reinterpret_cast< V* >( p + i ) = v;
   }
   else {
#pragma unroll
      for( int u = 0; u < kVec< T >; u++ )
         if( i + u < n )
            p[ i + u ] = r.e[ u ];
   }
}

inline bool aligned16( const void* p ) { return reinterpret_cast< uintptr_t >( p ) % 16 == 0; }

// Workgroups of a pass over n entries of T, kVec< T > per lane and step
template< typename T >
int passGrid( int64_t n )
{
   const int64_t per = (int64_t) kReduceBlock * kVec< T >;
   return (int) std::min< int64_t >( kReduceGrid, ( n + per - 1 ) / per );
}

// A pass over n entries with W sums: 16-byte lanes, the entries of the next step loaded before
// those of this one are worked on, and those of the first step before the scalars are there.
// Op: prefetch, begin as an operand's; In load( i, n ); apply( i, n, in, acc ).
template< int W, typename T, typename Op >
__global__ __launch_bounds__( kReduceBlock ) void passKernel( int64_t n, Op op, ReduceSlot out, Gate gate )
{
   op.prefetch( gate );
   const int64_t stride = (int64_t) gridDim.x * kReduceBlock * kVec< T >;
   int64_t i = ( (int64_t) blockIdx.x * kReduceBlock + threadIdx.x ) * kVec< T >;
   typename Op::In in = op.load( i, n );
   if( ! op.begin() )
      return;
   double acc[ W > 0 ? W : 1 ] = {};
   while( i < n ) {
      const typename Op::In next = op.load( i + stride, n );
      op.apply( i, n, in, acc );
      in = next;
      i += stride;
   }
   if constexpr( W > 0 )
      storeBlockPartials< W >( acc, out );
}

template< int W, typename T, typename Op >
void launchPass( int64_t n, const Op& op, ReduceSlot out, Gate gate, hipStream_t st )
{
   passKernel< W, T ><<< passGrid< T >( n ), kReduceBlock, 0, st >>>( n, op, out, gate );
   TNLHIP_CHECK( hipGetLastError() );
}

// x += alpha p; r -= alpha Ap; z = r / diag; acc = (r, z or r)
template< typename T >
struct CgUpdatePass
{
   T* x;
   T* r;
   T* z;
   const T* p;
   const T* Ap;
   const T* diag;
   bool wideX;
   CgAlpha a;
   double alpha = 0;
   struct In
   {
      Lane16< T > x, r, p, Ap, d;
   };
   __device__ __forceinline__ void prefetch( Gate gate ) { a.prefetch( gate ); }
   __device__ __forceinline__ bool begin() { return a.begin( alpha ); }
   __device__ __forceinline__ In load( int64_t i, int64_t n ) const
   {
      In v;
      v.Ap = load16( Ap, i, n );
      v.r = load16( r, i, n );
      if( diag )
         v.d = load16( diag, i, n );
      v.p = load16( p, i, n );
      v.x = load16( x, i, n, wideX );
      return v;
   }
   __device__ __forceinline__ void apply( int64_t i, int64_t n, const In& v, double ( &acc )[ 1 ] ) const
   {
      Lane16< T > xn, rn, zn;
#pragma unroll
      for( int u = 0; u < kVec< T >; u++ ) {
         xn.e[ u ] = (T) ( (double) v.x.e[ u ] + alpha * (double) v.p.e[ u ] );
         rn.e[ u ] = (T) ( (double) v.r.e[ u ] - alpha * (double) v.Ap.e[ u ] );
         zn.e[ u ] = diag ? rn.e[ u ] / v.d.e[ u ] : rn.e[ u ];
         if( i + u < n )
            acc[ 0 ] += (double) rn.e[ u ] * (double) zn.e[ u ];
      }
      store16( r, i, n, rn );
      if( diag )
         store16( z, i, n, zn );
      store16( x, i, n, xn, wideX );
   }
};

// p = z + beta p in place
template< typename T >
struct CgDirectionPass
{
   T* p;
   const T* z;
   CgNext next;
   double beta = 0;
   struct In
   {
      Lane16< T > z, p;
   };
   __device__ __forceinline__ void prefetch( Gate gate ) { next.prefetch( gate ); }
   __device__ __forceinline__ bool begin() { return next.begin( beta ); }
   __device__ __forceinline__ In load( int64_t i, int64_t n ) const { return In{ load16( z, i, n ), load16( p, i, n ) }; }
   __device__ __forceinline__ void apply( int64_t i, int64_t n, const In& v, double ( & )[ 1 ] ) const
   {
      Lane16< T > o;
#pragma unroll
      for( int u = 0; u < kVec< T >; u++ )
         o.e[ u ] = (T) __builtin_fma( beta, (double) v.p.e[ u ], (double) v.z.e[ u ] );
      store16( p, i, n, o );
   }
};

// x += alpha p + omega s; r = s - omega As; acc = { (r, r_ast), (r, r) }
template< typename T >
struct BiUpdatePass
{
   T* x;
   T* r;
   const T* p;
   const T* s;
   const T* As;
   const T* rast;
   bool wideX;
   BiOmega o;
   double omega = 0;
   struct In
   {
      Lane16< T > x, p, s, As, rast;
   };
   __device__ __forceinline__ void prefetch( Gate gate ) { o.prefetch( gate ); }
   __device__ __forceinline__ bool begin() { return o.begin( omega ); }
   __device__ __forceinline__ In load( int64_t i, int64_t n ) const
   {
      return In{ load16( x, i, n, wideX ), load16( p, i, n ), load16( s, i, n ), load16( As, i, n ),
                 load16( rast, i, n ) };
   }
   __device__ __forceinline__ void apply( int64_t i, int64_t n, const In& v, double ( &acc )[ 2 ] ) const
   {
      Lane16< T > xn, rn;
#pragma unroll
      for( int u = 0; u < kVec< T >; u++ ) {
         const double si = (double) v.s.e[ u ];
         xn.e[ u ] = (T) ( (double) v.x.e[ u ] + ( o.alpha * (double) v.p.e[ u ] + omega * si ) );
         rn.e[ u ] = (T) ( si - omega * (double) v.As.e[ u ] );
         if( i + u < n ) {
            acc[ 0 ] += (double) rn.e[ u ] * (double) v.rast.e[ u ];
            acc[ 1 ] += (double) rn.e[ u ] * (double) rn.e[ u ];
         }
      }
      store16( r, i, n, rn );
      store16( x, i, n, xn, wideX );
   }
};

// p = r + beta p - (beta omega) Ap in place
template< typename T >
struct BiDirectionPass
{
   T* p;
   const T* r;
   const T* Ap;
   BiNext next;
   double beta = 0, bo = 0;
   struct In
   {
      Lane16< T > p, r, Ap;
   };
   __device__ __forceinline__ void prefetch( Gate gate ) { next.prefetch( gate ); }
   __device__ __forceinline__ bool begin() { return next.begin( beta, bo ); }
   __device__ __forceinline__ In load( int64_t i, int64_t n ) const
   {
      return In{ load16( p, i, n ), load16( r, i, n ), load16( Ap, i, n ) };
   }
   __device__ __forceinline__ void apply( int64_t i, int64_t n, const In& v, double ( & )[ 1 ] ) const
   {
      Lane16< T > o;
#pragma unroll
      for( int u = 0; u < kVec< T >; u++ )
         o.e[ u ] = (T) __builtin_fma( -bo, (double) v.Ap.e[ u ],
                                       __builtin_fma( beta, (double) v.p.e[ u ], (double) v.r.e[ u ] ) );
      store16( p, i, n, o );
   }
};

// s = r - alpha Ap
template< typename T >
struct BiSPass
{
   T* s;
   const T* r;
   const T* Ap;
   BiAlpha a;
   double alpha = 0;
   struct In
   {
      Lane16< T > r, Ap;
   };
   __device__ __forceinline__ void prefetch( Gate gate ) { a.prefetch( gate ); }
   __device__ __forceinline__ bool begin() { return a.begin( alpha ); }
   __device__ __forceinline__ In load( int64_t i, int64_t n ) const { return In{ load16( r, i, n ), load16( Ap, i, n ) }; }
   __device__ __forceinline__ void apply( int64_t i, int64_t n, const In& v, double ( & )[ 1 ] ) const
   {
      Lane16< T > o;
#pragma unroll
      for( int u = 0; u < kVec< T >; u++ )
         o.e[ u ] = (T) __builtin_fma( -alpha, (double) v.Ap.e[ u ], (double) v.r.e[ u ] );
      store16( s, i, n, o );
   }
};

// ------------------------------------------------------------------ fused products

// Partials per sum a fused product may write (a reduction slot holds twice as many of each of two sums).  Every
// workgroup of the launch that follows folds them all, and beyond this the dot's own pass is cheaper: us per Jacobi
// CG iteration, separate passes / fused, 140^3 and 160^3 (10719 and 16000 workgroups) CSRScalar FP64 112.8 / 124.7 and
// 158.4 / 178.9, ChunkedEllpack FP64 109.6 / 108.5 and 151.6 / 151.6, FP32 76.3 / 81.6 and 100.2 / 111.0.
constexpr int kMaxFusedPartials = 8192;

// The grid, hence the number of partials per sum, of the fused products with A; 0 when A takes the
// separate passes (symmetric, binary and BF16 matrices, striped plans, nothing stored, more than
// kMaxFusedPartials workgroups, many rows of 32 or 64 lanes).  twoProducts: an iteration has two of them (BiCGStab).
int fusedGrid( const Matrix& A, bool twoProducts );

// Whether forming the operand where it is gathered pays for A.
bool fuseOperand( const Matrix& A );

// y = A op (/ diag), the operand's sums to `out`, gated.  x is the operand of the stored kinds.
template< typename T, typename Op >
void fusedProduct( const Matrix& A, const Op& op, const T* x, const T* diag, T* y, ReduceSlot out, Gate gate,
                   hipStream_t stream );

}  // namespace tnlhip

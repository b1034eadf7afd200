// ILU(0) preconditioner on the device: factors L (unit diagonal implied) and U with the
// sparsity of A, factorized and applied level by level.
#pragma once

#include "matrix.hpp"

namespace tnlhip {

struct Ilu0
{
   // one launch of a sweep: a single level spread over the device, or a run of consecutive small
   // levels taken step by step by one workgroup
   struct Launch
   {
      int32_t firstLevel, lastLevel;  // [first, last)
      int32_t firstStep, steps;
      int32_t firstSlice, slices;
      int32_t block;  // lanes of a run's workgroup
      bool wide;
   };
   // a triangular factor in level order
   struct Sweep
   {
      DeviceArray< int32_t > order;     // row at each position
      DeviceArray< int32_t > position;  // position of each row
      std::vector< int32_t > levels;    // level boundaries in positions (host copy)
      DeviceArray< int32_t > levelsDevice;
      std::vector< Launch > launches;
      DeviceArray< int32_t > len, steps, slices, sliceRest, slots, restCol;
      DeviceArray< uint8_t > val, diag, restVal;
      int32_t positions = 0, nslices = 0;
      int32_t rest = 0;               // entries in the rest arrays
      bool longRows = false;          // which W and D the sweep takes
   };

   int32_t n = 0;
   int dtype = TNLHIP_F64;  // value type of the factors and vectors (TNLHIP_F64 or TNLHIP_F32)
   DeviceArray< int32_t > Lrp, Lc, Urp, Uc;  // the factors in row order, until the sweeps are packed
   DeviceArray< uint8_t > Lv, Uv;
   Sweep lower, upper;
   DeviceArray< int32_t > between;  // lower position of the row at each upper position
   DeviceArray< uint8_t > work;     // two vectors in level order

   // symbolic split and level schedules on the host, numeric factorization on the device
   void build( const Matrix& A, int vectorDtype, hipStream_t stream );
   // x = U^-1 L^-1 b (b == x allowed), skipped on the device while the gate is closed
   void solve( const void* b, void* x, Gate gate, hipStream_t stream ) const;
   int32_t levelCount( bool upperSolve ) const
   {
      return (int32_t) ( upperSolve ? upper.levels.size() : lower.levels.size() ) - 1;
   }
};

}  // namespace tnlhip

// The kernels of small layers for one dtype.  Compiled three times (-DCATS_DT=F16 / BF16 / F32), beside cats_inst.hip.
#include <type_traits>

#include "cats_launch.h"

#ifndef CATS_DT
#error "compile with -DCATS_DT=F16|BF16|F32"
#endif

namespace cats {

namespace {

typedef void (*SmallKernel)(SmallArgs);

template <int B, bool ONE, bool TAIL>
SmallKernel rows_for_tail(int nch) {
  switch (nch) {
    case 1: return small_rows_kernel<CATS_DT, B, 1, ONE, TAIL>;
    case 2: return small_rows_kernel<CATS_DT, B, 2, ONE, TAIL>;
    case 3: return small_rows_kernel<CATS_DT, B, 3, ONE, TAIL>;
    case 4: return small_rows_kernel<CATS_DT, B, 4, ONE, TAIL>;
  }
  return nullptr;
}
template <int B, bool ONE>
SmallKernel rows_for(const RowsArgs& r) {
  return r.norm_w ? rows_for_tail<B, ONE, true>(r.nch) : rows_for_tail<B, ONE, false>(r.nch);
}

template <int NG>
SmallKernel mma_for(int steps) {
  switch (steps) {
    case 1: return small_mma_kernel<CATS_DT, 1, NG>;
    case 2: return small_mma_kernel<CATS_DT, 2, NG>;
    case 3: return small_mma_kernel<CATS_DT, 3, NG>;
    case 4: return small_mma_kernel<CATS_DT, 4, NG>;
    case 5: return small_mma_kernel<CATS_DT, 5, NG>;
  }
  return nullptr;
}

}  // namespace

template <>
hipError_t launch_small<CATS_DT>(bool mma, int grid, const SmallArgs& a, hipStream_t stream) {
  SmallKernel kern = nullptr;
  size_t lds = 0;
  if ((a.r.norm_w != nullptr) != (a.fin.residual != nullptr)) return hipErrorInvalidValue;  // TAIL stands for both
  if (mma) {
    const int steps = rows_mma_split(a.r).steps;
    kern = a.r.nb > 8 ? mma_for<2>(steps) : mma_for<1>(steps);
    lds = small_mma_lds_bytes(a.r.mma_slots, a.r.nb > 8 ? 2 : 1);
    if (hipError_t e = ensure_dynamic_lds((const void*)kern, lds); e != hipSuccess) return e;
  } else if (a.r.nb == 1) {
    kern = a.arrive ? rows_for<1, true>(a.r) : rows_for<1, false>(a.r);
  } else if (a.r.nb == 2) {
    kern = rows_for<2, false>(a.r);
  } else if constexpr (std::is_same<CATS_DT, F32>::value) {
    kern = rows_for<4, false>(a.r);
  }
  if (!kern) return hipErrorInvalidValue;
  return launch_kernel(kern, dim3(grid), dim3(kSmallThreads), lds, stream, a);
}

template <>
hipError_t launch_small_tail<CATS_DT>(int rows, const ReduceArgs& r, hipStream_t stream) {
  return launch_kernel(r.residual ? small_tail_kernel<CATS_DT, true> : small_tail_kernel<CATS_DT, false>, dim3(rows), dim3(kSmallThreads), 0, stream, r);
}

}  // namespace cats

// Gate pass of one batch row over a gate weight that is stored (H, I) -- one row per input element, x . W instead of W . x:
// partial[g][j] = sum over the rows k of group g of x[k] * w[k][j].  Bound by the weight stream (90 MB at 4096 x 11008 in 16 bits).
//
// A workgroup of sixteen waves owns one 16-byte vector per lane of columns and an equal range of the rows; its waves take the rows
// of the range in turn, 2 * U rows in flight each, and meet in LDS once at the end.  The rows are split into as many groups as make
// one workgroup per CU over all column slabs (at most kGateColsMaxGroups), and whoever reads the activations adds the
// groups' sums (gate_cols_activation): the single-pass kernel does that while it stages x, so no launch is spent on it.
// A row may start anywhere (an odd I): the vectors are read as they lie, which the memory system takes at any alignment of the
// element, and the lanes of the last slab are moved back to end with the row instead of being masked.
// Whole call at 4096 / 11008, fp16, half the neurons kept: 40.0 us (4.5 TB/s); with torch's product, SiLU, comparison and
// nonzero, which waits for the list's length, and the two list kernels behind them it was 121 us.
#pragma once
#include "cats_device.h"

namespace cats {

constexpr int kGateColsMaxGroups = 16;  // their sums fit the gate-activation scratch of the workspace, 16 * I floats
constexpr int kGateColsWaves = 16;

typedef u32x4 u32x4_any __attribute__((aligned(2)));  // a vector at any element

struct GateColsArgs {
  const void* x;     // (H,) dtype
  const void* w;     // (H, I) dtype, any alignment of the element
  float* partial;    // [groups][I]
  int H, I;
  int rows_per;      // rows of a group
  int nslab;         // column slabs of 64 vectors
};

template <class DT>
__global__ __launch_bounds__(kGateColsWaves* kWave) void gate_cols_kernel(GateColsArgs p) {
  typedef typename DT::st st;
  constexpr int VEC = DT::VEC, U = 8, SLAB = kWave * VEC;
  __shared__ float s_part[kGateColsWaves][SLAB];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slab = blockIdx.x % p.nslab, group = blockIdx.x / p.nslab;
  const int first = slab * SLAB;                         // first column that this workgroup owns
  const int col = min(first + lane * VEC, p.I - VEC);    // I >= VEC
  const int k0 = group * p.rows_per, k1 = min(k0 + p.rows_per, p.H);
  const st* w = (const st*)p.w + col;
  const int n = k1 > k0 + wave ? (k1 - k0 - wave + kGateColsWaves - 1) / kGateColsWaves : 0;  // rows of this wave
  const int kw = k0 + wave;

  // a row past `end` reads one cached vector, the same address in every lane, so that every batch is U loads
  auto issue = [&](int i0, int end, u32x4 (&v)[U]) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const bool in = i0 + u < end;  // uniform
      const st* r = in ? w + (size_t)(kw + (i0 + u) * kGateColsWaves) * p.I : (const st*)p.w;
      v[u] = __builtin_nontemporal_load((const u32x4_any*)r);
    }
  };
  float acc[VEC];
#pragma unroll
  for (int e = 0; e < VEC; e++) acc[e] = 0.f;
  float xl = 0.f;  // lane i: x of the wave's row (64 * block + i)
  auto take = [&](int i0, const u32x4 (&v)[U]) {
#pragma unroll
    for (int u = 0; u < U; u++)
      if (i0 + u < n)  // uniform
        DT::axpy(v[u], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(xl), (i0 + u) & (kWave - 1))), acc);
  };
  u32x4 va[U], vb[U];
  for (int b0 = 0; b0 < n; b0 += kWave) {
    xl = DT::tof(((const st*)p.x)[min(kw + (b0 + lane) * kGateColsWaves, p.H - 1)]);
    const int end = min(n, b0 + kWave);
    issue(b0, end, va);
    for (int i = b0; i < end; i += 2 * U) {
      issue(i + U, end, vb);
      take(i, va);
      issue(i + 2 * U, end, va);
      take(i + U, vb);
    }
  }
#pragma unroll
  for (int e = 0; e < VEC; e++) s_part[wave][e * kWave + lane] = acc[e];
  __syncthreads();
  // column first + c is element e of lane l; a lane that was moved back holds it shifted
  for (int c = threadIdx.x; c < SLAB && first + c < p.I; c += kGateColsWaves * kWave) {
    const int l = c / VEC, at = first + c - min(first + l * VEC, p.I - VEC);
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < kGateColsWaves; v++) s += s_part[v][at * kWave + l];
    p.partial[(size_t)group * p.I + first + c] = s;
  }
}

// The activation of neuron j from the groups' sums, rounded where the gate kernels round.
template <class DT>
__device__ __forceinline__ float gate_cols_activation(const float* __restrict__ part, int groups, int I, int j) {
  float v[kGateColsMaxGroups];
#pragma unroll
  for (int g = 0; g < kGateColsMaxGroups; g++) v[g] = part[(size_t)min(g, groups - 1) * I + j];
  float s = 0.f;
#pragma unroll
  for (int g = 0; g < kGateColsMaxGroups; g++) s += g < groups ? v[g] : 0.f;
  const float gr = DT::rnd(s);
  return DT::rnd(gr / (1.f + expf(-gr)));
}

// The same as a launch of its own, for the kernels that take activations.
template <class DT>
__global__ __launch_bounds__(256) void gate_cols_finish_kernel(const float* part, int groups, int I, void* a) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j < I) ((typename DT::st*)a)[j] = DT::fromf(gate_cols_activation<DT>(part, groups, I, j));
}

}  // namespace cats

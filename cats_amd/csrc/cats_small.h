// Whole CATS MLP of a small layer: one launch that leaves partial sums, and one that adds them.
//
// In a layer of a few megabytes the bytes are not what a call waits for: the streaming kernels pay a chain of memory trips (x, gate row, up row,
// down row; a list and z between two launches from three rows on), each about as long as reading the whole layer.  Here a workgroup of sixteen
// waves owns sixteen neurons and asks for everything it may need -- x, its gate rows, its up rows, its down rows -- before it waits for anything;
// rows of neurons that turn out dead are read for nothing and replaced by zeros before they are used.  All weights stay in registers.
//
//   small_rows_kernel   up to 2 batch rows (4 in fp32): a wave per neuron on the vector ALUs, the sums in rows_kernel's order
//   small_mma_kernel    the batches that rows_mma_kernel takes: its tiles, operands and sums, eight waves for gate and eight for up
//
// so a gate call, and a call of the same layer with more rows, agree with these on every activation.
//
// What bounds them: two dependent launches are 5 us of GPU time whatever they do, and 512 / 1024 at one row in fp16 takes 5.6 (streaming kernel and
// reduction: 9.6; three launches at 4 rows: 12.5, here 7.3).  From some 5 MB a matrix on it is the stream and the write-back of the partial
// sums: 2048 / 3072 at 4 rows has all 38 MB 7.7 us after its start, is done 2.5 us later, and writes 6.3 MB until 14 us.
// Thirty-two neurons a workgroup (half the sums, half the CUs): 1 to 3 us slower nearly everywhere; eight or eleven: no faster.
#pragma once
#include "cats_down_mma.h"
#include "cats_fused.h"
#include "cats_rows_mma.h"

namespace cats {

constexpr int kSmallWaves = 16;
constexpr int kSmallThreads = kSmallWaves * kWave;
constexpr int kSmallRows = 16;      // neurons a workgroup owns
constexpr int kSmallMaxVecs = 256;  // 16-byte vectors of a row: a down wave covers sixteen of them

struct SmallArgs {
  RowsArgs r;        // x, w (gate), w2 (up), K, N, nb, row_vecs, flag_out, t, norm_w, norm_eps; rows_per .. mma_slots as for rows_mma_kernel
  const u32x4* wd;   // (N, K) neuron-major
  float* partial;    // [grid][nb][K]
  int32_t* counts;   // [grid] neurons that some batch row keeps
  // one batch row in one launch: the workgroup that arrives last finishes the call, fin being what the reduction launch would take
  int32_t* arrive;   // zero between calls; NULL: the sums and counts are left
  ReduceArgs fin;
};

// ---- the partial sums of small layers -------------------------------------------------------------------------------------------

// Threads side by side over a row of H columns, four each; the 1024 / quads groups of threads take a range of the partials each.
__device__ inline int small_quads(int H) {
  int q = kWave;
  while (q < H / 4) q *= 2;
  return q;
}

// Batch row `row` of what reduce_partials_kernel does, by one workgroup, the next norm included: no hand-over between workgroups in front of it.
// Ranges of partials side by side, their sums in range order, then the count.  s_part: a float4 of LDS a thread.
// TAIL: the layer tail, with a residual and perhaps the next norm.
template <class DT, bool TAIL>
__device__ __forceinline__ void small_finish_row(const ReduceArgs& p, int row, float4* s_part, float* s_ssq) {
  typedef typename DT::st st;
  const int quads = small_quads(p.H);
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
  const int quad = tid & (quads - 1), range = tid / quads, ranges = kSmallThreads / quads;
  const bool on = quad * 4 < p.H;
  const int per = (p.G + ranges - 1) / ranges, g0 = range * per, g1 = min(p.G, g0 + per);
  const size_t col = (size_t)row * p.H + (on ? quad * 4 : 0);
  const bool mine = range == 0 && on;
  // What the sums are joined with comes in with the partials: steps of one layer 256 / 640, 4 rows 42.9 us without, 42.3 with; 512 / 1121, 1 row 32.8, 32.6.
  // In an instance of its own: with these loads behind conditions a plain call of 512 / 1024 took 8.18 us, without any 8.04.
  float residual[4] = {0.f, 0.f, 0.f, 0.f}, norm2[4] = {0.f, 0.f, 0.f, 0.f};
  if (TAIL && mine) {
#pragma unroll
    for (int e = 0; e < 4; e++) residual[e] = DT::tof(((const st*)p.residual)[col + e]);
  }
  if (TAIL && mine && p.norm2_out) {
#pragma unroll
    for (int e = 0; e < 4; e++) norm2[e] = DT::tof(((const st*)p.norm2_w)[quad * 4 + e]);
  }
  float4 s = {0.f, 0.f, 0.f, 0.f};
  constexpr int U = 8;  // sixteen: 0.9 us slower at 64 partials of 512
  for (int g = g0; g < g1; g += U) {
    float4 t[U];
#pragma unroll
    for (int u = 0; u < U; u++) t[u] = *(const float4*)(p.partial + (size_t)min(g + u, g1 - 1) * p.BH + col);
#pragma unroll
    for (int u = 0; u < U; u++)
      if (g + u < g1) { s.x += t[u].x; s.y += t[u].y; s.z += t[u].z; s.w += t[u].w; }
  }
  s_part[tid] = s;
  __syncthreads();
  float y[4] = {0.f, 0.f, 0.f, 0.f}, ss = 0.f;
  if (mine) {
    for (int r = 0; r < ranges; r++) {
      const float4 t = s_part[r * quads + quad];
      y[0] += t.x; y[1] += t.y; y[2] += t.z; y[3] += t.w;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      if (!TAIL && p.y32_acc) {
        unsafeAtomicAdd(p.y32_acc + col + e, y[e]);  // as in reduce_partials_kernel
      } else {
        const st o = DT::fromf(TAIL ? DT::rnd(y[e]) + residual[e] : y[e]);
        ((st*)p.y_out)[col + e] = o;
        y[e] = DT::tof(o);
        ss = fmaf(y[e], y[e], ss);
      }
    }
  }
  if (TAIL && p.norm2_out) {
    ss = wave_sum(ss);
    if (lane == 0) s_ssq[wave] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int w = 0; w < kSmallWaves; w++) tot += s_ssq[w];
    const float scale = rsqrtf(tot / (float)p.H + p.norm2_eps);
    if (mine) {
#pragma unroll
      for (int e = 0; e < 4; e++)
        ((st*)p.norm2_out)[col + e] = DT::fromf(norm2[e] * DT::rnd(y[e] * scale));
    }
  }
  if (p.count_out && row == 0 && wave == 0) {
    int k = 0;
    for (int g = lane; g < p.G; g += kWave) k += p.counts[g];
    k = (int)wave_sum((float)k);  // far below 2^24: exact in fp32
    if (lane == 0) *p.count_out = k;
  }
}

// As a launch: a workgroup per batch row.
template <class DT, bool TAIL>
__global__ __launch_bounds__(kSmallThreads) void small_tail_kernel(ReduceArgs p) {
  __shared__ float4 s_part[kSmallThreads];
  __shared__ float s_ssq[kSmallWaves];
  small_finish_row<DT, TAIL>(p, blockIdx.x, s_part, s_ssq);
}

// Two neighbouring partial sums.  THROUGH: another workgroup of the same launch reads them, so they are written to the level that all XCDs share.
template <bool THROUGH>
__device__ __forceinline__ void small_store2(float* to, float a, float b) {
  const uint64_t v = __float_as_uint(a) | (uint64_t)__float_as_uint(b) << 32;
  if (THROUGH) __hip_atomic_store((uint64_t*)to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *(uint64_t*)to = v;
}

// The end of a call of one row in one launch, for all threads of the workgroup.  Nobody waits: a workgroup whose sums have been acknowledged counts
// itself, and the one that finds itself the last adds up everything.  The counter is zero again before the launch ends.
template <class DT, bool TAIL>
__device__ __forceinline__ void small_arrive(const SmallArgs& a) {
  __shared__ float4 s_part[kSmallThreads];
  __shared__ float s_ssq[kSmallWaves];
  __shared__ int s_last;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    s_last = __hip_atomic_fetch_add(a.arrive, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
    if (s_last) __hip_atomic_store(a.arrive, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!s_last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  small_finish_row<DT, TAIL>(a.fin, 0, s_part, s_ssq);
}

// The sum of lo over this lane and the one W lanes away in the lower of the two, of hi in the upper.
template <int W>
__device__ __forceinline__ float small_fold(float lo, float hi) {
  const auto v = W == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(lo), __float_as_uint(hi), false, false)
                         : __builtin_amdgcn_permlane16_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
  return __uint_as_float(v[0]) + __uint_as_float(v[1]);
}

// NCH: 64-lane chunks of a row; a wave takes one neuron.
// Down: a wave owns 1/16 of the columns, CL lanes of one vector each; its 64 / CL lane groups take the neurons in turn and meet in
// registers, so nothing but z goes through LDS.  (The sums of all lane groups by __shfl_xor, 32 to 64 of them, cost 0.9 us a batch row.)
// TAIL: the layer tail, which brings a norm and a residual.
template <class DT, int B, int NCH, bool ONE, bool TAIL>
__global__ __launch_bounds__(kSmallThreads) void small_rows_kernel(SmallArgs a) {
  typedef typename DT::st st;
  constexpr int VEC = DT::VEC, CL = NCH == 1 ? 4 : NCH == 2 ? 8 : 16, GR = kWave / CL, DL = kSmallRows / GR;
  static_assert(NCH <= 4 && B * NCH <= kSmallWaves && kSmallRows == kSmallWaves, "one vector of x a thread, one neuron a wave");
  const RowsArgs& p = a.r;
  __shared__ u32x4 xs[B * NCH * kWave];
  __shared__ float s_z[kSmallRows * B];
  __shared__ int s_any[kSmallRows];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = blockIdx.x * p.rows_per, n = min(p.rows_per, p.N - row0);  // at least one neuron
  const int vlast = p.row_vecs - 1;

  const int xb = wave / NCH, xi = tid - xb * NCH * kWave;  // this thread's vector of x
  const bool x_in = xb < B && xb < p.nb && xi < p.row_vecs;
  u32x4 xv = p.x[x_in ? (size_t)xb * p.row_vecs + xi : 0];
  u32x4 nw = zero4();
  if (TAIL) nw = p.norm_w[x_in ? xi : 0];
  __builtin_amdgcn_sched_barrier(0);
  u32x4 wg[NCH], wu[NCH], wd[DL];
  const size_t own = (size_t)(row0 + min(wave, n - 1)) * p.row_vecs;
#pragma unroll
  for (int c = 0; c < NCH; c++) wg[c] = load_stream(p.w + own + min(c * kWave + lane, vlast));
#pragma unroll
  for (int c = 0; c < NCH; c++) wu[c] = load_stream(p.w2 + own + min(c * kWave + lane, vlast));
  const int cl = lane % CL, gr = lane / CL, v = wave * CL + cl;
#pragma unroll
  for (int d = 0; d < DL; d++) wd[d] = load_stream(a.wd + (size_t)(row0 + min(gr + d * GR, n - 1)) * p.row_vecs + min(v, vlast));
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < 4; e++) xv[e] = x_in ? xv[e] : 0u;
  if (TAIL) {  // NCH waves hold a row
    __shared__ float s_sq[B * NCH];
    const float sq = wave_sum(vec_sumsq<DT>(xv, 0.f));
    if (lane == 0 && xb < B) s_sq[wave] = sq;
    lds_barrier();
    if (x_in) {
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < NCH; c++) ss += s_sq[xb * NCH + c];
      xv = vec_norm_apply<DT>(xv, rsqrtf(ss / (float)p.K + p.norm_eps), nw);
    }
  }
  if (tid < B * NCH * kWave) xs[tid] = xv;
  lds_barrier();

  {
    float z[B];
    bool act[B], any = false;
#pragma unroll
    for (int b = 0; b < B; b++) {
      float g = 0.f, u = 0.f;
#pragma unroll
      for (int c = 0; c < NCH; c++) {
        const u32x4 x = xs[(b * NCH + c) * kWave + lane];
        g = DT::dot(wg[c], x, g);
        u = DT::dot(wu[c], x, u);
      }
      const float gs = DT::rnd(wave_sum(g)), av = DT::rnd(gs / (1.f + expf(-gs)));
      act[b] = wave < n && b < p.nb && fabsf(av) > p.t;
      z[b] = act[b] ? DT::rnd(av * DT::rnd(wave_sum(u))) : 0.f;
      any = any || act[b];
    }
    if (lane == 0) {
#pragma unroll
      for (int b = 0; b < B; b++) {
        s_z[wave * B + b] = z[b];
        if (p.flag_out && wave < n && b < p.nb) p.flag_out[(size_t)b * p.N + row0 + wave] = act[b] ? 1 : 0;
      }
      s_any[wave] = any ? 1 : 0;
    }
  }
  lds_barrier();
  if (wave == 0) {
    const uint64_t live = __ballot(lane < kSmallRows && s_any[lane & (kSmallRows - 1)] != 0);
    if (lane == 0) __hip_atomic_store(&a.counts[blockIdx.x], (int)__popcll(live), __ATOMIC_RELAXED, ONE ? __HIP_MEMORY_SCOPE_AGENT : __HIP_MEMORY_SCOPE_WORKGROUP);
  }

  float acc[B][VEC];
#pragma unroll
  for (int b = 0; b < B; b++)
#pragma unroll
    for (int e = 0; e < VEC; e++) acc[b][e] = 0.f;
#pragma unroll
  for (int d = 0; d < DL; d++) {
    const int q = gr + d * GR;
    const u32x4 w = s_any[q] ? wd[d] : zero4();  // a dead neuron's weights may be anything
#pragma unroll
    for (int b = 0; b < B; b++) DT::axpy(w, s_z[q * B + b], acc[b]);
  }
  // Lane groups meet: across the halves and the quarters of the wave each lane keeps half of the elements, inside a quarter (16 lanes) all
  // of them.  Lane (half h, quarter r of it) ends with elements K2 * (2 * h + r) ...
  constexpr int K2 = VEC / 4;
  float* out = a.partial + (size_t)blockIdx.x * p.nb * p.K + (size_t)v * VEC + K2 * (lane >> 4);
#pragma unroll
  for (int b = 0; b < B; b++) {
    float half[VEC / 2], s[K2];
#pragma unroll
    for (int e = 0; e < VEC / 2; e++) half[e] = small_fold<32>(acc[b][e], acc[b][e + VEC / 2]);
#pragma unroll
    for (int e = 0; e < K2; e++) {
      s[e] = small_fold<16>(half[e], half[e + K2]);
      if (CL <= 8) s[e] = dpp_add<0x128>(s[e]);  // row_ror:8
      if (CL <= 4) s[e] = dpp_add<0x124>(s[e]);  // row_ror:4
    }
    if ((lane & 15) < CL && b < p.nb && v <= vlast) {
      float* o = out + (size_t)b * p.K;
      if constexpr (K2 == 2) small_store2<ONE>(o, s[0], s[1]);
      else if (ONE) __hip_atomic_store(o, s[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else *o = s[0];
    }
  }
  if constexpr (ONE) small_arrive<DT, TAIL>(a);
}

// ---- batches on the matrix cores ----------------------------------------------------------------------------------------------
// Two tiles of eight neurons a workgroup, eight waves over K for the gate rows and eight for the up rows, both tiles' loads in flight at once.  STEPS, NG as for rows_mma_kernel.  Down: wave w owns sixteen vectors of the columns, sixteen neurons a step, the operands as
// in down_mma_kernel (16-bit types); in fp32 one v_mfma_f32_16x16x4 per element of the vectors takes four neurons.
// dynamic LDS: x operands | [two tiles][gate, up] partial sums | z
inline size_t small_mma_lds_bytes(int slots, int ng) {
  return (size_t)ng * slots * kWave * sizeof(u32x4) + (size_t)4 * ng * kMmaPartGroup * sizeof(float) + (size_t)kSmallRows * 16 * sizeof(float);
}

template <class DT, int STEPS, int NG>
__global__ __launch_bounds__(kSmallThreads) void small_mma_kernel(SmallArgs a) {
  typedef typename DT::st st;
  typedef MmaRows<DT, STEPS, 1, NG> Rows;
  constexpr bool HALF = sizeof(st) == 2;
  constexpr int VEC = DT::VEC, T = kSmallRows / kMmaTileRows, NV = ((STEPS * kMmaWaves + 2) * kWave + kSmallThreads - 1) / kSmallThreads;
  static_assert(T == 2, "one step of sixteen neurons in the down pass");
  const RowsArgs& p = a.r;
  extern __shared__ u32x4 xs[];
  __shared__ uint32_t s_bits[T * NG];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xgroup = p.mma_slots * kWave;
  float* part = (float*)(xs + (size_t)NG * xgroup);   // [T][gate, up][NG * kMmaPartGroup]
  float* s_z = part + T * 2 * NG * kMmaPartGroup;     // 16-bit: [64] operands of four; fp32: [16 neurons][16]

  // rows as in rows_mma_kernel; a workgroup behind the last row has none and stores zeros
  const int base = p.row_stride == 1 ? (int)blockIdx.x * p.rows_per : (int)(blockIdx.x >> 3) * 8 * p.rows_per + (int)(blockIdx.x & 7);
  const int nrows = max(0, min(p.rows_per, (p.N - base + p.row_stride - 1) / p.row_stride));
  const int kind = wave >> 3, kw = wave & 7;
  const Rows rows(kind ? p.w2 : p.w, base, p.row_vecs, xs, xgroup, p.mma_front, lane, kw);

  // ---- everything is asked for, x first ----
  auto x_vector = [&](int i) { return (i >> 6) * 8 + ((i >> 3) & 1) * 4 + ((i >> 4) & 3) - 8 * p.mma_front; };
  u32x4 xv[NG][NV], nw[NV];
#pragma unroll
  for (int k = 0; k < NV; k++) {
    const int v = x_vector(tid + k * kSmallThreads);
    nw[k] = (p.norm_w ? p.norm_w : p.x)[(unsigned)v < (unsigned)p.row_vecs ? v : 0];
  }
#pragma unroll
  for (int g = 0; g < NG; g++)
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const int i = tid + k * kSmallThreads, b = g * 8 + (i & 7), v = x_vector(i);
      const bool in = b < p.nb && (unsigned)v < (unsigned)p.row_vecs;
      xv[g][k] = p.x[in ? (unsigned)(b * p.row_vecs + v) : 0u];
    }
  __builtin_amdgcn_sched_barrier(0);
  u32x4 w[T][STEPS];
#pragma unroll
  for (int t = 0; t < T; t++) {
    const int q = t * kMmaTileRows + (lane & 7);
    rows.issue(base + q * p.row_stride, q < nrows, 0, w[t]);
  }
  const int q4 = lane >> 4, c16 = lane & 15, dv = wave * 16 + c16;
  const bool cols = wave * 16 < p.row_vecs && nrows > 0;  // uniform
  u32x4 wd[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int j = min(HALF ? 4 * q4 + r : 4 * r + q4, nrows - 1);
    wd[r] = load_stream(cols ? a.wd + (size_t)(base + j * p.row_stride) * p.row_vecs + min(dv, p.row_vecs - 1) : a.wd);
  }
  __builtin_amdgcn_sched_barrier(0);
  auto x_in = [&](int g, int k) {
    const int i = tid + k * kSmallThreads;
    return g * 8 + (i & 7) < p.nb && (unsigned)x_vector(i) < (unsigned)p.row_vecs;
  };
#pragma unroll
  for (int g = 0; g < NG; g++)
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
      for (int e = 0; e < 4; e++) xv[g][k][e] = x_in(g, k) ? xv[g][k][e] : 0u;
  if (p.norm_w) {  // as in MmaX: a thread's vectors are of one batch row
#pragma unroll
    for (int g = 0; g < NG; g++) {
      float ss = 0.f;
#pragma unroll
      for (int k = 0; k < NV; k++) ss = vec_sumsq<DT>(xv[g][k], ss);
      ss = lanes_sum_mod8(ss);
      if (lane < 8) part[(g * kSmallWaves + wave) * 8 + lane] = ss;
    }
    lds_barrier();
#pragma unroll
    for (int g = 0; g < NG; g++) {
      float ss = 0.f;
#pragma unroll
      for (int w = 0; w < kSmallWaves; w++) ss += part[(g * kSmallWaves + w) * 8 + (lane & 7)];
      const float scale = rsqrtf(ss / (float)p.K + p.norm_eps);
#pragma unroll
      for (int k = 0; k < NV; k++)
        if (x_in(g, k)) xv[g][k] = vec_norm_apply<DT>(xv[g][k], scale, nw[k]);
    }
  }
#pragma unroll
  for (int g = 0; g < NG; g++)
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const int i = tid + k * kSmallThreads;
      if (i < xgroup) xs[g * xgroup + i] = xv[g][k];
    }
  lds_barrier();

  // ---- gate and up sums ----
#pragma unroll
  for (int t = 0; t < T; t++) {
    typename Mma<DT>::Acc acc[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) acc[g] = Mma<DT>::zero();
    rows.multiply(w[t], 0, acc);
    mma_store_partials<DT, NG>(acc, part + (t * 2 + kind) * NG * kMmaPartGroup, lane, kw);
  }
  lds_barrier();
  if (wave < T * NG) {  // one wave a tile and group of eight batch rows, one thread per (row rj of the tile, batch row rb)
    const int t = wave / NG, g = wave % NG, rj = lane >> 3, rb = lane & 7, j = t * kMmaTileRows + rj, b = g * 8 + rb;
    const float* sums = part + t * 2 * NG * kMmaPartGroup;
    const bool valid = j < nrows && b < p.nb;
    const float gr = DT::rnd(mma_reduce<DT>(sums, g, rj, rb)), u = mma_reduce<DT>(sums + NG * kMmaPartGroup, g, rj, rb);
    const float av = DT::rnd(gr / (1.f + expf(-gr)));
    const bool act = valid && fabsf(av) > p.t;
    const float z = act ? DT::rnd(av * DT::rnd(u)) : 0.f;
    if (HALF) ((st*)s_z)[(((j >> 2) * 16 + b) << 2) + (j & 3)] = DT::fromf(z);
    else s_z[j * 16 + b] = z;
    if (valid && p.flag_out) p.flag_out[(size_t)b * p.N + base + j * p.row_stride] = act ? 1 : 0;
    const uint64_t bal = __ballot(act);
    uint32_t bits = 0u;
#pragma unroll
    for (int i = 0; i < 8; i++) bits |= ((bal >> (8 * i)) & 0xffull) ? (1u << i) : 0u;
    if (lane == 0) s_bits[wave] = bits;
  }
  lds_barrier();
  uint32_t bits = 0u;  // of the sixteen neurons
#pragma unroll
  for (int i = 0; i < T * NG; i++) bits |= s_bits[i] << (i / NG * 8);
  if (tid == 0) a.counts[blockIdx.x] = __popc(bits);
  if (wave * 16 >= p.row_vecs) return;
  // ---- down: batch rows 8.. of the operands are not written for NG = 1, and their sums are not stored ----
  constexpr int NA = HALF ? 8 : 4;
  f32x4 acc[NA];
#pragma unroll
  for (int e = 0; e < NA; e++) acc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 v[4];
#pragma unroll
  for (int r = 0; r < 4; r++) v[r] = (bits >> (HALF ? 4 * q4 + r : 4 * r + q4)) & 1u ? wd[r] : zero4();  // a dead neuron's weights may be anything
  if constexpr (HALF) {
    const u32x2 zop = ((const u32x2*)s_z)[lane];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const u32x2 lo = {__builtin_amdgcn_perm(v[1][i], v[0][i], 0x05040100u), __builtin_amdgcn_perm(v[3][i], v[2][i], 0x05040100u)};
      const u32x2 hi = {__builtin_amdgcn_perm(v[1][i], v[0][i], 0x07060302u), __builtin_amdgcn_perm(v[3][i], v[2][i], 0x07060302u)};
      acc[2 * i] = DownMma<DT>::run(zop, lo, acc[2 * i]);
      acc[2 * i + 1] = DownMma<DT>::run(zop, hi, acc[2 * i + 1]);
    }
  } else {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const float z = s_z[(4 * r + q4) * 16 + c16];
#pragma unroll
      for (int e = 0; e < 4; e++) acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(z, __uint_as_float(v[r][e]), acc[e], 0, 0, 0);
    }
  }
  if (dv < p.row_vecs) {
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (4 * q4 + i < p.nb) {
        float* out = a.partial + ((size_t)blockIdx.x * p.nb + 4 * q4 + i) * p.K + (size_t)dv * VEC;
#pragma unroll
        for (int h = 0; h < NA / 4; h++) *(float4*)(out + 4 * h) = make_float4(acc[4 * h][i], acc[4 * h + 1][i], acc[4 * h + 2][i], acc[4 * h + 3][i]);
      }
  }
}

// ---- host ---------------------------------------------------------------------------------------------------------------------
constexpr int kSmallMaxNeurons = 8192;
// Workgroups of a layer of I neurons at most: it bounds the partial sums.
inline int small_max_groups(int I) { return (I + 8 * kSmallRows - 1) / (8 * kSmallRows) * 8; }

// Fills rows_per .. mma_slots; returns the grid, 0 if a row is too long.
inline int small_layout(RowsArgs& a, bool mma) {
  if (a.row_vecs > kSmallMaxVecs) return 0;
  a.rows_per = kSmallRows;
  a.row_stride = mma && a.row_vecs % 8 != 0 ? 8 : 1;
  if (mma) {
    const MmaSplit sp = rows_mma_split(a);
    if (sp.chunks != 1 || sp.steps > 5) return 0;
    a.mma_front = sp.front;
    a.mma_slots = sp.slots;
  }
  return a.row_stride == 1 ? (a.N + kSmallRows - 1) / kSmallRows : small_max_groups(a.N);
}

}  // namespace cats

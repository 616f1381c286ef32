// Gate and fused gate + up pass for batches of 3..16 rows in 16-bit types and 5..16 rows of fp32, on the matrix cores.
//
// Why not the wave-per-row kernel: with B batch rows every 16-byte weight vector costs 4 * B v_dot2 and B / 2
// LDS reads of x per lane.  From B = 4 on, that arithmetic plus the LDS traffic takes as long as the HBM stream
// itself and the three do not overlap inside a wave.  One v_mfma_f32_16x16x32 eats 1 KiB of weights against all
// batch rows at once, with one 16-byte LDS read per lane, so the kernel goes back to being a weight stream.
//
// Tile shape.  The MFMA wants 16 "rows" x 32 k per instruction with 4 lanes per row, i.e. 64 contiguous bytes
// per weight row per load instruction -- half a cache line, which streams about 25 % slower than whole lines.
// So a tile is 8 weight rows x 64 k instead: MFMA row m holds weight row m % 8, k half m / 8, and MFMA column n
// holds batch row n % 8 with the same k half n / 8.  Eight lanes then read 128 contiguous bytes of a row.  The
// (m < 8, n < 8) and (m >= 8, n >= 8) quadrants of the result are the two halves of the dot products, the other
// two quadrants pair mismatched halves and are dropped.
//
// Work split.  One persistent workgroup per CU: x is staged once in LDS in operand order (one linear 16-byte
// read per lane per step).  A workgroup owns ceil(N / grid) rows, consecutive ones where the rows start on cache lines --
// the same number of weight bytes for every CU; dealing whole tiles instead leaves 96 of 256 workgroups with 6 tiles against 5 at N = 11008 and spreads their
// ends over 4-6 us instead of 1.3-2 (the kernel's duration is the same: the memory system is the limit) -- cut into
// tiles of eight, the last one partial (its missing rows fetch nothing).  The rows of a range do not end on multiples of eight, so the union of the flags goes out as one byte
// per row (ubytes_out) rather than as bits.  The waves of a workgroup split K.  Tiles move through a software
// pipeline, one per round:
//   round r:  MFMA on the gate rows of tile r (loaded two rounds ago) -> per-wave partial sums to LDS;
//             gate loads of tile r + 2 go out; wave 0 adds the partials in wave order, applies SiLU and the
//             threshold and publishes the tile's union bits; up loads of tile r go out for the active rows only
//             (lanes of inactive rows re-read one cached line, so no HBM bytes move for them); MFMA on the up rows of tile
//             r - 1 (loaded one round ago) -> partials -> wave 0 writes z = a * up for tile r - 1.
// So the gate rows of two tiles and the up rows of one are in flight while a fourth tile is being reduced; the
// only exposed latencies are the first gate load and the last up load.  The two load rings are addressed
// statically (the loop is unrolled by two): a register that a load in flight will write cannot be moved.
#pragma once
#include "cats_rows.h"

namespace cats {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// run: one 16-byte vector of weights times one of x per lane.  Acc: the sums of a tile; total: as one register set.
template <class DT> struct Mma;
template <> struct Mma<F16> {
  typedef f32x4 Acc;
  static __device__ __forceinline__ Acc zero() { return f32x4{0.f, 0.f, 0.f, 0.f}; }
  static __device__ __forceinline__ f32x4 total(const Acc& c) { return c; }
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mma<BF16> : Mma<F16> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};

// fp32: one v_mfma_f32_16x16x4 per element of the vectors.  Each of the four keeps sums of its own, so that a chain of additions is
// as long as a lane's in the wave-per-row kernel (K / 64 products) and the result no further off.
template <> struct Mma<F32> {
  struct Acc {
    f32x4 e[4];
  };
  static __device__ __forceinline__ Acc zero() {
    Acc c;
#pragma unroll
    for (int i = 0; i < 4; i++) c.e[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    return c;
  }
  static __device__ __forceinline__ f32x4 total(const Acc& c) {
    f32x4 s;
#pragma unroll
    for (int i = 0; i < 4; i++) s[i] = (c.e[0][i] + c.e[1][i]) + (c.e[2][i] + c.e[3][i]);
    return s;
  }
  static __device__ __forceinline__ Acc run(u32x4 a, u32x4 b, Acc c) {
#pragma unroll
    for (int i = 0; i < 4; i++) c.e[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[i]), __uint_as_float(b[i]), c.e[i], 0, 0, 0);
    return c;
  }
};

constexpr int kMmaWaves = 8;
constexpr int kMmaThreads = kMmaWaves * kWave;
constexpr int kMmaTileRows = 8;
constexpr int kMmaPart = 128;    // floats per wave in a partial buffer (the two useful quadrants)

// How a row of K elements is cut.  A step is 128 bytes, a whole cache line (64 16-bit elements or 32 of fp32): where the pitch of the rows is no multiple
// of 128 bytes the steps of a row start at the line its first element lies in, "phase" 16-byte vectors before it (phase =
// address / 16 mod 8), and the lanes in front of the row are padding like those behind it.  All rows of a tile need the same
// phase, because they share the x operand; rows eight apart have it, so a workgroup then owns every eighth row of a block
// (rows_mma_layout).  Steps cut at the row start instead straddle two lines each: 22.3 against 19.8 us for 8191 rows of 3080
// and 3072 elements, 78.7 against 63.5 us for 16000 rows of 6152 and 6144.
// The steps of a row are dealt to the eight waves as contiguous runs, the last waves one more if they do not divide evenly.  A
// register set holds up to nine steps of one tile; longer rows take two sets per tile ("chunks") and add both into the same
// accumulator.  steps: per wave and chunk (the kernels' template argument), chunks: 1 or 2; all 0 if the row is too long.
// slots: steps of an x operand in LDS -- those of the row with the largest phase; where there are phases one of zeros in front
// (`front`), and behind what the last wave's register sets can have past the end of its run: the rounding up to two chunks, and
// one for a phase that needs a step less or for a row that does not fill its steps.
struct MmaSplit {
  int steps, chunks, front, slots;
};
inline MmaSplit rows_mma_split(const RowsArgs& a) {
  const bool shifted = a.row_vecs % 8 != 0 || (((uintptr_t)a.w | (uintptr_t)a.w2) & 127u) != 0;
  const int total = (a.row_vecs + (shifted ? 7 : 0) + 7) / 8;
  const int per_wave = (total + kMmaWaves - 1) / kMmaWaves;
  if (per_wave > 18) return {0, 0, 0, 0};
  const int chunks = per_wave > 9 ? 2 : 1;
  const int steps = (per_wave + chunks - 1) / chunks, front = shifted ? 1 : 0;
  return {steps, chunks, front, front + total + (steps * chunks - per_wave) + (shifted || total < kMmaWaves * per_wave ? 1 : 0)};
}
// Which rows a workgroup owns, and the grid: about one persistent workgroup per CU.  Workgroup i owns rows base + q * stride for q <
// rows_per: `rows_per` consecutive rows (stride 1), or, where the rows' phases differ, every eighth row of the block of
// 8 * rows_per rows that it shares with seven others.
inline int rows_mma_layout(RowsArgs& a, int cus) {
  const int ntiles = (a.N + kMmaTileRows - 1) / kMmaTileRows;
  const int grid = ntiles < cus ? ntiles : cus;
  a.rows_per = (a.N + grid - 1) / grid;
  a.row_stride = a.row_vecs % 8 != 0 ? 8 : 1;
  return a.row_stride == 1 ? (a.N + a.rows_per - 1) / a.rows_per : 8 * ((a.N + 8 * a.rows_per - 1) / (8 * a.rows_per));
}
// dynamic LDS: x operands, gate partials, up partials -- each once per group of eight batch rows (ng = 1 or 2)
inline size_t rows_mma_lds_bytes(const RowsArgs& a, int ng = 1) {
  return (size_t)ng * ((size_t)rows_mma_split(a).slots * kWave * sizeof(u32x4) + 2u * kMmaWaves * kMmaPart * sizeof(float));
}

// This lane's view of one weight matrix: its place in a tile (weight row lane % 8, 16-byte piece `piece` of the row's 128-byte
// steps), its first vector of a row, the end of those it reads, and where it finds the x operand of its wave's first step.
// STEPS, CH: as MmaSplit.
template <class DT, int STEPS, int CH, int NG>
struct MmaRows {
  const u32x4* __restrict__ w;
  int row_vecs, vec0, vend;
  const u32x4* xs;   // x operands of this lane, first step of its wave
  int xgroup;        // operand vectors between the two groups of eight batch rows

  // Only a wave's first step can start in front of a row.  Only its last two can be missing or reach past the end (the last wave
  // has the longest run, one step less where this phase needs one step less than the largest), or three where two chunks
  // round the run up.  The checks of all others fold away.
  static __device__ __forceinline__ constexpr bool edge(int c, int s) { return (c == 0 && s == 0) || (c == CH - 1 && s >= STEPS - 1 - CH); }
  __device__ __forceinline__ bool outside(int c, int s) const { return edge(c, s) && ((unsigned)vec(c, s) >= (unsigned)vend); }
  __device__ __forceinline__ int vec(int c, int s) const { return vec0 + (c * STEPS + s) * 8; }

  // row: any row this workgroup owns (they share a phase)
  __device__ __forceinline__ MmaRows(const u32x4* w_, int row, int row_vecs_, const u32x4* xs_, int xgroup_, int front, int lane, int wave)
      : w(w_), row_vecs(row_vecs_), xgroup(xgroup_) {
    const int phase = (int)((((uintptr_t)w_ >> 4) + (size_t)row * row_vecs_) & 7u);
    const int steps = (row_vecs + phase + 7) >> 3;
    const int longer = kMmaWaves - steps % kMmaWaves;  // the first wave whose run is one step longer
    const int first = wave * (steps / kMmaWaves) + max(wave - longer, 0);
    const int count = steps / kMmaWaves + (wave >= longer ? 1 : 0);
    const int piece = ((lane >> 3) & 1) * 4 + (lane >> 4);
    vec0 = first * 8 + piece - phase;
    vend = max(0, min(row_vecs, (first + count) * 8 - phase));  // 0: a wave without steps
    xs = xs_ + slot(vec0 + 8 * front, lane & 7);
  }
  // x operands in LDS: vector v of batch row b (of a group of eight) sits at slot(v + 8 * front, b), so that the eight vectors of a step,
  // whatever the phase, are 64 slots with distinct banks in every quarter wave.
  static __device__ __forceinline__ int slot(int v, int b) { return (v >> 3) * kWave + (v & 3) * 16 + ((v >> 2) & 1) * 8 + b; }

  // Loads of chunk c of this lane's row, never predicated: a lane with nothing to fetch (mine false: rows past the end of the
  // range or without a flag; or outside the row) reads the first vector of the matrix over and over, which stays in
  // cache and moves nothing from HBM.
  __device__ __forceinline__ void issue(int row, bool mine, int c, u32x4 (&dst)[STEPS]) const {
    const u32x4* src = mine ? w + ((ptrdiff_t)row * row_vecs + vec(c, 0)) : w;
    const int stride = mine ? 8 : 0;
#pragma unroll
    for (int s = 0; s < STEPS; s++) dst[s] = load_stream(outside(c, s) ? w : src + s * stride);
  }
  // acc += chunk c of the tile times the staged x rows.  What a load outside the row brought are weights of another
  // place, perhaps infinities: replaced by zeros before they meet the zeros of the x padding.
  typedef typename Mma<DT>::Acc Acc;
  __device__ __forceinline__ void multiply(const u32x4 (&src)[STEPS], int c, Acc (&acc)[NG]) const {
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
      for (int s = 0; s < STEPS; s++)
        acc[g] = Mma<DT>::run(outside(c, s) ? zero4() : src[s], xs[g * xgroup + (c * STEPS + s) * kWave], acc[g]);
  }
  // The same with this lane's x operands of chunk 0 in registers.  The groups of batch rows take turns: their sums are two
  // independent chains of MFMAs.
  __device__ __forceinline__ void hold(u32x4 (&x)[NG][STEPS]) const {
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
      for (int s = 0; s < STEPS; s++) x[g][s] = xs[g * xgroup + s * kWave];
  }
  __device__ __forceinline__ void multiply(const u32x4 (&src)[STEPS], const u32x4 (&x)[NG][STEPS], Acc (&acc)[NG]) const {
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
      const u32x4 w = outside(0, s) ? zero4() : src[s];
#pragma unroll
      for (int g = 0; g < NG; g++) acc[g] = Mma<DT>::run(w, x[g][s], acc[g]);
    }
  }
};

constexpr int kMmaPartGroup = kMmaWaves * kMmaPart;  // partial-sum floats of one group of eight batch rows

// The two useful quadrants of the accumulators -> this wave's part of a partial buffer.
template <class DT, int NG>
__device__ __forceinline__ void mma_store_partials(const typename Mma<DT>::Acc (&acc)[NG], float* part, int lane, int wave) {
  const int ncol = lane & 15;
  const bool keep = (lane < 32) ? (ncol < 8) : (ncol >= 8);
  const int slot = (lane >> 5) * 16 + ((lane >> 4) & 1) * 8 + (ncol & 7);
  if (keep) {
#pragma unroll
    for (int g = 0; g < NG; g++) {
      float* dst = part + g * kMmaPartGroup + wave * kMmaPart + slot;
      const f32x4 sum = Mma<DT>::total(acc[g]);
#pragma unroll
      for (int i = 0; i < 4; i++) dst[i * 32] = sum[i];
    }
  }
}
// Adds the eight waves' partials (two halves each) of one output, src its first wave's: in wave order, in fp32 pairwise, as the
// wave-per-row kernel's lanes meet (its error is the measure there: sixteen additions in a row cost 2 to 6 % of it).
template <class DT>
__device__ __forceinline__ float mma_sum_waves(const float* src, int wave_stride) {
  if constexpr (sizeof(typename DT::st) == 4) {
    float v[kMmaWaves];
#pragma unroll
    for (int w = 0; w < kMmaWaves; w++) v[w] = src[w * wave_stride] + src[w * wave_stride + 16];
    return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  } else {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < kMmaWaves; w++) s += src[w * wave_stride] + src[w * wave_stride + 16];
    return s;
  }
}
// One thread per (row rj of the tile, batch row rb) of group g.
template <class DT>
__device__ __forceinline__ float mma_reduce(const float* part, int g, int rj, int rb) {
  return mma_sum_waves<DT>(part + g * kMmaPartGroup + (rj & 3) * 32 + (rj >> 2) * 8 + rb, kMmaPart);
}

// Staging of x: thread tid takes vectors tid + k * 512 of the nb rows, row by row in groups of eight; the loads of all are in flight together.
// The padding steps and the batch rows past nb are zero.  NV: vectors per thread, at least those of a whole operand.
template <int NV, int NG>
struct MmaX {
  u32x4 v[NG][NV];
  int tid, front;
  // Slot i of an operand holds vector(i), counted from the row's first, of batch row gb * 8 + i % 8.  No branches (x is
  // what everything waits for): a slot without one fetches the first vector of x and stores zeros.
  __device__ __forceinline__ int vector(int i) const { return (i >> 6) * 8 + ((i >> 3) & 1) * 4 + ((i >> 4) & 3) - 8 * front; }
  __device__ __forceinline__ bool in(const RowsArgs& p, int gb, int i) const {
    return (gb * 8 + (i & 7) < p.nb) & ((unsigned)vector(i) < (unsigned)p.row_vecs);
  }
  __device__ __forceinline__ void fetch(const RowsArgs& p) {
#pragma unroll
    for (int gb = 0; gb < NG; gb++)
#pragma unroll
      for (int k = 0; k < NV; k++) {
        const int i = front * kWave + tid + k * kMmaThreads;
        const unsigned o = (gb * 8 + (i & 7)) * p.row_vecs + vector(i);
        v[gb][k] = p.x[in(p, gb, i) ? o : 0u];
      }
  }
  // What padding slots and batch rows past nb have fetched becomes zero.
  __device__ __forceinline__ void mask(const RowsArgs& p) {
#pragma unroll
    for (int gb = 0; gb < NG; gb++)
#pragma unroll
      for (int k = 0; k < NV; k++) {
        const bool ok = in(p, gb, front * kWave + tid + k * kMmaThreads);
#pragma unroll
        for (int e = 0; e < 4; e++) v[gb][k][e] = ok ? v[gb][k][e] : 0u;
      }
  }
  // xgroup: slots of one group's operand; the last one is padding where fewer than NV * 512 are needed
  __device__ __forceinline__ void store(u32x4* xs, int xgroup) const {
#pragma unroll
    for (int gb = 0; gb < NG; gb++) {
      if (front && tid < kWave) xs[gb * xgroup + tid] = zero4();
#pragma unroll
      for (int k = 0; k < NV; k++) xs[gb * xgroup + min(front * kWave + tid + k * kMmaThreads, xgroup - 1)] = v[gb][k];
      for (int i = front * kWave + tid + NV * kMmaThreads; i < xgroup; i += kMmaThreads) xs[gb * xgroup + i] = zero4();
    }
  }
  // The RMS norm of the masked rows, in registers: slots of one thread, and of the eight lanes that agree modulo eight, are of one batch row.
  // The squares are added by thread, then over those lanes, then over the waves in their order.  s_sq: 64 floats of LDS a group.
  // The weights have been asked for with x: behind the first tile they would come in with it.
  __device__ __forceinline__ void fetch_norm(const RowsArgs& p, u32x4 (&nw)[NV]) const {
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const int q = vector(front * kWave + tid + k * kMmaThreads);
      nw[k] = p.norm_w[(unsigned)q < (unsigned)p.row_vecs ? q : 0];
    }
  }
  template <class DT>
  __device__ __forceinline__ void norm(const RowsArgs& p, const u32x4 (&nw)[NV], float* s_sq) {
    const int lane = tid & (kWave - 1), wave = tid >> 6;
#pragma unroll
    for (int gb = 0; gb < NG; gb++) {
      float ss = 0.f;
#pragma unroll
      for (int k = 0; k < NV; k++) ss = vec_sumsq<DT>(v[gb][k], ss);
      ss = lanes_sum_mod8(ss);
      if (lane < 8) s_sq[(gb * kMmaWaves + wave) * 8 + lane] = ss;
    }
    lds_barrier();
#pragma unroll
    for (int gb = 0; gb < NG; gb++) {
      float ss = 0.f;
#pragma unroll
      for (int w = 0; w < kMmaWaves; w++) ss += s_sq[(gb * kMmaWaves + w) * 8 + (lane & 7)];
      const float scale = rsqrtf(ss / (float)p.K + p.norm_eps);
#pragma unroll
      for (int k = 0; k < NV; k++) {
        // two register sets of bf16: else all of x is taken apart into floats at once, into twice its registers, and spilled
        if constexpr (NV > 9) asm volatile("" : "+v"(v[gb][k]));
        if (in(p, gb, front * kWave + tid + k * kMmaThreads)) v[gb][k] = vec_norm_apply<DT>(v[gb][k], scale, nw[k]);
      }
    }
  }
};

// UP = false is the gate pass alone (activations, flags and union bits out; no up rows, no z).
// NG = 2 takes 9..16 batch rows in one pass over the weights: the second group of eight rows is a second x operand in
// LDS and a second MFMA on the weight registers the first one just used, so the weights are still read once.
// CH = 2 (rows of more than 72 steps, 4608 16-bit elements; their x fills 128 KiB of LDS at 8192): a tile is two register sets, so the gate ring
// holds one tile ahead instead of two, and the up sums of tile r - 1 are taken before the up rows of tile r overwrite their set.
// A wave multiplies the same steps of K for every tile, so one chunk's x operands stay in its registers (kHeld) once they are
// staged: read from LDS for every tile they cost a CU 1 KiB (2 KiB at 9..16 rows) of LDS traffic a KiB of weights, 6 us of a 43 us
// kernel at sixteen rows, part of it in front of the next loads (4096 / 14336 bf16 16 rows: kernel 43.7 / 41.7 us, call 70.6 / 70.0;
// 3080 / 8191 3 rows 33.25 / 33.0; 4 and 8 rows of 4096 as before).
// x may be given before its RMS norm (p.norm_w, UP only).  With two register sets that is an instance of its own, NORM: all of x and the
// norm's weights beside the first set are up to 80 registers more, and whole calls without a norm held them, or spilled: 8160 / 12288 bf16
// 4 rows 105.4 us, now 101.3, 8 rows 112.8, 109.0; 8192 / 12288 fp16 4 rows 95.6, 94.8; fp32 4512 / 11008 8 rows 123.5, 122.1.  One
// set takes as many with and without.
template <class DT, int STEPS, int CH, bool UP, int NG, bool NORM>
__global__ __launch_bounds__(kMmaThreads) void rows_mma_kernel(RowsArgs p) {
  typedef typename DT::st st;
  typedef MmaRows<DT, STEPS, CH, NG> Rows;
  static_assert(!NORM || (UP && CH == 2), "an instance of its own where there are two register sets");
  constexpr bool kHeld = CH == 1 && NG * STEPS <= (sizeof(st) == 2 ? 16 : 9);  // more would not fit beside four sets of weights
  const bool norm = CH == 2 ? NORM : UP && p.norm_w != nullptr;
  extern __shared__ u32x4 xs[];  // [NG][mma_slots][64] x operands, then the partial buffers
  __shared__ uint32_t s_any;

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xgroup = p.mma_slots * kWave;
  float* part_g = (float*)(xs + (size_t)NG * xgroup);
  float* part_u = part_g + NG * kMmaPartGroup;

  // this workgroup's rows: base + q * stride, q < nrows
  const int base = p.row_stride == 1 ? (int)blockIdx.x * p.rows_per : (int)(blockIdx.x >> 3) * 8 * p.rows_per + (int)(blockIdx.x & 7);
  const int nrows = max(0, min(p.rows_per, (p.N - base + p.row_stride - 1) / p.row_stride));
  const int my_tiles = (nrows + kMmaTileRows - 1) / kMmaTileRows;
  const int jl = lane & 7;  // this lane's weight row in a tile
  const Rows gate(p.w, base, p.row_vecs, xs, xgroup, p.mma_front, lane, wave);
  const Rows up(UP ? p.w2 : p.w, base, p.row_vecs, xs, xgroup, p.mma_front, lane, wave);

  auto issue_gate = [&](int it, int c, u32x4 (&dst)[STEPS]) {
    const int q = it * kMmaTileRows + jl;
    gate.issue(base + q * p.row_stride, q < nrows, c, dst);
  };
  auto issue_up = [&](int it, int c, u32x4 (&dst)[STEPS]) {  // only the rows of the tile that some batch row keeps
    const int q = it * kMmaTileRows + jl;
    up.issue(base + q * p.row_stride, q < nrows && ((s_any >> jl) & 1u), c, dst);
  };
  // wave 0, one thread per (row rj of the tile, batch row rb)
  const int rj = (lane >> 3), rb = lane & 7;

  // wave 0 carries the gate results of the previous tile until its up sums arrive
  float prev_a[NG];
  bool prev_act[NG], prev_valid[NG];
#pragma unroll
  for (int g = 0; g < NG; g++) {
    prev_a[g] = 0.f;
    prev_act[g] = prev_valid[g] = false;
  }
  uint32_t prev_bits = 0u;
  int prev_row = 0;

  u32x4 held[NG][STEPS];
  const bool one_phase = gate.xs == up.xs;  // uniform; else the two matrices start at different places of a line and take turns in `held`
  // gbuf, ubuf, uprev: the register sets of the round.  One chunk: gbuf[0] is the tile's set, ubuf[0] takes its up rows, uprev[0]
  // holds those of the tile before.  Two chunks: gbuf[0..1] and ubuf[0..1] are the tile's two sets, uprev is ubuf.
  auto round_body = [&](int r, u32x4 (&ga)[STEPS], u32x4 (&gb)[STEPS], u32x4 (&ucur)[STEPS], u32x4 (&uprev)[STEPS]) {
    typename Mma<DT>::Acc acc[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) acc[g] = Mma<DT>::zero();
    if constexpr (kHeld) {
      if (UP && !one_phase) gate.hold(held);
      gate.multiply(ga, held, acc);
    } else {
      gate.multiply(ga, 0, acc);
    }
    if constexpr (CH == 2) {
      issue_gate(r + 1, 0, ga);
      gate.multiply(gb, 1, acc);
      mma_store_partials<DT, NG>(acc, part_g, lane, wave);
      issue_gate(r + 1, 1, gb);
    } else {
      mma_store_partials<DT, NG>(acc, part_g, lane, wave);
      issue_gate(r + 2, 0, ga);
    }
    __syncthreads();
    float a[NG];
    bool act[NG], valid[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) {
      a[g] = 0.f;
      act[g] = valid[g] = false;
    }
    uint32_t bits8 = 0u;
    const int row = base + (r * kMmaTileRows + rj) * p.row_stride;
    const bool row_in = r * kMmaTileRows + rj < nrows;
    if (wave == 0 && r < my_tiles) {
      uint64_t bal = 0ull;
#pragma unroll
      for (int g = 0; g < NG; g++) {
        const int b = g * 8 + rb;  // batch row of this thread in group g
        valid[g] = row_in && b < p.nb;
        const float gr = DT::rnd(mma_reduce<DT>(part_g, g, rj, rb));
        a[g] = DT::rnd(gr / (1.f + expf(-gr)));
        act[g] = valid[g] && fabsf(a[g]) > p.t;
        bal |= __ballot(act[g]);
        if (valid[g] && p.flag_out) p.flag_out[(size_t)b * p.N + row] = act[g] ? 1 : 0;
        if (!UP && valid[g] && p.a_out) ((st*)p.a_out)[(size_t)b * p.N + row] = DT::fromf(a[g]);
      }
#pragma unroll
      for (int j = 0; j < 8; j++) bits8 |= ((bal >> (8 * j)) & 0xffull) ? (1u << j) : 0u;
      if (lane == 0) s_any = bits8;
      if (p.ubytes_out && rb == 0 && row_in) p.ubytes_out[row] = (uint8_t)((bits8 >> rj) & 1u);
    }
    __syncthreads();
    if (!UP) return;
#pragma unroll
    for (int g = 0; g < NG; g++) acc[g] = Mma<DT>::zero();
    if constexpr (CH == 2) {
      up.multiply(ucur, 0, acc);
      issue_up(r, 0, ucur);
      up.multiply(uprev, 1, acc);
      issue_up(r, 1, uprev);
    } else {
      issue_up(r, 0, ucur);
      if constexpr (kHeld) {
        if (!one_phase) up.hold(held);
        up.multiply(uprev, held, acc);
      } else {
        up.multiply(uprev, 0, acc);
      }
    }
    mma_store_partials<DT, NG>(acc, part_u, lane, wave);
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int g = 0; g < NG; g++) {
        if (r >= 1 && prev_valid[g]) {
          const float u = mma_reduce<DT>(part_u, g, rj, rb);
          const float z = prev_act[g] ? DT::rnd(prev_a[g] * DT::rnd(u)) : 0.f;
          const size_t o = (size_t)(g * 8 + rb) * p.N + prev_row;
          if (p.z32_out && ((prev_bits >> rj) & 1u)) p.z32_out[o] = z;
          if (p.zt_out) ((st*)p.zt_out)[o] = DT::fromf(z);
        }
        prev_a[g] = a[g]; prev_act[g] = act[g]; prev_valid[g] = valid[g];
      }
      prev_bits = bits8; prev_row = row;
    }
  };

  CATS_RSTAMP(0);
  // ---- prologue.  x is requested before the first weight load goes out, so that its read does not queue behind
  // the weight requests of the whole machine. ---------------------------------------------------------------------
  u32x4 g0[STEPS], g1[STEPS], u0[STEPS], u1[STEPS];
  {
    MmaX<STEPS * CH, NG> x;
    x.tid = tid;
    x.front = p.mma_front;
    x.fetch(p);
    u32x4 nw[STEPS * CH];
    if (norm) x.fetch_norm(p, nw);
    // the first gate set goes out behind x, before x is waited for: it is a memory round trip ahead when the staging is done
    __builtin_amdgcn_sched_barrier(0);
    issue_gate(0, 0, g0);
    __builtin_amdgcn_sched_barrier(0);
    x.mask(p);
    if (norm) x.template norm<DT>(p, nw, part_g);
    x.store(xs, xgroup);
#pragma unroll
    for (int c = 0; c < STEPS; c++) u1[c] = zero4();  // defined before the first (unused) up product
    if constexpr (CH == 2) {
#pragma unroll
      for (int c = 0; c < STEPS; c++) u0[c] = zero4();
    }
  }
  // a barrier for LDS only: __syncthreads() would also wait for the gate loads in flight
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  // The second gate set goes out after the barrier: a wave blocks at issue once the CU's miss queue is full, so
  // everything issued before the barrier delays the moment the staged x becomes usable.
  issue_gate(CH == 2 ? 0 : 1, CH == 2 ? 1 : 0, g1);
  if constexpr (CH == 2) __builtin_amdgcn_sched_barrier(0);  // all of it: else its last loads wait behind the first products
  CATS_RSTAMP(1);
  if constexpr (kHeld) gate.hold(held);

  // rounds 0 .. my_tiles: the last one only drains the up sums of the last tile
  const int last = UP ? my_tiles : my_tiles - 1;
  if constexpr (CH == 2) {
    for (int r = 0; r <= last; r++) {
      round_body(r, g0, g1, u0, u1);
#ifdef CATS_TIMING
      if (r < 10) CATS_RSTAMP(2 + (r >> 1));
#endif
    }
  } else {
    for (int r = 0; r <= last; r += 2) {
      round_body(r, g0, g0, u0, u1);
      if (r + 1 <= last) round_body(r + 1, g1, g1, u1, u0);
#ifdef CATS_TIMING
      if (r < 10) CATS_RSTAMP(2 + (r >> 1));
#endif
    }
  }
  CATS_RSTAMP(7);
}

// The up pass alone, for callers that bring the gate activations (kUp; flags = |a| > t, or the caller's flag bytes):
//   z[b, j] = a[b, j] * (x[b] . wup[j])  where flag[b, j], else 0; rows of W_up without a flag in any batch row are not read.
// Out: the union of the flags to ubytes_out (optional); z as fp32 for the rows that were read (flags derived: the sparse
// down pass that follows reads no others) or for every row (flags given), and / or in the storage type for every row.
// Same tiles, operand layout and work split as rows_mma_kernel.  With a given, every tile's union bits are known before
// the first weight byte moves: the workgroup stages its range of a in LDS, derives the bits of all its tiles, and then
// streams W_up with two tiles in flight (a ring of two register sets, the loop unrolled by two) and one barrier per tile
// (the per-wave partial sums alternate between two buffers: wave 0 adds up tile r while the others multiply tile r + 1).
// NG = 2 takes 9..16 batch rows: a second x operand in LDS and a second MFMA on the same weight registers.
// dynamic LDS, per group of eight batch rows: x operands | two partial buffers | a of the range, [8][rows_pad] in storage
// type | its flags, [8][rows_pad] bytes; then one byte of union bits per tile
inline size_t rows_mma_up_lds_bytes(const RowsArgs& a, int rows_pad, int ng) {
  return rows_mma_lds_bytes(a, ng) + (size_t)ng * 8 * rows_pad * 3 + (size_t)(rows_pad / 8 + 15) / 16 * 16;
}

template <class DT, int STEPS, int CH, int NG>
__global__ __launch_bounds__(kMmaThreads) void rows_mma_up_kernel(RowsArgs p) {
  typedef typename DT::st st;
  typedef MmaRows<DT, STEPS, CH, NG> Rows;
  static_assert(sizeof(st) == 2, "16-bit types only");
  extern __shared__ u32x4 xs[];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xgroup = p.mma_slots * kWave;

  // this workgroup's rows: base + q * stride, q < nrows
  const int base = p.row_stride == 1 ? (int)blockIdx.x * p.rows_per : (int)(blockIdx.x >> 3) * 8 * p.rows_per + (int)(blockIdx.x & 7);
  const int nrows = max(0, min(p.rows_per, (p.N - base + p.row_stride - 1) / p.row_stride));
  const int rows_pad = (p.rows_per + kMmaTileRows - 1) / kMmaTileRows * kMmaTileRows;
  const int my_tiles = (nrows + kMmaTileRows - 1) / kMmaTileRows;
  const int jl = lane & 7;
  const Rows up(p.w, base, p.row_vecs, xs, xgroup, p.mma_front, lane, wave);
  constexpr int NB = NG * 8;                                // batch rows the kernel is laid out for
  float* part = (float*)(xs + NG * xgroup);                 // [2][NG][kMmaPartGroup]
  st* s_a = (st*)(part + 2 * NG * kMmaPartGroup);           // [NB][rows_pad]
  uint8_t* s_f = (uint8_t*)(s_a + NB * rows_pad);           // [NB][rows_pad]
  uint8_t* s_bits = s_f + NB * rows_pad;                    // [rows_pad / 8]
  const int rj = lane >> 3, rb = lane & 7;

  CATS_RSTAMP(0);
  // ---- prologue: x -> LDS in operand order (as rows_mma_kernel), a of the range -> LDS, the bits of every tile ----------
  {
    MmaX<STEPS * CH, NG> x;
    x.tid = tid;
    x.front = p.mma_front;
    x.fetch(p);
    const st* ain = (const st*)p.a_in;
    for (int e = tid; e < NB * rows_pad; e += kMmaThreads) {
      const int b = e / rows_pad, j = e - b * rows_pad;
      const bool in = b < p.nb && j < nrows;  // the padding of the range and of the batch is never flagged
      const size_t o = (size_t)b * p.N + base + j * p.row_stride;
      const st av = in ? ain[o] : DT::fromf(0.f);
      s_a[e] = av;
      s_f[e] = in && (p.flag_in ? p.flag_in[o] != 0 : fabsf(DT::tof(av)) > p.t) ? 1 : 0;
    }
    x.mask(p);
    x.store(xs, xgroup);
  }
  __syncthreads();
  // one thread per row of the range: any batch row flagged?  Eight neighbouring lanes make a tile's byte.
  for (int j0 = 0; j0 < rows_pad; j0 += kMmaThreads) {
    const int j = j0 + tid;
    bool any = false;
    if (j < rows_pad) {
#pragma unroll
      for (int b = 0; b < NB; b++) any = any || s_f[b * rows_pad + j] != 0;
      if (p.ubytes_out && j < nrows) p.ubytes_out[base + j * p.row_stride] = any ? 1 : 0;
    }
    const uint64_t bal = __ballot(any);
    if (j < rows_pad && (lane & 7) == 0) s_bits[j >> 3] = (uint8_t)((bal >> (lane & 56)) & 0xffull);
  }
  __syncthreads();
  CATS_RSTAMP(1);

  auto issue = [&](int it, int c, u32x4 (&dst)[STEPS]) {
    const int q = it * kMmaTileRows + jl;
    const uint32_t bits = it < my_tiles ? s_bits[it] : 0u;
    up.issue(base + q * p.row_stride, q < nrows && ((bits >> jl) & 1u), c, dst);
  };
  // wave 0, one thread per (row rj of the tile, batch row rb): the eight waves' partials in wave order, then z = a * up
  auto finish = [&](int r, const float* my_part) {
    const int j = r * kMmaTileRows + rj;
    const int row = base + j * p.row_stride;
    const bool live = (s_bits[r] >> rj) & 1u;       // the row was read
#pragma unroll
    for (int gb = 0; gb < NG; gb++) {
      const int b = gb * 8 + rb;
      const float u = mma_reduce<DT>(my_part, gb, rj, rb);
      const float a = DT::tof(s_a[b * rows_pad + j]);
      if (j < nrows && b < p.nb) {
        const float z = s_f[b * rows_pad + j] ? DT::rnd(a * DT::rnd(u)) : 0.f;  // u of a row that was not read is noise: never used
        const size_t o = (size_t)b * p.N + row;
        if (p.z32_out && (live || p.flag_in)) p.z32_out[o] = z;
        if (p.zt_out) ((st*)p.zt_out)[o] = DT::fromf(z);
      }
    }
  };
  // one tile: ra (and with two chunks rb2) hold it; they are refilled with what follows in the ring
  auto body = [&](int r, u32x4 (&ra)[STEPS], u32x4 (&rb2)[STEPS], float* my_part) {
    typename Mma<DT>::Acc acc[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) acc[g] = Mma<DT>::zero();
    up.multiply(ra, 0, acc);
    if constexpr (CH == 2) {
      issue(r + 1, 0, ra);
      up.multiply(rb2, 1, acc);
      mma_store_partials<DT, NG>(acc, my_part, lane, wave);
      issue(r + 1, 1, rb2);
    } else {
      mma_store_partials<DT, NG>(acc, my_part, lane, wave);
      issue(r + 2, 0, ra);
    }
    __syncthreads();
    if (wave == 0 && r < my_tiles) finish(r, my_part);
  };

  u32x4 u0[STEPS], u1[STEPS];
  issue(0, 0, u0);
  issue(CH == 2 ? 0 : 1, CH == 2 ? 1 : 0, u1);
  // always in pairs (an odd count ends with a tile of dummy loads): a branch around the second body would leave the
  // compiler with a path on which its counted waits for the ring degrade to "wait for everything"
  for (int r = 0; r < my_tiles; r += 2) {
    body(r, u0, CH == 2 ? u1 : u0, part);
    body(r + 1, CH == 2 ? u0 : u1, u1, part + NG * kMmaPartGroup);
  }
  CATS_RSTAMP(7);
}

}  // namespace cats

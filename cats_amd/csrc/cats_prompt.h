// The thresholded MLP over the tokens of a prompt, 16-bit types: two matrix products on the matrix cores, the activation between them
// in the epilogue of the first.
//
//   prompt_kernel<GATE_UP>   z = a * (x . Wup^T),  a = SiLU(x . Wgate^T), 0 where |a| <= t (a NaN is kept, as torch's mask keeps it)
//   prompt_kernel<plain>     y = z . Wdown^T, or its partial sums over ranges of K
//   prompt_sum_kernel        adds those
//
// The sums are fp32 and rounded where torch's separate operations round: gate, a, up, z, y.
//
// A workgroup owns BM tokens times BN weight rows (half of them gate, half up rows of the same neurons, so the epilogue finds both
// sums of a neuron in one lane).  Steps of BK elements of both operands go global memory -> registers -> LDS; the loads of the
// next step are in flight while the matrix cores work on the present one.  In LDS the eight 16-byte pieces of every 128 bytes
// are permuted by the row (piece ^ row % 8): a fragment read takes the same piece of sixteen rows, which this spreads over all banks.
// Rows may start at any element (an odd intermediate size makes the down weight's rows do so): the vectors are read as
// they lie, and only the step in which K ends looks where a vector ends.
//
// What bounds it at 4096 / 11008 in fp16 (medians of kernel traces, and counters): at 32 tokens the weight stream, 42 us for gate and up
// and 18.5 for down (4.3 and 4.9 TB/s); at 512 tokens the barrier of each step and what the waves wait for around it, 94 and 53 us (980
// and 880 TFLOP/s; matrix cores busy 43 and 35 % of the time, LDS 31 %, no bank conflicts).  The chip lowers its clock when
// the matrix cores start: in a program's first 5 ms the same launches take up to 131 us.  Whole call, steady: 153 us at 512
// tokens, 148 against 189 with the library's products and one kernel between them; 68 against 79 at 16; 304 / 569 at 22 tokens 20
// against 78, host time mostly.
// Against 102 and 61 us in the same trace: 110 and 65 with the end of K looked for in every step, 101 and 64 without the dealing of
// the loads between the MFMAs, and that 142 against 130 for the 128 x 128 tile.
// Measured and not taken: four waves with 128 x 96 sums each (155 us), two steps of loads in the registers of the large tiles (no
// change), raised wave priority around the multiplications (no change).
#pragma once
#include <type_traits>

#include "cats_rows_mma.h"

namespace cats {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef u32x4 u32x4_elem __attribute__((aligned(2)));  // a vector at any 16-bit element

struct PromptArgs {
  const void* x;    // (M, ldx) dtype
  const void* w;    // (N, K) dtype, pitch K
  const void* w2;   // GATE_UP: the up weight, w is the gate weight
  void* out;        // (M, ldo) dtype; with splits > 1 the partial sums [splits][M][ldo] fp32
  int M, N, K;
  int ldx, ldo;     // elements; ldo a multiple of 4, GATE_UP: at least N, columns N..ldo-1 are zeroed.  Plain, one split: ldo = N
  int steps;        // K steps of a split
  int splits;
  int mblocks, nblocks;
  float t;
};

// WM x WN waves of FM x FN fragments (16 tokens x 16 weight rows) each, steps of BK elements, AHEAD (1 or an even number) steps of loads in registers.
template <int WM_, int WN_, int FM_, int FN_, int BK_, int AHEAD_>
struct PromptTile {
  static constexpr int WM = WM_, WN = WN_, FM = FM_, FN = FN_, BK = BK_, AHEAD = AHEAD_;
  static_assert(AHEAD == 1 || AHEAD % 2 == 0, "sets and LDS buffers turn together");
  static constexpr int THREADS = WM * WN * kWave, BM = WM * FM * 16, BN = WN * FN * 16;
  static constexpr int P = BK / 8;                 // 16-byte pieces of a row
  static constexpr int STEP = (BM + BN) * P;       // vectors of one LDS buffer
  static constexpr size_t LDS = 2 * (size_t)STEP * sizeof(u32x4);
  static constexpr int PASS = THREADS / P;         // rows that the threads load at a time
  static_assert(BM % PASS == 0 && BN % PASS == 0 && PASS % 8 == 0 && BN % 32 == 0 && BK % 64 == 0, "whole passes");
};

// Asks the scheduler to place RD LDS reads, WR LDS writes and LD loads, in this order, evenly between M MFMAs.
template <int M, int RD, int WR, int LD>
struct PromptDeal {
  static constexpr int N = RD + WR + LD;
  template <int I>
  static __device__ __forceinline__ void go() {
    if constexpr (I < N) {
      __builtin_amdgcn_sched_group_barrier(I < RD ? 0x100 : I < RD + WR ? 0x200 : 0x020, 1, 0);
      constexpr int m = (I + 1) * M / N - I * M / N;
      if constexpr (m > 0) __builtin_amdgcn_sched_group_barrier(0x008, m, 0);
      go<I + 1>();
    }
  }
};

template <class DT, class T, bool GATE_UP>
__global__ __launch_bounds__(T::THREADS) void prompt_kernel(PromptArgs p) {
  typedef typename DT::st st;
  static_assert(sizeof(st) == 2, "16-bit types");
  constexpr int FM = T::FM, FN = T::FN, P = T::P, VA = T::BM / T::PASS, VB = T::BN / T::PASS;
  extern __shared__ u32x4 lds[];  // [2][BM + BN rows][P pieces]

  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / T::WN, wn = wave % T::WN;

  // The blocks of all tokens over the same weights run on one XCD, next to each other: its L2 serves the weights to all but the
  // first.  The ranges of K come next: an XCD keeps to one of them where their number divides eight.
  const int xcd = blockIdx.x & 7, turn = blockIdx.x >> 3;
  const int mb = turn % p.mblocks, g = (turn / p.mblocks) * 8 + xcd;
  if (g >= p.nblocks * p.splits) return;
  const int split = g % p.splits, nblk = g / p.splits;
  const int m0 = mb * T::BM, n0 = nblk * (GATE_UP ? T::BN / 2 : T::BN);
  const int kbegin = split * p.steps * T::BK;
  const int nsteps = min(p.steps, (p.K - kbegin + T::BK - 1) / T::BK);

  // this thread's vectors: piece `piece` of rows tid / P + i * PASS; rows past the end re-read the last one, their sums are dropped
  const int piece = tid % P, row = tid / P;
  // GATE_UP: sixteen gate rows and the sixteen up rows of the same neurons take turns (a wave's rows are all of one kind)
  uint32_t oa[VA], ob[VB];
  const int half16 = __builtin_amdgcn_readfirstlane(row >> 4);
  auto is_up = [&](int i) { return GATE_UP && ((half16 + i * T::PASS / 16) & 1); };
#pragma unroll
  for (int i = 0; i < VA; i++) oa[i] = ((uint32_t)min(m0 + row + i * T::PASS, p.M - 1) * (uint32_t)p.ldx + piece * 8) * 2u;
#pragma unroll
  for (int i = 0; i < VB; i++) {
    const int r = row + i * T::PASS, n = n0 + (GATE_UP ? (r >> 5) * 16 + (r & 15) : r);
    ob[i] = ((uint32_t)min(n, p.N - 1) * (uint32_t)p.K + piece * 8) * 2u;
  }
  // Elements of this thread's vector of a step that lie behind K.  The vector in which K ends is read so that it ends with the row
  // and shifted down before it is stored; those behind it are stored as zeros.
  auto over = [&](int step) { return max(kbegin + step * T::BK + piece * 8 + 8 - p.K, 0); };
  u32x4 ring_a[T::AHEAD][VA], ring_b[T::AHEAD][VB];  // the steps that are stored next
  auto load = [&](int step, u32x4 (&ra)[VA], u32x4 (&rb)[VB]) {
    const uint32_t at = (uint32_t)(kbegin + step * T::BK - over(step)) * 2u;
#pragma unroll
    for (int i = 0; i < VB; i++) rb[i] = *(const u32x4_elem*)((const char*)(is_up(i) ? p.w2 : p.w) + (ob[i] + at));
#pragma unroll
    for (int i = 0; i < VA; i++) ra[i] = *(const u32x4_elem*)((const char*)p.x + (oa[i] + at));
  };
  auto shifted = [](u32x4 v, int s) {  // s elements down, 0 <= s
    const unsigned long long lo = v[0] | (unsigned long long)v[1] << 32, hi = v[2] | (unsigned long long)v[3] << 32;
    const int b = (s & 3) * 16;
    const unsigned long long mid = b ? (lo >> b) | (hi << (64 - b)) : lo;
    const unsigned long long rlo = s >= 8 ? 0ull : s >= 4 ? hi >> b : mid, rhi = s >= 4 ? 0ull : hi >> b;
    return u32x4{(uint32_t)rlo, (uint32_t)(rlo >> 32), (uint32_t)rhi, (uint32_t)(rhi >> 32)};
  };
  const int put = row * P + (piece ^ (row & 7));  // PASS is a multiple of 8: the same permutation for all of a thread's rows
  auto store = [&](int step, int buf, u32x4 (&ra)[VA], u32x4 (&rb)[VB], auto ends) {
    if (ends && kbegin + (step + 1) * T::BK > p.K) {  // uniform
      const int s = over(step);
#pragma unroll
      for (int i = 0; i < VA; i++) ra[i] = shifted(ra[i], s);
#pragma unroll
      for (int i = 0; i < VB; i++) rb[i] = shifted(rb[i], s);
    }
    u32x4* a = lds + buf * T::STEP + put;
#pragma unroll
    for (int i = 0; i < VA; i++) a[i * T::PASS * P] = ra[i];
#pragma unroll
    for (int i = 0; i < VB; i++) a[(T::BM + i * T::PASS) * P] = rb[i];
  };

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int fr = lane & 15, fq = lane >> 4;  // a fragment: row lane % 16, piece lane / 16 of four
  const int arow = (wm * FM * 16 + fr) * P;
  auto brow = [&](int j) {
    const int f = wn * FN + (GATE_UP ? (j < FN / 2 ? 2 * j : 2 * (j - FN / 2) + 1) : j);
    return (T::BM + f * 16 + fr) * P;
  };
  // Two sets of fragments: one is read while the matrix cores work on the other.
  constexpr int KK = T::BK / 32;
  u32x4 fa[2][FM], fb[2][FN];
  auto fetch = [&](int buf, int kk) {
    const u32x4* b = lds + buf * T::STEP;
    const int at = (kk * 4 + fq) ^ (fr & 7);
#pragma unroll
    for (int j = 0; j < FN; j++) fb[kk & 1][j] = b[brow(j) + at];
#pragma unroll
    for (int i = 0; i < FM; i++) fa[kk & 1][i] = b[arow + i * 16 * P + at];
  };
  auto multiply = [&](int set) {
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
      for (int j = 0; j < FN; j++) acc[i][j] = Mma<DT>::run(fb[set][j], fa[set][i], acc[i][j]);
  };
  // One barrier a step, in front of its last multiplication: by then everybody has read this step's buffer to the end (which the next
  // step overwrites) and written the next step's, whose first fragments arrive during that multiplication.  Steps past the
  // last are loaded (the end of the rows again) and stored as well, and not used.  `ends`: K may end in the step that is stored.
  // The LDS and memory instructions are dealt out between the MFMAs: issued in one go they queue, all waves of the CU at once, while
  // the matrix cores wait.
  auto step = [&](int s, int buf, u32x4 (&ra)[VA], u32x4 (&rb)[VB], auto ends) {
    fetch(buf, 1);
    store(s + 1, buf ^ 1, ra, rb, ends);
    // steps past the last: the last one again, which the caches hold
    load(T::AHEAD == 1 ? s + 2 : min(s + 1 + T::AHEAD, nsteps), ra, rb);
    multiply(0);
    if constexpr (KK == 2) PromptDeal<FM * FN, FM + FN, VA + VB, VA + VB>::template go<0>();
#pragma unroll
    for (int kk = 1; kk < KK; kk++) {
      if (kk + 1 < KK) fetch(buf, kk + 1);
      else {
        __builtin_amdgcn_sched_barrier(0);  // the multiplications stay on their sides
        __syncthreads();
        fetch(buf ^ 1, 0);
      }
      multiply(kk & 1);
    }
    if constexpr (KK == 2) PromptDeal<(FM * FN < FM + FN ? FM * FN : FM + FN), FM + FN, 0, 0>::template go<0>();
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int AHEAD = T::AHEAD, TURN = AHEAD == 1 ? 2 : AHEAD;
  load(0, ring_a[0], ring_b[0]);
  store(0, 0, ring_a[0], ring_b[0], std::true_type());
#pragma unroll
  for (int i = 1; i <= AHEAD; i++) load(min(i, nsteps), ring_a[i % AHEAD], ring_b[i % AHEAD]);
  __syncthreads();
  fetch(0, 0);
  const int whole = min(nsteps, (p.K - kbegin) / T::BK);  // steps that K does not end in
  int s = 0;  // the loads of step s + 1 are in set (s + 1) % AHEAD
  for (; s + TURN < whole; s += TURN) {
#pragma unroll
    for (int i = 0; i < TURN; i++) step(s + i, i & 1, ring_a[(i + 1) % AHEAD], ring_b[(i + 1) % AHEAD], std::false_type());
  }
  for (; s < nsteps; s += TURN) {
#pragma unroll
    for (int i = 0; i < TURN; i++)
      if (s + i < nsteps) step(s + i, i & 1, ring_a[(i + 1) % AHEAD], ring_b[(i + 1) % AHEAD], std::true_type());
  }

  // lane: token fr of a fragment, four consecutive weight rows fq * 4 ..
  if (GATE_UP) {
#pragma unroll
    for (int i = 0; i < FM; i++) {
      const int m = m0 + (wm * FM + i) * 16 + fr;
#pragma unroll
      for (int j = 0; j < FN / 2; j++) {
        const int n = n0 + (wn * (FN / 2) + j) * 16 + fq * 4;
        st z[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float gr = DT::rnd(acc[i][j][e]), a = DT::rnd(gr / (1.f + expf(-gr)));
          z[e] = n + e < p.N ? DT::fromf((fabsf(a) <= p.t ? 0.f : a) * DT::rnd(acc[i][FN / 2 + j][e])) : (st)0;
        }
        const u32x2 v = {(uint32_t)z[0] | (uint32_t)z[1] << 16, (uint32_t)z[2] | (uint32_t)z[3] << 16};
        if (m < p.M && n < p.ldo) *(u32x2*)((st*)p.out + (size_t)m * p.ldo + n) = v;
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < FM; i++) {
      const int m = m0 + (wm * FM + i) * 16 + fr;
#pragma unroll
      for (int j = 0; j < FN; j++) {
        const int n = n0 + (wn * FN + j) * 16 + fq * 4;
        if (m >= p.M || n >= p.ldo) continue;
        if (p.splits > 1) {
          *(f32x4*)((float*)p.out + ((size_t)split * p.M + m) * p.ldo + n) = acc[i][j];
        } else {
          st* y = (st*)p.out + (size_t)m * p.ldo + n;
          st v[4];
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = DT::fromf(acc[i][j][e]);
          if ((p.ldo & 3) == 0) *(u32x2*)y = u32x2{(uint32_t)v[0] | (uint32_t)v[1] << 16, (uint32_t)v[2] | (uint32_t)v[3] << 16};
          else
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (n + e < p.ldo) y[e] = v[e];
        }
      }
    }
  }
}

// y = the sum over the splits, in their order.  One thread per four columns.
struct PromptSumArgs {
  const float* partial;  // [splits][M][ldp]
  void* y;               // (M, N)
  int M, N, ldp, splits;
};
template <class DT>
__global__ __launch_bounds__(256) void prompt_sum_kernel(PromptSumArgs p) {
  typedef typename DT::st st;
  const int quads = p.ldp / 4;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)p.M * quads) return;
  const size_t stride = (size_t)p.M * p.ldp;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  for (int g = 0; g < p.splits; g++) s += *(const f32x4*)(p.partial + g * stride + i * 4);
  const int n = (int)(i % quads) * 4;
  st* y = (st*)p.y + (i / quads) * p.N + n;
  st v[4];
#pragma unroll
  for (int e = 0; e < 4; e++) v[e] = DT::fromf(s[e]);
  if ((p.N & 3) == 0) *(u32x2*)y = u32x2{(uint32_t)v[0] | (uint32_t)v[1] << 16, (uint32_t)v[2] | (uint32_t)v[3] << 16};
  else
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (n + e < p.N) y[e] = v[e];
}

// ---- host: which tile, how many ranges of K ----------------------------------------------------------------------------

// us a step takes on a CU that has one workgroup of this tile, and per workgroup on a CU that has several; from whole kernels over
// 4096 / 11008, 4096 / 8000, 2048 / 5461 and 1024 / 2731 at 32 to 512 tokens.
struct PromptShape {
  int BM, BN, BK;
  float alone, shared;
};
// Tiles 0 and 2 have a second instance with two steps of loads in registers, taken where a CU has at most one workgroup and so too
// few bytes in flight, from ten steps on (whole call in us, one / two steps ahead: 2048 / 5461 2 tokens 28.7 / 26.3 and 192 tokens
// 47.6 / 42.8, 4096 / 11008 96 tokens 83.7 / 74.8, 3072 / 8192 192 tokens 68.8 / 62.6, 1536 / 4096 32 tokens 23.2 / 22.2).  With more
// workgroups a CU the registers cost more than they give (4096 / 11008 64 tokens 74.8 / 76.8), and so does the longer start of a short
// range (512 / 1365, four steps, 192 tokens 16.3 / 17.0).  Four steps ahead: slower than two nearly everywhere (32 tokens 69.6 for
// 66.3).  Tile 1 has none: up to 5 % less on weights from HBM, 3 % more on weights that the caches hold.
template <int AHEAD> using PromptTile0 = PromptTile<2, 2, 1, 2, 128, AHEAD>;
typedef PromptTile<2, 2, 2, 2, 128, 1> PromptTile1;
template <int AHEAD> using PromptTile2 = PromptTile<4, 2, 2, 4, 64, AHEAD>;
typedef PromptTile<4, 2, 4, 4, 64, 1> PromptTile3;
typedef PromptTile<4, 2, 4, 6, 64, 1> PromptTile4;
// Half of tile 0: two or three workgroups a CU where tile 0 has one on most and two on some, so the weights come in evenly (4096 / 11008
// 2 tokens: gate and up 3.4 us less, down 1.6; at 32 tokens, where it reads x twice as often, 0.5 and 0.7).  Up to two blocks of tokens
// (at 128 tokens of 512 / 1365 13.9 us without it, 14.5 with), and where it takes more than one round of the CUs only if at most a fifth
// of the places of all its rounds stay empty: 342 workgroups of 2048 / 5461 at 30 tokens, weights in cache, 23.7 us against 22.8.  Whole call at 2, 16 and 32 tokens, before / now: 4096 / 11008 64.2 / 59.6,
// 65.0 / 60.9, 66.5 / 63.7; 1024 / 2731 18.5 / 16.5, 19.0 / 17.0, 19.3 / 17.3.
typedef PromptTile<2, 1, 1, 2, 128, 1> PromptTile5;
constexpr int kPromptTiles = 6;
constexpr PromptShape kPromptShapes[kPromptTiles] = {
    {PromptTile0<1>::BM, PromptTile0<1>::BN, PromptTile0<1>::BK, 0.8f, 0.55f}, {PromptTile1::BM, PromptTile1::BN, PromptTile1::BK, 0.9f, 0.65f},
    {PromptTile2<1>::BM, PromptTile2<1>::BN, PromptTile2<1>::BK, 0.7f, 0.65f}, {PromptTile3::BM, PromptTile3::BN, PromptTile3::BK, 1.1f, 1.1f},
    {PromptTile4::BM, PromptTile4::BN, PromptTile4::BK, 1.45f, 1.45f},
    {PromptTile5::BM, PromptTile5::BN, PromptTile5::BK, 0.6f, 0.33f}};

struct PromptPlan {
  int tile, mblocks, nblocks, steps, splits;
};
// The cheapest by  steps * max(alone, workgroups per CU * shared), and for ranges of K the launch that adds them and the traffic of
// their sums (written and read at about 4 TB/s).  The model's choice was within 10 % of the fastest measured tile and split, and mostly it.
inline PromptPlan prompt_plan(bool gate_up, int M, int N, int K, int cus) {
  PromptPlan best = {0, 0, 0, 0, 0};
  double best_us = 0;
  for (int t = 0; t < kPromptTiles; t++) {
    const PromptShape& h = kPromptShapes[t];
    const int bn = gate_up ? h.BN / 2 : h.BN, ksteps = (K + h.BK - 1) / h.BK;
    const int mblocks = (M + h.BM - 1) / h.BM, nblocks = (N + bn - 1) / bn;
    if (h.BN == PromptTile5::BN && mblocks > 2) continue;
    for (int want = 1; want <= (gate_up ? 1 : 8); want++) {
      const int steps = (ksteps + want - 1) / want, splits = (ksteps + steps - 1) / steps;
      const long long groups = (long long)mblocks * nblocks * splits, rounds = (groups + cus - 1) / cus;
      if (h.BN == PromptTile5::BN && rounds > 1 && 4 * rounds * cus > 5 * groups) continue;  // see there
      const double per_cu = rounds * (double)h.shared;
      const double us = steps * (per_cu > h.alone ? per_cu : h.alone) + (splits > 1 ? 2.5 + 8e-6 * splits * M * N / 4 : 0.);
      if (best.splits == 0 || us < best_us) {
        best_us = us;
        best = {t, mblocks, nblocks, steps, splits};
      }
    }
  }
  return best;
}
// Steps of loads in registers: two in the second instances of tiles 0 and 2, see there.
inline int prompt_steps_ahead(const PromptPlan& p, int cus) {
  return (p.tile == 0 || p.tile == 2) && p.steps >= 10 && (long long)p.mblocks * p.nblocks * p.splits <= cus ? 2 : 1;
}
inline int prompt_pitch(int I) { return (I + 7) / 8 * 8; }   // of z
inline int prompt_sum_pitch(int H) { return (H + 3) / 4 * 4; }  // of partial sums

}  // namespace cats

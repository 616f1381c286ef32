// The projections of a decode step (cats_decode.h) for 3..8 batch rows of a 16-bit type, on the matrix cores.
//
// proj_kernel spends 4 * B dot instructions a weight vector and stages all rows of x in every workgroup of sixteen weight rows: at four
// rows it reaches 4.1 TB/s on an output head of 32000 x 2048 and 1.9 on the three matrices of 2048 x 2048.  This kernel, traced in steps of four rows: 24.1 us
// (5.4 TB/s) and 9.4 (2.7), at 4096 42.0 (6.2) and 20.9 (4.8).  It reads what it must (131.3 of 131.1 MB, 25.5 of 25.2); LDS is busy a tenth of the time and the
// matrix cores 4 %, so the weight stream and, at 2048, the trips in front of it are the bound.  The tiles, operands
// and the split of K over eight waves are rows_mma_kernel's, one workgroup a CU owns consecutive tiles, and x is staged (and
// normed) once a CU.  TILES tiles are multiplied a round, so that a round is some eight loads a wave whatever the row length, two rounds of loads are in
// flight, and their sums are added by as many waves side by side.
// kProjQkv: a tile is four pairs of the elements that the rotary embedding mixes, d .. d + 3 and the same + head_dim / 2; what it needs
// of the tables lies in LDS, asked for behind the first round's weights (in finish it would wait for the weights in flight).
#pragma once
#include "cats_decode.h"
#include "cats_rows_mma.h"

namespace cats {

constexpr int proj_mma_tiles(int steps, int ch) { return ch == 2 || steps > 4 ? 1 : steps > 2 ? 2 : steps == 2 ? 4 : 8; }
constexpr int kProjMaxHeadDim = 256;  // 32 lanes of 8 elements a cache slot, the most that attention takes

// The three matrices as one list of rows, in tiles of eight; a.r as rows_mma_split takes it.
inline int proj_mma_ntiles(const ProjArgs& a, int mode) { return mode == kProjQkv ? 3 * (a.r.N / 8) : (a.r.N + 7) / 8; }
// dynamic LDS: x operands | two rounds of partial sums | cos and sin of the position
inline size_t proj_mma_lds_bytes(const MmaSplit& sp) {
  return (size_t)sp.slots * kWave * sizeof(u32x4) + 2u * proj_mma_tiles(sp.steps, sp.chunks) * kMmaPartGroup * sizeof(float) + 2u * kProjMaxHeadDim * sizeof(float);
}

template <class DT, int STEPS, int CH, int MODE>
__global__ __launch_bounds__(kMmaThreads) void proj_mma_kernel(ProjArgs a) {
  typedef typename DT::st st;
  typedef MmaRows<DT, STEPS, CH, 1> Rows;
  static_assert(sizeof(st) == 2, "16-bit types only");
  constexpr int TILES = proj_mma_tiles(STEPS, CH);
  const RowsArgs& p = a.r;
  extern __shared__ u32x4 xs[];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xgroup = p.mma_slots * kWave;
  float* part = (float*)(xs + xgroup);                  // [2][TILES][kMmaPartGroup]
  float* s_cs = part + 2 * TILES * kMmaPartGroup;       // [cos, sin][head_dim]

  const int per_matrix = MODE == kProjQkv ? p.N / 8 : (p.N + 7) / 8, ntiles = MODE == kProjQkv ? 3 * per_matrix : per_matrix;
  const int first = blockIdx.x * p.rows_per, my_tiles = min(p.rows_per, ntiles - first);  // rows_per: tiles of a workgroup
  const int jl = lane & 7;
  const Rows rows(p.w, 0, p.row_vecs, xs, xgroup, 0, lane, wave);
  // Row j of tile t of its matrix
  auto row_of = [&](int t, int j) {
    if (MODE != kProjQkv) return t * 8 + j;
    const int i = t * 4, head = i / a.half;  // four pairs of one head: half is a multiple of four
    return head * 2 * a.half + (i - head * a.half) + (j & 3) + (j >> 2) * a.half;
  };
  auto which_of = [&](int tile) { return MODE == kProjQkv ? tile / per_matrix : 0; };
  auto issue = [&](int round, int t, int c, u32x4 (&dst)[STEPS]) {
    const int it = round * TILES + t;
    const bool on = it < my_tiles;  // uniform
    const int tile = on ? first + it : 0, which = which_of(tile), row = row_of(tile - which * per_matrix, jl);
    Rows m = rows;
    m.w = which == 1 ? a.wk : which == 2 ? a.wv : p.w;
    m.issue(row, on && (MODE == kProjQkv || row < p.N), c, dst);
  };

  long long pos = 0;
  if (MODE == kProjQkv) pos = *a.pos;
  const bool pos_ok = pos >= 0 && pos < (long long)a.max_len;
  u32x4 w0[TILES][STEPS], w1[TILES][STEPS];
  {
    MmaX<STEPS * CH, 1> x;
    x.tid = tid;
    x.front = 0;
    x.fetch(p);
    u32x4 nw[STEPS * CH];
    if (p.norm_w) x.fetch_norm(p, nw);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < TILES; t++) issue(0, t, 0, w0[t]);
    __builtin_amdgcn_sched_barrier(0);
    x.mask(p);
    if (p.norm_w) x.template norm<DT>(p, nw, part);
    x.store(xs, xgroup);
  }
  float cs[2] = {0.f, 0.f};
  const int hd = 2 * a.half;
  if (MODE == kProjQkv && tid < hd) {
    const size_t o = (size_t)(pos_ok ? pos : 0) * hd + tid;
    cs[0] = DT::tof(((const st*)a.cos_t)[o]);
    cs[1] = DT::tof(((const st*)a.sin_t)[o]);
  }
  lds_barrier();
#pragma unroll
  for (int t = 0; t < TILES; t++) issue(CH == 2 ? 0 : 1, t, CH == 2 ? 1 : 0, w1[t]);
  if (MODE == kProjQkv && tid < hd) {
    s_cs[tid] = cs[0];
    s_cs[hd + tid] = cs[1];
  }

  // one thread per (row rj of the tile, batch row rb)
  const int rj = lane >> 3, rb = lane & 7;
  auto finish = [&](int it, const float* sums, float res) {
    const int tile = first + it, which = which_of(tile), row = row_of(tile - which * per_matrix, rj);
    float u = mma_reduce<DT>(sums, 0, rj, rb);
    if (MODE == kProjQkv) {
      if (which < 2) {  // uniform
        const float other = __shfl_xor(u, 32, kWave);  // rj ^ 4
        const int d = row % hd;
        u = rj < 4 ? u * s_cs[d] - other * s_cs[hd + d] : u * s_cs[d] + other * s_cs[hd + d];
      }
      if (rb < p.nb) {
        if (which == 0) a.q_out[(size_t)rb * p.N + row] = u;
        else if (pos_ok) ((st*)(which == 1 ? a.k_cache : a.v_cache))[(((size_t)rb * a.heads + row / hd) * a.max_len + (size_t)pos) * hd + row % hd] = DT::fromf(u);
      }
    } else if (rb < p.nb && row < p.N) {
      ((st*)p.zt_out)[(size_t)rb * p.N + row] = DT::fromf(MODE == kProjAdd ? u + res : u);
    }
  };
  auto body = [&](int round, u32x4 (&wa)[TILES][STEPS], u32x4 (&wb)[TILES][STEPS], float* sums) {
    const int it = round * TILES + wave;  // the tile this wave will finish
    float res = 0.f;
    if (MODE == kProjAdd && wave < TILES && it < my_tiles) {
      const int row = row_of(first + it, rj);
      if (rb < p.nb && row < p.N) res = DT::tof(((const st*)a.residual)[(size_t)rb * p.N + row]);
    }
#pragma unroll
    for (int t = 0; t < TILES; t++) {
      typename Mma<DT>::Acc acc[1] = {Mma<DT>::zero()};
      rows.multiply(wa[t], 0, acc);
      if constexpr (CH == 2) {
        issue(round + 1, t, 0, wa[t]);
        rows.multiply(wb[t], 1, acc);
        mma_store_partials<DT, 1>(acc, sums + t * kMmaPartGroup, lane, wave);
        issue(round + 1, t, 1, wb[t]);
      } else {
        mma_store_partials<DT, 1>(acc, sums + t * kMmaPartGroup, lane, wave);
        issue(round + 2, t, 0, wa[t]);
      }
    }
    lds_barrier();
    if (wave < TILES && it < my_tiles) finish(it, sums + wave * kMmaPartGroup, res);
  };
  // in pairs, an odd count ends with dummy loads (see rows_mma_up_kernel).  The sums of a round are added while the next one is multiplied
  // into the other half; the barrier after that lies between them and the round that writes this half again.
  const int rounds = (my_tiles + TILES - 1) / TILES;
  for (int r = 0; r < rounds; r += 2) {
    body(r, w0, CH == 2 ? w1 : w0, part);
    body(r + 1, CH == 2 ? w0 : w1, w1, part + TILES * kMmaPartGroup);
  }
}

}  // namespace cats

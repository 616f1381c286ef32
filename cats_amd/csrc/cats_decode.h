// The rest of a decoder layer around the MLP, for one new token per batch row:
//
//   proj_kernel<kProjQkv>      q, k, v = x . W{q,k,v}^T, rotary embedding on q and k, k and v into the cache      (one launch)
//   attn_decode_kernel         softmax(q . K^T / sqrt(d)) . V over the cache slots 0..position, per batch row and head
//   proj_kernel<kProjAdd>      out = residual + x . W^T                                              (the output projection)
//   proj_kernel<kProjPlain>    out = x . W^T                                                         (the output head)
//
// x may be given before its RMS norm (norm_w), which is then applied while x is staged.  Everything between the weight
// matrices stays in fp32 and is rounded once where it is stored.  All of it is bound by the weight stream: one wave owns two to eight
// rows of a matrix, whose loads are all in flight at once, as in rows_kernel.
// One step of four layers 4096 / 11008, 32 heads, 32000 words, 256 tokens in the cache, fp16, one row: 309 us, of which the MLP
// kernels take 148; with torch's operations in place of these kernels (about 25 launches a layer) it was 761.  Kernel trace: q, k, v
// 17.4 us with the norm (5.8 TB/s), attention 8.1 and the output projection, whose weights it has had fetched, 4.7 (8.1
// without that), output head 40.7 (6.4 TB/s).  With x staged behind the weights: 18.8, 7.6, 5.2 and 42.7.
#pragma once
#include "cats_rows.h"

namespace cats {

enum ProjMode { kProjPlain = 0, kProjAdd = 1, kProjQkv = 2 };

struct ProjArgs {
  RowsArgs r;            // x, w, K, N, nb, nch, row_vecs, norm_w, norm_eps; zt_out is the output of kProjPlain / kProjAdd
  const void* residual;  // kProjAdd: (nb, N) dtype
  // kProjQkv (w is Wq; N = heads * head_dim rows of each of the three matrices)
  const u32x4* wk;
  const u32x4* wv;
  float* q_out;          // (nb, N) fp32, rotated
  void* k_cache;         // (nb, heads, max_len, head_dim) dtype
  void* v_cache;
  const void* cos_t;     // (max_len, head_dim) dtype
  const void* sin_t;
  const int64_t* pos;    // one position for all batch rows; outside [0, max_len) nothing is stored
  int half;              // head_dim / 2
  int heads;
  int max_len;
};

// R rows per wave.  For kProjQkv they are two, the elements of a head that the rotary embedding mixes, d and d + head_dim / 2,
// so it is applied to the two sums where they are; the wave's number counts these pairs over the three matrices.
// Short rows are taken by blocks of CB = 2 or 4 chunks of 64 vectors instead of eight, and where the result is stored as it is (the output head) by
// 16 / CB rows a wave: as many loads in flight, and x is staged once for as many weight bytes.
template <class DT, int B, int CB, int R, bool FULL, int MODE, int WAVES>
__global__ __launch_bounds__(WAVES* kWave) __attribute__((amdgpu_waves_per_eu(rows_waves_per_simd(B, FULL), 8)))
void proj_kernel(ProjArgs a) {
  typedef typename DT::st st;
  static_assert(MODE != kProjQkv || R == 2, "a pair of elements a wave");
  const RowsArgs& p = a.r;
  extern __shared__ u32x4 xs[];  // [B][round_up(nch, CB) * 64] vectors
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  const int item = blockIdx.x * WAVES + wave;
  int row[R];
  bool on[R];
  const u32x4* w = p.w;
  int which = 0, d = 0;
  long long pos = 0;
  if (MODE == kProjQkv) {
    const int pairs = p.N / 2;
    which = item / pairs;
    const int i = item - which * pairs;
    const int head = i / a.half;
    d = i - head * a.half;
    on[0] = on[1] = which < 3;
    row[0] = on[0] ? head * 2 * a.half + d : 0;
    row[1] = on[0] ? row[0] + a.half : 0;
    w = which == 1 ? a.wk : which == 2 ? a.wv : p.w;
    pos = *a.pos;
  } else {
#pragma unroll
    for (int r = 0; r < R; r++) {
      on[r] = item * R + r < p.N;
      row[r] = on[r] ? item * R + r : p.N - 1;
    }
  }
  const bool pos_ok = pos >= 0 && pos < (long long)a.max_len;

  // What the sums will be joined with is asked for first, and the elements of the rotary embedding behind the weights: after the sums each
  // would be one more trip.  The weights go out behind x, before x is waited for; at one and two rows half of them when x is staged: its registers.
  float res[R][B];
  if (MODE == kProjAdd) {
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int b = 0; b < B; b++) res[r][b] = DT::tof(((const st*)a.residual)[(size_t)min(b, p.nb - 1) * p.N + row[r]]);
  }
  constexpr int kXPreAll = (B * CB + WAVES - 1) / WAVES, kXPre = kXPreAll < 4 ? kXPreAll : 4;  // rows of CB chunks
  constexpr int kFirst = B <= 2 ? R * CB / 2 : R * CB;
  u32x4 wv[R][CB];
  __shared__ float s_sq[kStagedMaxChunks + B];
  RowsX<DT, B, WAVES, kXPre, MODE != kProjAdd ? kNormAhead : kNormLater> x;
  x.lane = lane;
  x.wave = wave;
  x.nchp = (p.nch + CB - 1) / CB * CB;
  x.fetch(p);
  __builtin_amdgcn_sched_barrier(0);
  rows_issue_all<0, kFirst, R, CB, FULL>(w, row, 0, p, lane, wv);
  __builtin_amdgcn_sched_barrier(0);
  x.store(p, xs, s_sq);
  rows_issue_all<kFirst, R * CB, R, CB, FULL>(w, row, 0, p, lane, wv);
  float cs = 0.f;  // lane 0: cos of d, 1: of d + half, 2 and 3: sin
  if (MODE == kProjQkv) {
    const st* t = (const st*)(lane & 2 ? a.sin_t : a.cos_t);
    cs = DT::tof(t[(size_t)(pos_ok ? pos : 0) * 2 * a.half + d + (lane & 1) * a.half]);
  }

  float g[R][B];
  rows_dot<DT, B, R, CB, FULL, true, true>(w, row, on, xs, p.x, p, lane, wv, g);

  auto cs_of = [&](int i) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cs), i)); };
  const float c0 = cs_of(0), c1 = cs_of(1), s0 = cs_of(2), s1 = cs_of(3);
  if (lane != 0) return;
  if (MODE == kProjQkv) {
    if (!on[0]) return;
    if (which == 0 || which == 1) {
#pragma unroll
      for (int b = 0; b < B; b++) {
        const float lo = g[0][b], hi = g[1][b];
        g[0][b] = lo * c0 - hi * s0;
        g[1][b] = hi * c1 + lo * s1;
      }
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int b = 0; b < B; b++)
        if (b < p.nb) {
          if (which == 0) a.q_out[(size_t)b * p.N + row[r]] = g[r][b];
          else if (pos_ok) {
            const int head = row[r] / (2 * a.half), e = row[r] - head * 2 * a.half;
            st* cache = (st*)(which == 1 ? a.k_cache : a.v_cache);
            cache[(((size_t)b * a.heads + head) * a.max_len + (size_t)pos) * 2 * a.half + e] = DT::fromf(g[r][b]);
          }
        }
  } else {
    st* out = (st*)p.zt_out;
#pragma unroll
    for (int r = 0; r < R; r++)
      if (on[r]) {
#pragma unroll
        for (int b = 0; b < B; b++)
          if (b < p.nb) {
            const size_t o = (size_t)b * p.N + row[r];
            out[o] = DT::fromf(MODE == kProjAdd ? g[r][b] + res[r][b] : g[r][b]);
          }
      }
  }
}

struct AttnArgs {
  const float* q;        // (nb, heads * head_dim) fp32
  const u32x4* k;        // (nb, heads, max_len, head_dim) dtype
  const u32x4* v;
  const int64_t* pos;    // slots 0..pos take part; outside [0, max_len) the output is NaN
  void* out;             // (nb, heads * head_dim) dtype
  float scale;           // log2(e) / sqrt(head_dim)
  int max_len;
  int pairs;             // batch rows x heads: the workgroups that attend; those behind them fetch `next` ahead
  const u32x4* next;     // weights of the projection that follows, in pieces of one of its workgroups each
  unsigned next_vecs;    // less than 2^28
  int piece_vecs;
};

// The projection that follows depends on this launch, and attention leaves most CUs and the memory idle.  So the workgroups behind the
// attending ones read its weights into the caches: the pieces that an XCD's workgroups will ask for on this XCD (workgroups go
// round the eight XCDs in both launches).  They start about 2 us late, when the cache slots have been asked for: at once they hold
// those up (attention 10.1 us for 6.6), and as much is fetched as comes in meanwhile.  Step of four layers as above, both timed in turn:
// 327.0 us without, 324.7 with.  Beside each other in one run: 24 MiB 320.6, 32 MiB 322 to 325, 16 MiB 322.1; started at once 325 to 335.
// Nothing is fetched where the cache slots and the weights together exceed the L2s (eight of 4 MiB): attention then needs the memory
// itself and its slots take the weights' place.  Steps of two layers 4096 / 11008, one row, without, with, with this limit, in us: 256
// slots 160.6, 156.5, 156.3;  480 160.9, 158.7, 159.1;  1000 168.2, 171.3, 168.4;  2000 186, 194, 187;  two rows at 480 198.9, 200.9,
// 199.2; one row of 16 heads and 2048 / 5461 (8 MiB of weights) at 2000 slots 111.3, 109.8, 109.7.
constexpr unsigned kAttnAheadVecs = (24u << 20) / 16;
constexpr long long kL2Vecs = (32 << 20) / 16;
constexpr int kAttnAheadSleeps = 5;  // of 1024 clocks each
template <int LPS>
__device__ __forceinline__ void attn_fetch_next(const AttnArgs& p) {
  constexpr int kLoads = 10;  // in flight per thread
  const unsigned xcd = blockIdx.x & 7, groups = (gridDim.x - p.pairs) / 8;  // workgroups on this XCD
  const unsigned piece = p.piece_vecs, first = (blockIdx.x - p.pairs) / 8 * 1024 + threadIdx.x;
  const long long pos = *p.pos;
  for (int i = 0; i < kAttnAheadSleeps; i++) __builtin_amdgcn_s_sleep(16);
  if (pos < 0 || pos >= (long long)p.max_len || 2 * LPS * (long long)p.pairs * (pos + 1) + p.next_vecs > kL2Vecs) return;
  const unsigned pieces = (p.next_vecs + piece - 1) / piece, mine = ((pieces + 7 - xcd) / 8) * piece;  // vectors for this XCD
  for (unsigned t = first; t < mine; t += kLoads * groups * 1024) {
    u32x4 w[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
      const unsigned at = min(t + i * groups * 1024, mine - 1), n = at / piece;
      w[i] = p.next[min((xcd + 8 * n) * piece + (at - n * piece), p.next_vecs - 1)];
    }
#pragma unroll
    for (int i = 0; i < kLoads; i++) asm volatile("" ::"v"(w[i]));
  }
}

// One workgroup of sixteen waves per (batch row, head).  A slot's head_dim elements sit in LPS lanes of one 16-byte vector
// each, so a wave holds 64 / LPS slots side by side and the workgroup 16 * 64 / LPS; every lane group runs its own online
// softmax over the slots it meets, U slots a turn with the loads of K and V of all of them in flight together (256 slots of 128
// 16-bit elements are one turn), and the groups' results are merged at the end, in a fixed order.  What bounds it is dependent
// memory trips, not the bytes (131 KiB a head at 256 slots): so (AHEAD) the first turn's slots are asked for with the position, whatever
// it is (slots behind it hold anything and are masked), and the next turn's before this one's are used.  Where the heads fill more than
// a quarter of the chip the slots behind the position cost more than the trip (steps of two layers 4096 / 11008, 4 rows of 32 heads at 60 slots
// 230.7 us with, 228.6 without).  The last turn asks for nothing: its registers would be waited for (one row at 480 slots 159.1 us, so
// 156.7; 4 rows of 16 heads, 2048 / 5461, 132.8, 130.4).
template <class DT, int LPS, bool AHEAD>
__global__ __launch_bounds__(1024) void attn_decode_kernel(AttnArgs p) {
  typedef typename DT::st st;
  constexpr int VEC = DT::VEC, HD = LPS * VEC, G = kWave / LPS, WAVES = 16, S = WAVES * G, U = 4;
  __shared__ float s_acc[WAVES][HD];
  __shared__ float s_m[WAVES], s_l[WAVES];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  const int sub = lane % LPS;
  const int slot0 = wave * G + lane / LPS;
  if ((int)blockIdx.x >= p.pairs) return attn_fetch_next<LPS>(p);
  const u32x4* kb = p.k + (size_t)blockIdx.x * p.max_len * LPS + sub;
  const u32x4* vb = p.v + (size_t)blockIdx.x * p.max_len * LPS + sub;
  const long long pos = *p.pos;
  float q[VEC];
#pragma unroll
  for (int e = 0; e < VEC; e++) q[e] = p.q[(size_t)blockIdx.x * HD + sub * VEC + e] * p.scale;

  auto elem = [](u32x4 x, int e) {
    if constexpr (sizeof(st) == 4) return __uint_as_float(x[e]);
    else return DT::tof((st)(x[e / 2] >> (16 * (e & 1))));
  };
  u32x4 kv[U], vv[U], kn[U], vn[U];
  auto fetch = [&](int s0, int last, u32x4 (&k)[U], u32x4 (&v)[U]) {
#pragma unroll
    for (int u = 0; u < U; u++) k[u] = kb[(size_t)min(s0 + u * S + slot0, last) * LPS];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = vb[(size_t)min(s0 + u * S + slot0, last) * LPS];
  };
  if constexpr (AHEAD) fetch(0, p.max_len - 1, kv, vv);
  const int n = pos >= 0 && pos < (long long)p.max_len ? (int)pos + 1 : 0;
  float m = -INFINITY, l = 0.f, acc[VEC];
#pragma unroll
  for (int e = 0; e < VEC; e++) acc[e] = 0.f;
  auto turn = [&](int s0) {
    float sc[U], mu = m;
#pragma unroll
    for (int u = 0; u < U; u++) {
      float t = 0.f;
#pragma unroll
      for (int e = 0; e < VEC; e++) t = fmaf(q[e], elem(kv[u], e), t);
#pragma unroll
      for (int o = 1; o < LPS; o <<= 1) t += __shfl_xor(t, o, kWave);
      sc[u] = s0 + u * S + slot0 < n ? t : -INFINITY;
      mu = fmaxf(mu, sc[u]);
    }
    const float base = mu == -INFINITY ? 0.f : mu;  // a group that has met no slot yet keeps zeros
    const float keep = exp2f(m - base);
    l *= keep;
#pragma unroll
    for (int e = 0; e < VEC; e++) acc[e] *= keep;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const bool in = s0 + u * S + slot0 < n;
      const float pr = exp2f(sc[u] - base);
      l += in ? pr : 0.f;
#pragma unroll
      for (int e = 0; e < VEC; e++) acc[e] = in ? fmaf(pr, elem(vv[u], e), acc[e]) : acc[e];
    }
    m = mu;
  };
  if constexpr (AHEAD) {
    int s0 = 0;
    for (; s0 + S * U < n; s0 += S * U) {
      fetch(s0 + S * U, n - 1, kn, vn);
      turn(s0);
#pragma unroll
      for (int u = 0; u < U; u++) {
        kv[u] = kn[u];
        vv[u] = vn[u];
      }
    }
    if (n > 0) turn(s0);
  } else {
    for (int s0 = 0; s0 < n; s0 += S * U) {
      fetch(s0, n - 1, kv, vv);
      turn(s0);
    }
  }
  // the wave's groups, then the waves
  float mw = m;
#pragma unroll
  for (int o = LPS; o < kWave; o <<= 1) mw = fmaxf(mw, __shfl_xor(mw, o, kWave));
  const float f = exp2f(m - (mw == -INFINITY ? 0.f : mw));
  l *= f;
#pragma unroll
  for (int o = LPS; o < kWave; o <<= 1) l += __shfl_xor(l, o, kWave);
#pragma unroll
  for (int e = 0; e < VEC; e++) {
    acc[e] *= f;
#pragma unroll
    for (int o = LPS; o < kWave; o <<= 1) acc[e] += __shfl_xor(acc[e], o, kWave);
  }
  if (lane < LPS) {
#pragma unroll
    for (int e = 0; e < VEC; e++) s_acc[wave][sub * VEC + e] = acc[e];
    if (lane == 0) { s_m[wave] = mw; s_l[wave] = l; }
  }
  __syncthreads();
  for (int c = threadIdx.x; c < HD; c += WAVES * kWave) {
    float mt = -INFINITY;
#pragma unroll
    for (int i = 0; i < WAVES; i++) mt = fmaxf(mt, s_m[i]);
    const float base = mt == -INFINITY ? 0.f : mt;
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES; i++) {
      const float e = exp2f(s_m[i] - base);
      num = fmaf(e, s_acc[i][c], num);
      den = fmaf(e, s_l[i], den);
    }
    ((st*)p.out)[(size_t)blockIdx.x * HD + c] = DT::fromf(num / den);
  }
}

// Between the matrix products of a prompt:  z = a * u with a = SiLU(g), 0 where |a| <= t (a NaN is kept, as torch's mask keeps it),
// rounded where torch's separate operations round.  One pass over the three arrays; as silu, abs, compare, masked fill and multiply
// they were eleven: 512 x 11008 in 16 bits took 32 us.
struct SiluMaskMulArgs {
  const void* g;
  const void* u;
  void* z;
  size_t n;
  float t;
};
template <class DT>
__global__ __launch_bounds__(256) void silu_mask_mul_kernel(SiluMaskMulArgs p) {
  typedef typename DT::st st;
  constexpr int VEC = DT::VEC;
  auto one = [&](st g, st u) {
    const float gf = DT::tof(g), a = DT::rnd(gf / (1.f + expf(-gf)));
    return DT::fromf((fabsf(a) <= p.t ? 0.f : a) * DT::tof(u));
  };
  const size_t nv = p.n / VEC, i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < nv) {
    u32x4 gv = ((const u32x4*)p.g)[i], uv = ((const u32x4*)p.u)[i], zv;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const uint32_t gw = gv[w], uw = uv[w];
      if constexpr (sizeof(st) == 4) zv[w] = __float_as_uint(one(__uint_as_float(gw), __uint_as_float(uw)));
      else zv[w] = (uint32_t)one((st)gw, (st)uw) | ((uint32_t)one((st)(gw >> 16), (st)(uw >> 16)) << 16);
    }
    ((u32x4*)p.z)[i] = zv;
  } else if (i == nv) {
    for (size_t j = nv * VEC; j < p.n; j++) ((st*)p.z)[j] = one(((const st*)p.g)[j], ((const st*)p.u)[j]);
  }
}

}  // namespace cats

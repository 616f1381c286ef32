// C ABI of the CATS sparse-MLP decode kernels (declared in include/cats_gemv.h): argument checks,
// workspace carving, launch-shape selection and dispatch on dtype.  No allocation, no synchronisation
// (cats_read_count excepted), everything on the caller's stream.
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>

#include <mutex>
#include <unordered_map>

#include "cats_gemv.h"
#include "cats_launch.h"

// Built-in scratch of cats_mlp_noalloc: the per-workgroup partial sums and active counts of the single-pass kernel and of small layers'.
// Every GPU the library runs on holds its own copy of this array, at its own address, until the process ends.
constexpr size_t kScratchPartialBytes = (size_t)256 * 8192 * 4;  // 256 workgroups x (B * H <= 8192) fp32 partial sums
constexpr size_t kScratchCountBytes = 4096;                      // one int32 count per workgroup
constexpr size_t kScratchPoolBytes = 4096;                       // neuron-pool counters of 32 workgroup groups
constexpr size_t kScratchBytes = kScratchPartialBytes + kScratchCountBytes + kScratchPoolBytes;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace cats {

// Per-dtype launchers live in cats_inst.hip.
template <> hipError_t launch_rows<F16>(int, int, const RowsArgs&, hipStream_t);
template <> hipError_t launch_rows<BF16>(int, int, const RowsArgs&, hipStream_t);
template <> hipError_t launch_rows<F32>(int, int, const RowsArgs&, hipStream_t);
template <> hipError_t launch_down<F16>(int, bool, const DownArgs&, int, hipStream_t);
template <> hipError_t launch_down<BF16>(int, bool, const DownArgs&, int, hipStream_t);
template <> hipError_t launch_down<F32>(int, bool, const DownArgs&, int, hipStream_t);
template <> hipError_t launch_fused<F16>(int, int, int, const FusedArgs&, const ReduceArgs&, hipStream_t);
template <> hipError_t launch_fused<BF16>(int, int, int, const FusedArgs&, const ReduceArgs&, hipStream_t);
template <> hipError_t launch_fused<F32>(int, int, int, const FusedArgs&, const ReduceArgs&, hipStream_t);
template <> hipError_t launch_proj<F16>(int, int, const ProjArgs&, hipStream_t);
template <> hipError_t launch_proj<BF16>(int, int, const ProjArgs&, hipStream_t);
template <> hipError_t launch_proj<F32>(int, int, const ProjArgs&, hipStream_t);
template <> hipError_t launch_attn<F16>(int, int, AttnArgs, hipStream_t);
template <> hipError_t launch_attn<BF16>(int, int, AttnArgs, hipStream_t);
template <> hipError_t launch_attn<F32>(int, int, AttnArgs, hipStream_t);
template <> hipError_t launch_gate_cols<F16>(const GateColsArgs&, int, hipStream_t);
template <> hipError_t launch_gate_cols<BF16>(const GateColsArgs&, int, hipStream_t);
template <> hipError_t launch_gate_cols<F32>(const GateColsArgs&, int, hipStream_t);
template <> hipError_t launch_gate_cols_finish<F16>(const GateColsArgs&, int, void*, hipStream_t);
template <> hipError_t launch_gate_cols_finish<BF16>(const GateColsArgs&, int, void*, hipStream_t);
template <> hipError_t launch_gate_cols_finish<F32>(const GateColsArgs&, int, void*, hipStream_t);
template <> hipError_t launch_silu_mask_mul<F16>(const SiluMaskMulArgs&, hipStream_t);
template <> hipError_t launch_silu_mask_mul<BF16>(const SiluMaskMulArgs&, hipStream_t);
template <> hipError_t launch_silu_mask_mul<F32>(const SiluMaskMulArgs&, hipStream_t);
template <> hipError_t launch_prompt<F16>(bool, const PromptPlan&, PromptArgs, hipStream_t);
template <> hipError_t launch_prompt<BF16>(bool, const PromptPlan&, PromptArgs, hipStream_t);
template <> hipError_t launch_prompt_sum<F16>(const PromptSumArgs&, hipStream_t);
template <> hipError_t launch_prompt_sum<BF16>(const PromptSumArgs&, hipStream_t);
hipError_t ensure_dynamic_lds(const void* kern, size_t bytes) {
  if (bytes <= 48 * 1024) return hipSuccess;
  static std::mutex mu;
  static std::unordered_map<uintptr_t, size_t> granted;  // (kernel, device) -> bytes; the attribute is per device
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
  const uintptr_t key = (uintptr_t)kern * 64u + (uintptr_t)dev;
  std::lock_guard<std::mutex> lock(mu);
  auto it = granted.find(key);
  if (it != granted.end() && it->second >= bytes) return hipSuccess;
  hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e == hipSuccess) granted[key] = bytes;
  return e;
}

int current_device_cus() {
  constexpr int kDevs = 64;
  static int cus[kDevs];  // 0 = not asked yet; written once per device with the same value, so a plain atomic will do
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kDevs) return 256;
  int n = __atomic_load_n(&cus[dev], __ATOMIC_RELAXED);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    __atomic_store_n(&cus[dev], n, __ATOMIC_RELAXED);
  }
  return n;
}

namespace {

Tuning g_tuning = {0, 0, 0, 0};
#ifdef CATS_TIMING
long long* g_tbuf_rows = nullptr;
long long* g_tbuf_down = nullptr;
long long* g_tbuf_fused = nullptr;
#endif

constexpr int kMaxSlabs = 128;
constexpr int kKernelBatch = 8;  // rows one launch handles; the entry points take up to CATS_MAX_BATCH rows in passes of this many
// Head of the workspace.  [0, 4096): the neuron-pool counters of the single-pass kernel (one 128-byte line per group of
// workgroups; pool builds only).  then the arrival counters of the reduction launch that also writes the next norm
// (144 lines of 128 bytes), and the one counter of small layers' one-launch calls.  Both are zeroed by cats_workspace_init and put back to zero by every call that uses them.
// Last: the per-workgroup sums of squares of that launch (overwritten by every call).
constexpr size_t kPoolCounterBytes = 4096;
constexpr size_t kArriveOffset = kPoolCounterBytes;
constexpr size_t kSmallArriveOffset = kArriveOffset + (size_t)(kArriveRows * kArriveGroups + kArriveRows) * kArriveStride * 4;
constexpr size_t kSsqOffset = kSmallArriveOffset + 256;  // one counter, and whole regions of 256 bytes
constexpr size_t kSsqFloats = 4096;  // workgroups of the reduction launch: B * H / 32
constexpr size_t kCounterBytes = kSsqOffset + kSsqFloats * 4;
#ifndef CATS_POOL_NUM  // share of a workgroup's neurons that goes to its group's pool (builds with -DCATS_FUSED_POOL=1 only)
#define CATS_POOL_NUM 1
#define CATS_POOL_DEN 4
#endif

__global__ void fill_zero_kernel(u32x4* p, size_t n16) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (size_t)gridDim.x * blockDim.x) p[i] = zero4();
}

// Read stream of known size for the measured bandwidth ceiling: every workgroup walks its own contiguous span (the
// fastest of the shapes tried: 7.0 TB/s on the MI355X against 6.7 for a grid-strided walk), every thread reads 16-byte
// vectors with the same streaming loads the weight rows take, eight in flight, and folds them into one word that is
// stored only if the fold hits a value the caller chooses (so the loads cannot be dropped and nothing is written).
__global__ __launch_bounds__(512) void read_probe_kernel(const u32x4* __restrict__ src, size_t n16, uint32_t never, uint32_t* sink) {
  constexpr int U = 8;
  const size_t span = (n16 + gridDim.x - 1) / gridDim.x;
  const size_t lo = (size_t)blockIdx.x * span < n16 ? (size_t)blockIdx.x * span : n16;
  const size_t hi = lo + span < n16 ? lo + span : n16;
  uint32_t acc = 0;
  // every pass issues U loads per thread; past the end of the span a thread re-reads the span's last vector (cached)
  // and drops it, so the tail of a span costs one pass like any other instead of a chain of single loads
  for (size_t i = lo + threadIdx.x; i < hi; i += (size_t)U * blockDim.x) {
    u32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const size_t j = i + (size_t)u * blockDim.x;
      v[u] = load_stream(src + (j < hi ? j : hi - 1));
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const size_t j = i + (size_t)u * blockDim.x;
      if (j < hi) acc ^= v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
    }
  }
  if (acc == never) *sink = acc;
}

// Number of neurons flagged in any of the B rows of flags (B, I): the count of a call that ran as several passes.
__global__ __launch_bounds__(1024) void union_count_kernel(const uint8_t* __restrict__ flags, int B, int I, int32_t* count_out) {
  __shared__ int s_part[16];
  int k = 0;
  for (int j = threadIdx.x; j < I; j += blockDim.x) {
    uint32_t on = 0;
    for (int b = 0; b < B; b++) on |= flags[(size_t)b * I + j];
    k += on != 0;
  }
  k = (int)wave_sum((float)k);  // at most I / 16 per wave, far below 2^24: exact in fp32
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  if (lane == 0) s_part[wave] = k;
  __syncthreads();
  if (threadIdx.x == 0) {
    int tot = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) tot += s_part[w];
    *count_out = tot;
  }
}

inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

struct WsLayout {
  size_t counters, mask, ubytes, z32, zt, partial, atmp, fin, total;
  size_t room() const { return mask - partial; }  // bytes of the partial sums
  bool mask_bytes = false;  // not part of the carving: the pass that just ran left the union of the flags in `ubytes`, not `mask`
};

constexpr int kMaxGroups = 64;  // neuron groups of the sparse down kernel; bounds the partial-sum scratch

// Bytes of partial sums that small layers' kernels may leave at most in a call that small_takes lets through, by how many workgroups there are
// (crowded: more than one a CU) and whether it is 9 to 16 rows of fp32.
constexpr int kSmallCuGroups = 256;
inline bool small_crowded(int groups) { return groups > kSmallCuGroups; }
inline size_t small_sums_most(bool crowded, bool f32_wide) { return (crowded ? 8500000u : 11000000u) * (size_t)(f32_wide ? 2 : 1); }
constexpr int kSmallCrowdedVecs = 128;  // of a row, at most

// What of that a layer of (H, I) can come to over all types and batches; 0 if no call of it is a small one.
size_t small_sum_bytes(int H, int I) {
  if (I > kSmallMaxNeurons) return 0;
  const int groups = small_max_groups(I);
  const size_t all = (size_t)groups * CATS_MAX_BATCH * H * 4;
  size_t most = 0;
  for (const int vec : {8, 4}) {
    if (H / vec > (small_crowded(groups) ? kSmallCrowdedVecs : kSmallMaxVecs)) continue;
    const size_t cap = small_sums_most(small_crowded(groups), vec == 4);
    if (most < (all < cap ? all : cap)) most = all < cap ? all : cap;
  }
  return most;
}

// The carving depends on (H, I) only -- every region is sized for kKernelBatch rows -- so calls with
// different batch sizes can share one workspace.  Nothing in it has to survive from one call to the next.
WsLayout ws_layout(int H, int I) {
  WsLayout l;
  const int B = kKernelBatch;
  size_t o = 0;
  l.counters = o; o += kCounterBytes;
  const size_t sums = (size_t)kMaxGroups * B * ((size_t)(H + 511) / 512 * 512) * 4, small = small_sum_bytes(H, I);
  l.partial = o;  o += align_up(sums > small ? sums : small, 256);
  l.mask = o;     o += align_up((size_t)((I + 63) / 64) * 8, 256);
  l.ubytes = o;   o += align_up((size_t)I + 8, 256);  // the same as a byte per neuron, read eight at a time
  l.z32 = o;      o += align_up((size_t)CATS_MAX_BATCH * I * 4, 256);  // 16 rows: the one-pass gate + up of 9..16 rows fills it whole
  l.zt = o;       o += align_up((size_t)B * I * 4, 256);
  l.atmp = o;     o += align_up((size_t)B * I * 4, 256);
  l.fin = o;      o += align_up((size_t)CATS_MAX_BATCH * H * 4, 256);  // finished columns as fp32, for the launch that also writes the next norm
  l.total = o;
  return l;
}

inline int elem_size(int dtype) { return dtype == CATS_F32 ? 4 : 2; }
inline int vec_elems(int dtype) { return dtype == CATS_F32 ? 4 : 8; }
inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// float -> fp16 bits, round to nearest even (host side, for the threshold).
uint16_t f32_to_f16_bits(float f) {
  uint32_t x;
  memcpy(&x, &f, 4);
  const uint32_t sign = (x >> 16) & 0x8000u;
  x &= 0x7fffffffu;
  if (x > 0x7f800000u) return (uint16_t)(sign | 0x7e00u);           // NaN
  if (x >= 0x47800000u) return (uint16_t)(sign | 0x7c00u);          // >= 65536 -> inf (65520 rounds up below)
  if (x < 0x38800000u) {                                             // below the smallest normal half
    if (x < 0x33000000u) return (uint16_t)sign;                      // < 2^-25 -> 0
    const int e = (int)(x >> 23);                                     // biased fp32 exponent
    uint32_t m = (x & 0x7fffffu) | 0x800000u;                         // 24-bit significand
    const int shift = 126 - e;                                        // 14..24: bits dropped to reach 2^-24 units
    const uint32_t half = 1u << (shift - 1);
    const uint32_t rem = m & ((1u << shift) - 1u);
    m >>= shift;
    if (rem > half || (rem == half && (m & 1u))) m++;
    return (uint16_t)(sign | m);
  }
  uint32_t h = ((x - 0x38000000u) >> 13);                            // rebias exponent, keep 10 mantissa bits
  const uint32_t rem = x & 0x1fffu;
  if (rem > 0x1000u || (rem == 0x1000u && (h & 1u))) h++;            // may carry into the exponent (and to inf)
  return (uint16_t)(sign | h);
}

float f16_bits_to_f32(uint16_t h) {
  const uint32_t sign = (uint32_t)(h & 0x8000u) << 16;
  uint32_t e = (h >> 10) & 0x1fu, m = h & 0x3ffu, x;
  if (e == 0) {
    if (m == 0) {
      x = sign;
    } else {
      int s = 0;
      while (!(m & 0x400u)) { m <<= 1; s++; }
      x = sign | ((uint32_t)(113 - s) << 23) | ((m & 0x3ffu) << 13);
    }
  } else if (e == 31) {
    x = sign | 0x7f800000u | (m << 13);
  } else {
    x = sign | ((e + 112) << 23) | (m << 13);
  }
  float f;
  memcpy(&f, &x, 4);
  return f;
}

float round_through(int dtype, float t) {
  if (dtype == CATS_F16) return f16_bits_to_f32(f32_to_f16_bits(t));
  if (dtype == CATS_BF16) {
    uint32_t u;
    memcpy(&u, &t, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return t;
    u += 0x7fffu + ((u >> 16) & 1u);
    u &= 0xffff0000u;
    float f;
    memcpy(&f, &u, 4);
    return f;
  }
  return t;
}

int batch_template(int B) { return B <= 1 ? 1 : (B <= 2 ? 2 : (B <= 4 ? 4 : 8)); }

int check_common(int B, int H, int I, int dtype) {
  if (dtype != CATS_F16 && dtype != CATS_BF16 && dtype != CATS_F32) return CATS_ERR_DTYPE;
  if (B < 1 || B > kKernelBatch) return CATS_ERR_BATCH;
  if (H <= 0 || I <= 0) return CATS_ERR_SHAPE;
  if (((size_t)H * elem_size(dtype)) % 16 != 0) return CATS_ERR_ALIGN;
  return CATS_OK;
}

void fill_rows(RowsArgs& a, const void* x, const void* w, int K, int N, int nb, int dtype) {
  memset(&a, 0, sizeof(a));
  a.x = (const u32x4*)x;
  a.w = (const u32x4*)w;
  a.K = K;
  a.N = N;
  a.nb = nb;
  a.out_pitch = N;
  const int vec = vec_elems(dtype);
  a.row_vecs = K / vec;
  a.nch = (a.row_vecs + kWave - 1) / kWave;
}

bool rows_take_mma(int mode, int dtype, int bt, const RowsArgs& a) {
  return dtype == CATS_F16 ? rows_takes_mma<F16>(mode, bt, a) : dtype == CATS_BF16 ? rows_takes_mma<BF16>(mode, bt, a) : rows_takes_mma<F32>(mode, bt, a);
}

// Whether do_rows' pass writes the union of the flags as bytes (a.ubytes_out, the matrix-core kernel) rather than as bits
// (a.mask_out); the down pass that follows has to be told (WsLayout::mask_bytes).
bool rows_mask_is_bytes(int mode, int dtype, RowsArgs a) {
  a.mma = g_tuning.gate_variant >= 0;
  const int bt = batch_template(a.nb);
  return rows_take_mma(mode, dtype, bt, a);
}

int do_rows(int mode, int dtype, const RowsArgs& a_in, hipStream_t s) {
  RowsArgs a = a_in;
  a.mma = g_tuning.gate_variant >= 0;  // gate_variant < 0: keep batches of 2..8 on the wave-per-row kernel
  if (g_tuning.gate_variant > 0) a.lds_floor = (160 * 1024) / g_tuning.gate_variant - 1024;  // at most gate_variant workgroups per CU
#ifdef CATS_TIMING
  a.tbuf = g_tbuf_rows;
#endif
  const int bt = batch_template(a.nb);
  hipError_t e;
  if (dtype == CATS_F16) e = launch_rows<F16>(mode, bt, a, s);
  else if (dtype == CATS_BF16) e = launch_rows<BF16>(mode, bt, a, s);
  else e = launch_rows<F32>(mode, bt, a, s);
  return e == hipSuccess ? CATS_OK : CATS_ERR_LAUNCH;
}

// Optional second output of the launch that finishes y: next.out = next.w * rms_norm(y).
struct NextNorm {
  const void* w = nullptr;
  float eps = 0.f;
  void* out = nullptr;
};

// What follows two matrix-core GEMVs over W_gate and W_up, for fp32 rows whose x operands do not fit in LDS whole (rows_mma_kernel): flags,
// their union and z from the sums g = x . Wgate^T and u = x . Wup^T, both (nb, N).  One thread per neuron.  z may take u's place or g's.
// The wave-per-row kernel reads x from global memory there: 12936 rows of 4912 at 8 batch rows 570 us, this way 140.
struct GateUpJoinArgs {
  const float* g;
  const float* u;
  float* z;
  uint8_t* flag_out;    // optional (nb, N)
  uint8_t* ubytes_out;  // optional (N,)
  int N, nb;
  float t;
};
__global__ __launch_bounds__(256) void gate_up_join_kernel(GateUpJoinArgs p) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= p.N) return;
  bool any = false;
  for (int b = 0; b < p.nb; b++) {
    const size_t o = (size_t)b * p.N + j;
    const float g = p.g[o], u = p.u[o], a = g / (1.f + expf(-g));
    const bool act = fabsf(a) > p.t;
    any = any || act;
    if (p.flag_out) p.flag_out[o] = act ? 1 : 0;
    p.z[o] = act ? a * u : 0.f;
  }
  if (p.ubytes_out) p.ubytes_out[j] = any ? 1 : 0;
}

constexpr int kJoinRows = 32;  // weight rows a workgroup of the fp32 matrix-core GEMV takes at most

// fp32 gate + up (a as for kGateUp, no norm, at least five batch rows) as two dense GEMVs and gate_up_join_kernel, where rows_mma_kernel
// does not take all the rows of x at once.  It reads every row of W_up, which from five batch rows on is little more than their union.
// The gate call and the gate + up call go the same way there, so that all three agree on every activation.
bool joined_takes(int dtype, const RowsArgs& a) {
  if (dtype != CATS_F32 || a.nb <= 4 || a.nb > CATS_MAX_BATCH || a.norm_w || g_tuning.gate_variant < 0) return false;
  RowsArgs one = a;
  one.mma = 1;
  return a.nb > kKernelBatch ? !rows_mma16_supported<F32>(one) : !rows_takes_mma<F32>(kGateUp, kKernelBatch, one);
}
// x . w^T in launches of at most kJoinRows rows a workgroup; a.zt_out, a_in, a_out and flag_out as gemv_mma_kernel takes them.
int do_joined_product(const RowsArgs& a, const u32x4* w, hipStream_t s) {
  const int most = current_device_cus() * kJoinRows, parts = (a.N + most - 1) / most;
  const int per = ((a.N + parts - 1) / parts + 7) / 8 * 8;
  for (int n0 = 0; n0 < a.N; n0 += per) {
    RowsArgs g = a;
    g.w = w + (size_t)n0 * a.row_vecs;
    g.w2 = nullptr;
    g.N = a.N - n0 < per ? a.N - n0 : per;
    if (g.zt_out) g.zt_out = (float*)a.zt_out + n0;
    if (g.a_in) g.a_in = (const float*)a.a_in + n0;
    if (g.a_out) g.a_out = (float*)a.a_out + n0;
    if (g.flag_out) g.flag_out = a.flag_out + n0;
    if (int st = do_rows(kGemv, CATS_F32, g, s)) return st;
  }
  return CATS_OK;
}
// The gate call (a as for kGate): the same sums and the same activations as do_joined's.
int do_joined_gate(const RowsArgs& a, hipStream_t s) { return do_joined_product(a, a.w, s); }
// The gate + up call (a as for kGateUp with zt_out and no mask): the activations wait in zt_out for the up sums.
int do_joined_gate_up(const RowsArgs& a, hipStream_t s) {
  RowsArgs g = a;
  g.zt_out = nullptr;
  g.a_out = a.zt_out;
  if (int st = do_joined_product(g, a.w, s)) return st;
  g = a;
  g.a_in = a.zt_out;
  g.flag_out = nullptr;
  return do_joined_product(g, a.w2, s);
}
// sums: nb * N floats of scratch, z: (nb, N), which takes the up sums first
int do_joined(const RowsArgs& a, float* sums, float* z, hipStream_t s) {
  RowsArgs g = a;
  g.z32_out = nullptr;
  g.flag_out = g.mask_out = g.ubytes_out = nullptr;
  for (int m = 0; m < 2; m++) {
    g.zt_out = m ? z : sums;
    if (int st = do_joined_product(g, m ? a.w2 : a.w, s)) return st;
  }
  GateUpJoinArgs j = {sums, z, z, a.flag_out, a.ubytes_out, a.N, a.nb, a.t};
  return launch_kernel(gate_up_join_kernel, dim3((a.N + 255) / 256), dim3(256), 0, s, j) == hipSuccess ? CATS_OK : CATS_ERR_LAUNCH;
}

int do_reduce(const ReduceArgs& r, int dtype, hipStream_t s) {
  const hipError_t e = dtype == CATS_F16 ? launch_reduce<F16>(r, s) : dtype == CATS_BF16 ? launch_reduce<BF16>(r, s) : launch_reduce<F32>(r, s);
  return e == hipSuccess ? CATS_OK : CATS_ERR_LAUNCH;
}

// Fills the next-norm fields of the reduction launch; CATS_ERR_SHAPE if the launch cannot carry it.
int set_next_norm(ReduceArgs& r, const NextNorm& next, char* ws, const WsLayout& l) {
  if (!next.out) return CATS_OK;
  if (r.H % kReduceCols != 0 || (size_t)(r.BH / kReduceCols) > kSsqFloats) return CATS_ERR_SHAPE;
  r.norm2_out = next.out;
  r.norm2_w = next.w;
  r.norm2_eps = next.eps;
  r.arrive = (int32_t*)(ws + l.counters + kArriveOffset);
  r.ssq_part = (float*)(ws + l.counters + kSsqOffset);
  r.fin = (float*)(ws + l.fin);
  return CATS_OK;
}

constexpr int kFusedMaxGrid = 256;  // partials of 256 workgroups x 2 batch rows fit the workspace's partial-sum region
constexpr int kNotTaken = -1;  // internal: the shape or type rules this way out, take the other one

// Neurons (or list entries) of a group of the sparse down pass, out of zcols; 0 if a group's list and z would not fit in LDS.
// About one workgroup per CU over all slabs.
int down_chunk(int zcols, int nslab, int B) {
  int ngroup = g_tuning.down_groups > 0 ? g_tuning.down_groups : 256 / nslab;
  if (ngroup < 1) ngroup = 1;
  if (ngroup > kMaxGroups) ngroup = kMaxGroups;
  if (B > kKernelBatch && ngroup > kMaxGroups / 2) ngroup = kMaxGroups / 2;  // the partial sums of 16 rows take twice the room
  const int chunk = ((zcols + ngroup - 1) / ngroup + 7) / 8 * 8;
  return (size_t)chunk * (1 + batch_template(B < kKernelBatch ? B : kKernelBatch)) * 4 > 96 * 1024 ? 0 : chunk;
}

// Sparse down over mask words already in the workspace.  Up to kKernelBatch rows; 16-bit types with an output that goes
// through partial sums also take up to CATS_MAX_BATCH rows in one pass over W_down^T (matrix-core kernel) -- a call with
// more than kKernelBatch rows that cannot go that way returns kNotTaken before anything is launched.
int do_down(const void* z, bool zf32, const void* wdown_t, float* y32, void* y_out, int32_t* count_out, int B, int H, int I,
            int dtype, char* ws, const WsLayout& l, hipStream_t s, const void* residual = nullptr, const uint8_t* flags = nullptr,
            const int64_t* idx = nullptr, int M = 0, const void* bias = nullptr, const NextNorm& next = NextNorm()) {
  DownArgs d;
  memset(&d, 0, sizeof(d));
  d.wd = (const u32x4*)wdown_t;
  d.z = z;
  d.mask = (const uint8_t*)(ws + (l.mask_bytes ? l.ubytes : l.mask));
  d.mask_bytes = l.mask_bytes ? 1 : 0;
  d.flags = flags;
  d.idx = idx;
  d.M = M;
  // The caller's fp32 accumulator: up to two rows the workgroups add into it themselves (one launch); from three rows
  // on that is eight or more rows of atomics per workgroup and slower than leaving partial sums for the reduction launch,
  // which then adds the total into the accumulator (measured at 4 / 8 / 16 rows: 53.9 / 64.6 / 104 us against 52.8 / 59.1 / 87.5).
  const bool reduce_into_y32 = y32 != nullptr && y_out == nullptr && B >= 3;
  d.y32 = y32;
  d.y_out = y_out;
  d.partial_out = (y_out != nullptr || reduce_into_y32) ? 1 : 0;
  d.partial = (float*)(ws + l.partial);
  d.count_out = count_out;
  d.H = H; d.I = I; d.nb = B;
  d.row_vecs = H / vec_elems(dtype);
  d.nslab = (d.row_vecs + kWave - 1) / kWave;
  if (d.nslab > kMaxSlabs) return CATS_ERR_SHAPE;
  int block = g_tuning.down_block > 0 ? g_tuning.down_block : 1024;
  if (block < 128) block = 128;  // wave 0 builds the index list, the others stage z
  if (block > 1024) block = 1024;
  while (block & (block - 1)) block &= block - 1;  // the fold across waves halves their number per round
  const int bt = batch_template(B < kKernelBatch ? B : kKernelBatch);
  const int zcols = idx ? M : I;  // what the groups split: the index list, or the neuron range
  d.chunk = down_chunk(zcols, d.nslab, B);
  if (d.chunk == 0) return B > kKernelBatch ? kNotTaken : CATS_ERR_SHAPE;
  d.ngroup = (zcols + d.chunk - 1) / d.chunk;
#ifdef CATS_TIMING
  d.tbuf = g_tbuf_down;
#endif
  // Three rows and more of a 16-bit type: the matrix-core kernel (gate_variant < 0 or an explicit down_block keep the
  // wave-per-row-pair kernel, for comparison).  At one and two rows the latter is the faster one (stand-alone down at
  // 50 % flags per row: 14.0 / 18.9 us against 15.1 / 19.3).
  bool mma = dtype != CATS_F32 && B >= 3 && d.partial_out && g_tuning.gate_variant >= 0 && g_tuning.down_block == 0;
  if (mma) mma = dtype == CATS_F16 ? down_mma_supported<F16>(d) : down_mma_supported<BF16>(d);
  if (B > kKernelBatch && !mma) return kNotTaken;
  hipError_t e;
  if (mma) e = dtype == CATS_F16 ? launch_down_mma<F16>(zf32, d, s) : launch_down_mma<BF16>(zf32, d, s);
  else if (dtype == CATS_F16) e = launch_down<F16>(bt, zf32, d, block, s);
  else if (dtype == CATS_BF16) e = launch_down<BF16>(bt, zf32, d, block, s);
  else e = launch_down<F32>(bt, zf32, d, block, s);
  if (e != hipSuccess) return CATS_ERR_LAUNCH;
  if (!d.partial_out) return CATS_OK;
  // The groups' partial sums are added by the reduction launch: rounded into y_out (and the residual added), or added to y32.
  ReduceArgs r;
  memset(&r, 0, sizeof(r));
  r.partial = d.partial;
  r.y_out = y_out;
  r.y32_acc = reduce_into_y32 ? y32 : nullptr;
  r.residual = residual;
  r.bias = bias;
  r.H = H;
  r.G = d.ngroup;
  r.BH = B * H;
  if (int st = set_next_norm(r, next, ws, l)) return st;
  return do_reduce(r, dtype, s);
}

// Whether the kernels of small layers take this call (a as for kGateUp, the neurons' down rows as (I, H)), and the grid.  They read every row of
// all three matrices and leave partial sums of sixteen neurons each, against kept rows only and one launch more, or a chain of trips more, in the other
// kernels.  GPU time by HIP graph, those against these, us at 50 to 70 % sparsity:
//   1 row, 16 bits    512 / 1024 9.6, 5.6   1024 / 2731 11.5, 7.9   2048 / 3072 12.2, 11.0 (at 90 % 11.1, 11.0)   2048 / 4096 13.4, 13.0 (12.0, 13.0)
//   1 row, fp32       512 / 1024 9.6, 6.4   1024 / 3300 12.1, 11.1 (11.1, 10.8)   1024 / 4096 13.0, 12.6 (11.6, 12.5)   4 rows 19.6, 15.9
//   4 rows            512 / 1024 12.5, 7.3   1024 / 2731 15.3, 10.4   2048 / 3072 18.4, 16.1   8 rows 20.3, 19.5
//   8 rows            1024 / 4096 16.5, 14.6 (8.4 MB of sums)   1536 / 4096 19.1, 19.3 (12.6 MB)
//   16 rows           1024 / 1600 15.5, 14.1 (6.6 MB)   1024 / 2731 17.6, 17.1 (11.2 MB)   1400 / 3000 20.1, 22.1 (16.8 MB)
//   16 rows, fp32     1024 / 2731 36.0, 22.6   1024 / 4096 40.0, 27.1 (16.8 MB; the other way reads the down weight twice)
// Beyond one workgroup a CU: 512 / 8000 15.0, 9.9 at 1 row and 17.8, 15.0 at 8;  704 / 6000 17.3, 17.1 at 8 (8.4 MB);  1024 / 5000 13.4, 11.4 at 1,
// 17.8, 19.8 at 8 (10.3 MB);  1200 / 5000 (rows of 150 vectors, one workgroup a CU at a time) 12.0, 13.3 at 1 row and 90 %.
// What is read for nothing grows with the sparsity, so from three rows on the lines are drawn with 30, 60 and 90 % of it measured: by the sums, and by
// a matrix and the sums together (MB of both below).  Those and these in us at 30 / 60 / 90 %:
//   a workgroup a CU       3 rows 2048 / 3700 18.9, 17.6 / 18.7, 17.9 / 18.2, 17.3 (5.7, 20.8)   2048 / 4096 19.9, 19.2 / 19.6, 19.5 / 19.0, 19.4 (6.3, 23.1)
//                          5 rows 1792 / 4000 18.8, 17.2 / 18.7, 17.2 / 18.1, 17.1 (9.0, 23.3)   2048 / 3700 20.0, 19.9 / - / 19.5, 19.7 (9.5, 24.7)
//                          8 rows 1536 / 3500 17.9, 17.1 / 17.9, 17.1 / 17.5, 17.1 (10.8, 21.5)
//     rows of more than 224 vectors are what the others are best at, four slabs of 64:
//                          5 rows 2048 / 3300 18.6, 18.5 / 18.5, 18.5 / 18.1, 18.5 (8.4, 21.9)   2040 / 3500 20.3, 20.2 / 20.2, 20.1 / 19.6, 20.2 (8.9, 23.2)
//                          8 rows 2048 / 2600 18.6, 18.8 / 18.7, 18.8 / 18.2, 18.7 (10.7, 21.3)
//   two a CU               4 rows 1024 / 5000 16.5, 15.9 / 16.3, 15.9 / 15.9, 15.8 (5.1, 15.4)   6 rows 1024 / 4300 16.7, 16.6 / 16.6, 16.7 / 16.2, 16.7 (6.6, 15.4)
//                          6 rows 840 / 5000 17.1, 17.5 / 17.0, 17.5 / 16.7, 17.5 (6.5, 14.9)   704 / 6000 16.5, 15.7 / 16.4, 15.8 / 15.9, 15.7 (6.3, 14.8)
//     short rows, slabs that the others do not fill:   8 rows 512 / 8000 17.3, 14.9 / 17.2, 14.9 / 16.8, 14.9 (8.2, 16.4)   520 / 8000 18.1, 16.9 / 18.0,
//                          16.9 / 17.4, 16.9 (8.3, 16.6)
//   more than one a CU, but no place for two: more than 64 registers from three steps a wave on, at nine rows and more from two
//                          3 rows 1000 / 4200 17.3, 16.7 / 17.1, 16.7 / 16.7, 16.7 (3.2, 11.6)   6 rows 17.9, 19.2 / - / 17.4, 19.2 (6.3, 14.7)
//                          12 rows 520 / 5000 19.8, 19.1 / 19.8, 19.1 / 17.8, 19.1 (7.8, 13.0)   11 rows 640 / 4500 19.2, 19.3 / - / 17.6, 19.3 (7.9, 13.7)
//   fp32                   5 rows 1024 / 4096 23.2, 20.6 / 22.6, 20.9 / 19.6, 20.9 (5.2, 22.0)   8 rows 23.9, 22.7 / - / 20.6, 23.0 (8.4, 25.2)
//                          8 rows 512 / 5000 20.5, 19.4 / - / 18.6, 19.4 (5.1, 15.4)   512 / 8000 24.3, 22.9 / - / 20.8, 22.9 (8.2, 24.6)
// At one and two rows the gain at low sparsity is the larger: 2048 / 3300 at one row 12.6, 11.8 at 50 % and 11.5, 11.8 at 90 %.
// room: bytes there are for the sums.
bool small_takes(RowsArgs& a, int dtype, size_t room, bool& mma, int& grid) {
  if (g_tuning.path == 1 || g_tuning.gate_variant != 0 || g_tuning.down_groups > 0 || g_tuning.down_block > 0) return false;
  if (a.nb < 1 || a.nb > CATS_MAX_BATCH || a.N > kSmallMaxNeurons) return false;
  mma = a.nb > (dtype == CATS_F32 ? 4 : 2);  // as takes_mma has it for the gate
  grid = small_layout(a, mma);
  if (grid <= 0 || grid > small_max_groups(a.N)) return false;
  const size_t bytes = (size_t)a.N * a.K * elem_size(dtype), sums = (size_t)grid * a.nb * a.K * 4;
  if (sums > room) return false;
  const bool crowded = small_crowded(grid);  // two workgroups a CU fit where a row is at most 128 vectors
  if (crowded && a.row_vecs > kSmallCrowdedVecs) return false;
  if (!mma) return bytes <= (dtype == CATS_F32 && a.nb > 2 ? 17000000u : crowded ? 11000000u : 13600000u);
  const bool f32_wide = dtype == CATS_F32 && a.nb > kKernelBatch;  // the other way reads the down weight twice
  // no place for two 16-bit workgroups a CU with more registers than these steps take; fp32 as measured
  const bool two_fit = dtype == CATS_F32 || rows_mma_split(a).steps <= (a.nb > kKernelBatch ? 1 : 2);
  const size_t most = !crowded ? 23500000u : two_fit ? 17000000u : 13500000u;
  if (dtype != CATS_F32 && sums > (crowded ? (a.row_vecs > 80 ? 6400000u : 8500000u) : a.row_vecs > 224 ? 8500000u : 11000000u)) return false;
  return sums <= small_sums_most(crowded, f32_wide) && bytes + sums <= most * (f32_wide ? 2 : 1);
}

// Sums of a batch row that one workgroup adds up sooner than a launch over all CUs and, for the layer tail, the hand-over in front of its norm
// (tail with the next norm, one row: 512 / 1024, 131 KB, 7.8 us against 10.1; 704 / 1451, 256 KB, 11.1; 1024 / 1965, 504 KB, 13.2 against 11.8).
constexpr size_t kSmallTailBytes = 300000;
// One batch row up to here is one launch: the call then takes 8.0 us, what its kernel takes (8.2 to 8.6 traced; the host needs 6.1 for the same call over
// 64 / 64, 5.1 for one projection), instead of 8.7 to 9.2, the host's pace with a second launch, though the kernel takes 1 to 2 us more than the two; 512 / 2048, 262 KB: 10.1 against 8.6.  In a captured graph launches are cheap: two there, with the
// sums in the same order.
constexpr size_t kSmallOneLaunchBytes = 131072;

// y32: the caller's fp32 sums, which the call adds to.  partial, counts: instead of those in ws (then NULL), memory without an arrival
// counter that calls keep at zero, so two launches.
int do_small(const RowsArgs& a, bool mma, int grid, int stage, const void* wdown_t, void* y_out, const void* residual, float* y32, int32_t* count_out,
             int dtype, char* ws, const WsLayout& l, hipStream_t s, const NextNorm& next = NextNorm(), float* partial = nullptr, int32_t* counts = nullptr) {
  SmallArgs k;
  memset(&k, 0, sizeof(k));
  k.r = a;
  k.wd = (const u32x4*)wdown_t;
  k.partial = partial ? partial : (float*)(ws + l.partial);
  k.counts = counts ? counts : (int32_t*)(ws + l.z32);
  ReduceArgs& r = k.fin;
  r.partial = k.partial;
  r.counts = k.counts;
  r.count_out = count_out;
  r.y_out = y_out;
  r.y32_acc = y32;
  r.residual = residual;
  r.H = a.K;
  r.G = grid;
  r.BH = a.nb * a.K;
  if (int st = set_next_norm(r, next, ws, l)) return st;
  const size_t row = (size_t)grid * a.K * 4;
  const bool one = a.nb == 1 && row <= kSmallOneLaunchBytes;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (one && stage == 0 && ws && hipStreamIsCapturing(s, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone)
    k.arrive = (int32_t*)(ws + l.counters + kSmallArriveOffset);
  hipError_t e = hipSuccess;
  if (stage != 2) e = dtype == CATS_F16 ? launch_small<F16>(mma, grid, k, s) : dtype == CATS_BF16 ? launch_small<BF16>(mma, grid, k, s) : launch_small<F32>(mma, grid, k, s);
  if (e != hipSuccess) return CATS_ERR_LAUNCH;
  if (stage == 1 || k.arrive) return CATS_OK;
  if (!one && (!residual || row > kSmallTailBytes)) return do_reduce(r, dtype, s);
  e = dtype == CATS_F16    ? launch_small_tail<F16>(a.nb, r, s)
      : dtype == CATS_BF16 ? launch_small_tail<BF16>(a.nb, r, s)
                           : launch_small_tail<F32>(a.nb, r, s);
  return e == hipSuccess ? CATS_OK : CATS_ERR_LAUNCH;
}

int check_ws(const void* ws, size_t ws_bytes, int H, int I, WsLayout& l) {
  l = ws_layout(H, I);
  if (ws == nullptr || ws_bytes < l.total || ((uintptr_t)ws & 255u) != 0) return CATS_ERR_WORKSPACE;
  return CATS_OK;
}


constexpr int kFusedPerCU = 16 / kFusedWaves;  // workgroups per CU: 1, or 2 in the 512-thread experiment build (one batch row only)

// Whether the single-pass kernel covers this call, and with what launch shape: one workgroup per CU, each with an
// equal, contiguous share of the neurons.
// `any_path`: ignore the A/B knob that keeps whole-MLP calls on the separate kernels (cats_set_tuning(path = 1)).
bool fused_eligible(int B, int H, int I, int dtype, FusedArgs& f, int& grid, bool any_path = false) {
  if ((g_tuning.path == 1 && !any_path) || B > 2) return false;
  const int vec = vec_elems(dtype);
  memset(&f, 0, sizeof(f));
  f.H = H; f.I = I; f.nb = B;
  f.row_vecs = H / vec;
  f.nch = (f.row_vecs + kWave - 1) / kWave;
  const int bt = batch_template(B);
  const int dw = fused_down_waves(bt), rw = kFusedWaves - dw;
  if (f.row_vecs > kFusedMaxKV * dw * kWave) return false;
  int maxgrid = current_device_cus();
  if (maxgrid > kFusedMaxGrid) maxgrid = kFusedMaxGrid;
  if (B == 1) maxgrid *= kFusedPerCU;  // at two rows twice the workgroups would not fit the partial-sum region
  int rpw = (I + maxgrid - 1) / maxgrid;
  // Small matrices: at least half as many neurons as row waves, so that a wave takes one at most -- a second neuron is one more memory
  // trip in a chain of four.  Fewer workgroups with two neurons a wave: 13.1 against 10.8 us at 512 / 1024, 14.4 against 12.0 at
  // 1024 / 2731, 15.1 against 12.2 at two rows of 512 / 1995; one neuron a wave and no idle wave: 11.1, 12.3, 12.1.
  if (rpw < rw / 2) rpw = rw / 2;
  grid = (I + rpw - 1) / rpw;
  f.rpw = rpw;
  f.spw = rpw;
  f.cap = rpw;
  return fused_lds_bytes(bt, f.nch, f.cap, vec, dw) <= kStagedMaxBytes;
}

// Give the call a neuron pool if its shape allows: a fixed fraction of every workgroup's neurons goes to the pool of
// its group.  `counters`: pool counter lines, zero, at least kPoolStride int32 per group of kFusedGroup workgroups.
void fused_enable_pool(FusedArgs& f, int grid, int dtype, int32_t* counters, size_t counter_bytes) {
  if (!kFusedPool || !f.wg || CATS_POOL_NUM == 0) return;  // given activations: no gate rows to balance, shares stay fixed
  const int bt = batch_template(f.nb);
  const int dw = fused_down_waves(bt), rw = kFusedWaves - dw;
  const int spw = f.rpw - f.rpw * CATS_POOL_NUM / CATS_POOL_DEN;
  const int groups = (grid + kFusedGroup - 1) / kFusedGroup;
  if (spw == f.rpw || spw < 2 * rw || (size_t)groups * kPoolStride * 4 > counter_bytes) return;
  const int cap = fused_slot_cap(spw, f.rpw, rw, true);
  if (fused_lds_bytes(bt, f.nch, cap, vec_elems(dtype), dw) > kStagedMaxBytes) return;
  f.spw = spw;
  f.cap = cap;
  f.pool = counters;
}

// y32 set: the streaming kernel adds into the caller's fp32 accumulator itself and nothing is launched after it,
// unless the caller wants the count of active neurons (then the second launch does only that).
int do_fused(FusedArgs& f, int grid, int stage, void* y_out, const void* residual, int32_t* count_out, int dtype, char* ws,
             const WsLayout& l, hipStream_t s, float* y32 = nullptr, const NextNorm& next = NextNorm()) {
  f.partial = (float*)(ws + l.partial);
  f.counts = (int32_t*)(ws + l.z32);
  f.y32 = y32;
  fused_enable_pool(f, grid, dtype, (int32_t*)(ws + l.counters), kPoolCounterBytes);
#ifdef CATS_TIMING
  f.tbuf = g_tbuf_fused;
#endif
  ReduceArgs r;
  memset(&r, 0, sizeof(r));
  r.partial = f.partial;
  r.counts = f.counts;
  r.y_out = y_out;
  r.residual = residual;
  r.count_out = count_out;
  r.H = f.H;
  r.G = grid;
  r.BH = f.nb * f.H;
  if (y32) {
    r.BH = 0;  // no columns to finish
    if (stage == 0 && !count_out) stage = 1;
  }
  if (int st = set_next_norm(r, next, ws, l)) return st;
  const int bt = batch_template(f.nb);
  hipError_t e;
  if (dtype == CATS_F16) e = launch_fused<F16>(bt, grid, stage, f, r, s);
  else if (dtype == CATS_BF16) e = launch_fused<BF16>(bt, grid, stage, f, r, s);
  else e = launch_fused<F32>(bt, grid, stage, f, r, s);
  return e == hipSuccess ? CATS_OK : CATS_ERR_LAUNCH;
}

// Device address of this GPU's copy of `scratch`.  The array's name means nothing to a kernel when it is used in host
// code, so the address is asked for once per device (with that device current) and kept.
constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices];
std::mutex g_scratch_mu;

int scratch_address(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return CATS_ERR_LAUNCH;
  void* p = __atomic_load_n(&g_scratch_ptr[dev], __ATOMIC_ACQUIRE);
  if (p == nullptr) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    p = g_scratch_ptr[dev];
    if (p == nullptr) {
      if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) return CATS_ERR_LAUNCH;
      __atomic_store_n(&g_scratch_ptr[dev], p, __ATOMIC_RELEASE);
    }
  }
  *out = p;
  return CATS_OK;
}

}  // namespace
}  // namespace cats

using namespace cats;

namespace {  // pass helpers of the public entry points
inline const void* at_cbytes(const void* p, size_t bytes) { return p ? (const char*)p + bytes : nullptr; }
inline void* at_bytes(void* p, size_t bytes) { return p ? (char*)p + bytes : nullptr; }
inline size_t esz(int dtype) { return dtype == CATS_F32 ? 4 : 2; }
template <class F>
int in_passes(int B, F&& pass) {
  if (B < 1 || B > CATS_MAX_BATCH) return CATS_ERR_BATCH;
  for (int b0 = 0; b0 < B; b0 += kKernelBatch) {
    const int nb = B - b0 < kKernelBatch ? B - b0 : kKernelBatch;
    if (int st = pass((size_t)b0, nb)) return st;
  }
  return CATS_OK;
}
}  // namespace

extern "C" {

#ifdef CATS_TIMING
void cats_timing_buffers(void* rows, void* down) { g_tbuf_rows = (long long*)rows; g_tbuf_down = (long long*)down; }
void cats_timing_buffer_fused(void* fused) { g_tbuf_fused = (long long*)fused; }
#endif

int cats_version(void) { return 100; }

const char* cats_status_string(int status) {
  switch (status) {
    case CATS_OK: return "ok";
    case CATS_ERR_DTYPE: return "unsupported dtype (expected 0=fp16, 1=bf16, 2=fp32)";
    case CATS_ERR_SHAPE: return "unsupported shape (H, I must be positive; H <= 128 slabs of 64 x 16 bytes)";
    case CATS_ERR_ALIGN: return "pointer or row pitch not 16-byte aligned";
    case CATS_ERR_BATCH: return "unsupported batch (1..16 rows; the active-neuron count is available for 1..8)";
    case CATS_ERR_NULL: return "required pointer is NULL";
    case CATS_ERR_WORKSPACE: return "workspace missing, misaligned (256 bytes) or smaller than cats_workspace_bytes()";
    case CATS_ERR_LAUNCH: return "HIP kernel launch failed";
    case CATS_ERR_SCRATCH: return "call does not fit the built-in scratch of cats_mlp_noalloc (1..2 rows, B * H <= 8192, rows of at most 1024 16-byte vectors at 1 row and 2048 at 2 rows)";
  }
  return "unknown status";
}

int cats_set_tuning(int gate_variant, int down_groups, int down_block, int path) {
  g_tuning.gate_variant = gate_variant;
  g_tuning.down_groups = down_groups;
  g_tuning.down_block = down_block;
  g_tuning.path = path;
  return CATS_OK;
}

size_t cats_workspace_bytes(int B, int H, int I) {
  if (B < 1 || H < 1 || I < 1) return 0;
  return ws_layout(H, I).total;
}

int cats_workspace_init(void* ws, size_t ws_bytes, void* stream) {
  if (ws == nullptr) return CATS_ERR_NULL;
  if (((uintptr_t)ws & 255u) != 0 || ws_bytes % 16 != 0) return CATS_ERR_WORKSPACE;
  const size_t n16 = ws_bytes / 16;
  int grid = (int)((n16 + 255) / 256);
  if (grid > 2048) grid = 2048;
  if (grid < 1) grid = 1;
  return launch_kernel(fill_zero_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream, (u32x4*)ws, n16) == hipSuccess ? CATS_OK : CATS_ERR_LAUNCH;
}

// Launches the matrix-core kernel for 9..16 rows (gate + up when a.w2 is set, else the gate pass); kNotTaken if it does
// not take the shape.
static int rows_wide(RowsArgs& a, int dtype, void* stream) {
  a.mma = g_tuning.gate_variant >= 0;
#ifdef CATS_TIMING
  a.tbuf = g_tbuf_rows;
#endif
  const hipStream_t s = (hipStream_t)stream;
  if (!(dtype == CATS_F16 ? rows_mma16_supported<F16>(a) : dtype == CATS_BF16 ? rows_mma16_supported<BF16>(a) : rows_mma16_supported<F32>(a))) return kNotTaken;
  const hipError_t e = dtype == CATS_F16 ? launch_rows_mma16<F16>(a, s) : dtype == CATS_BF16 ? launch_rows_mma16<BF16>(a, s) : launch_rows_mma16<F32>(a, s);
  return e == hipSuccess ? CATS_OK : CATS_ERR_LAUNCH;
}

// B above kKernelBatch: all rows in one pass over W_gate where the matrix-core kernel takes the call, else kNotTaken.
static int gate_flag_pass(const void* x, const void* wgate, void* a_out, uint8_t* flag_out, int B, int H, int I, int dtype,
                   float threshold, void* stream) {
  const bool wide = B > kKernelBatch;
  if (wide && B > CATS_MAX_BATCH) return kNotTaken;
  int st = check_common(wide ? kKernelBatch : B, H, I, dtype);
  if (st) return st;
  if (!x || !wgate || (!a_out && !flag_out)) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(wgate)) return CATS_ERR_ALIGN;
  RowsArgs a;
  fill_rows(a, x, wgate, H, I, B, dtype);
  a.a_out = a_out;
  a.flag_out = flag_out;
  a.t = round_through(dtype, threshold);
  if (joined_takes(dtype, a)) return do_joined_gate(a, (hipStream_t)stream);
  return wide ? rows_wide(a, dtype, stream) : do_rows(kGate, dtype, a, (hipStream_t)stream);
}

int cats_gate_compact(const void* x, const void* wgate, void* vals_out, int64_t* idx_out, int32_t* count_out, int H, int I,
                      int dtype, float threshold, void* ws, size_t ws_bytes, void* stream) {
  int st = check_common(1, H, I, dtype);
  if (st) return st;
  if (!x || !wgate || !idx_out || !count_out) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(wgate)) return CATS_ERR_ALIGN;
  WsLayout l;
  st = check_ws(ws, ws_bytes, H, I, l);
  if (st) return st;
  // launch 1: the gate pass, activations and mask bytes into the workspace
  RowsArgs a;
  fill_rows(a, x, wgate, H, I, 1, dtype);
  a.a_out = (char*)ws + l.atmp;
  a.mask_out = (uint8_t*)ws + l.mask;
  a.t = round_through(dtype, threshold);
  st = do_rows(kGate, dtype, a, (hipStream_t)stream);
  if (st) return st;
  // launch 2: mask bytes -> ascending list, values, count
  CompactArgs c;
  c.mask = a.mask_out;
  c.a = a.a_out;
  c.idx_out = idx_out;
  c.vals_out = vals_out;
  c.count_out = count_out;
  c.N = I;
  const int nbytes = (I + 7) / 8;
  int groups = (nbytes + 255) / 256;  // at least one pass of 256 bytes each; more groups than that gain nothing
  if (groups > 64) groups = 64;
  c.bytes_per_group = (nbytes + groups - 1) / groups;
  groups = (nbytes + c.bytes_per_group - 1) / c.bytes_per_group;  // the last group's range is never empty: it writes the count
  const hipError_t e = elem_size(dtype) == 2 ? launch_kernel(compact_kernel<2>, dim3(groups), dim3(256), 0, (hipStream_t)stream, c)
                                             : launch_kernel(compact_kernel<4>, dim3(groups), dim3(256), 0, (hipStream_t)stream, c);
  return e == hipSuccess ? CATS_OK : CATS_ERR_LAUNCH;
}

int cats_probe_read(const void* src, size_t bytes, uint32_t* sink, void* stream) {
  if (!src || !sink) return CATS_ERR_NULL;
  if (!aligned16(src) || bytes % 16 != 0 || bytes == 0) return CATS_ERR_ALIGN;
  const int grid = current_device_cus() * 4;
  return launch_kernel(read_probe_kernel, dim3(grid), dim3(512), 0, (hipStream_t)stream, (const u32x4*)src, bytes / 16, 0x9e3779b9u, sink) == hipSuccess
             ? CATS_OK
             : CATS_ERR_LAUNCH;
}

int cats_read_count(const int32_t* count_dev, void* stream) {
  // One asynchronous copy into pinned host memory behind the caller's work on the stream, then one wait for the stream.
  // The pinned word is allocated on first use and shared, so readers take turns.
  static std::mutex mu;
  static int32_t* pinned = nullptr;
  if (!count_dev) return -1;
  std::lock_guard<std::mutex> lock(mu);
  if (!pinned && hipHostMalloc((void**)&pinned, 64, hipHostMallocDefault) != hipSuccess) {
    pinned = nullptr;
    return -1;
  }
  *pinned = -1;
  if (hipMemcpyAsync(pinned, count_dev, sizeof(int32_t), hipMemcpyDeviceToHost, (hipStream_t)stream) != hipSuccess) return -1;
  if (hipStreamSynchronize((hipStream_t)stream) != hipSuccess) return -1;
  return *pinned;
}

// B above kKernelBatch: all rows in one pass over W_up where the matrix-core kernel takes the call, else kNotTaken.
static int up_flag_pass(const void* x, const void* wup, const void* a_in, const uint8_t* flag, void* out, int out_is_f32, int B,
                 int H, int I, int dtype, void* stream) {
  const bool wide = B > kKernelBatch;
  if (wide && (B > CATS_MAX_BATCH || dtype == CATS_F32)) return kNotTaken;
  int st = check_common(wide ? kKernelBatch : B, H, I, dtype);
  if (st) return st;
  if (!x || !wup || !a_in || !flag || !out) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(wup)) return CATS_ERR_ALIGN;
  RowsArgs a;
  fill_rows(a, x, wup, H, I, B, dtype);
  a.a_in = a_in;
  a.flag_in = flag;
  if (out_is_f32) a.z32_out = (float*)out; else a.zt_out = out;
  if (wide && !rows_mask_is_bytes(kUp, dtype, a)) return kNotTaken;  // i.e. the matrix-core up kernel does not take it
  return do_rows(kUp, dtype, a, (hipStream_t)stream);
}

// B above kKernelBatch: all rows in one pass over W_down^T where the matrix-core down kernel takes the call, else kNotTaken.
static int down_flag_pass(const void* z, const void* wdown_t, const uint8_t* flag, float* y_f32, void* y_out, int B, int H, int I,
                   int dtype, void* ws, size_t ws_bytes, void* stream) {
  if (B > kKernelBatch && (B > CATS_MAX_BATCH || dtype == CATS_F32)) return kNotTaken;
  int st = check_common(B < kKernelBatch ? B : kKernelBatch, H, I, dtype);
  if (st) return st;
  if (!z || !wdown_t || !flag || ((y_f32 == nullptr) == (y_out == nullptr))) return CATS_ERR_NULL;
  if (!aligned16(wdown_t)) return CATS_ERR_ALIGN;
  WsLayout l;
  st = check_ws(ws, ws_bytes, H, I, l);
  if (st) return st;
  // the down kernel ORs the per-row flag bytes of its range itself: no separate packing launch
  float* acc = y_f32;
  return do_down(z, false, wdown_t, acc, y_out, nullptr, B, H, I, dtype, (char*)ws, l, (hipStream_t)stream, nullptr, flag);
}

// B above kKernelBatch: all rows in one pass over both matrices where the matrix-core kernel takes the call, else kNotTaken.
static int gate_up_pass(const void* x, const void* wgate, const void* wup, void* out, uint8_t* flag_out, int B, int H, int I,
                 int dtype, float threshold, void* stream) {
  const bool wide = B > kKernelBatch;
  if (wide && B > CATS_MAX_BATCH) return kNotTaken;
  int st = check_common(wide ? kKernelBatch : B, H, I, dtype);
  if (st) return st;
  if (!x || !wgate || !wup || !out) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(wgate) || !aligned16(wup)) return CATS_ERR_ALIGN;
  RowsArgs a;
  fill_rows(a, x, wgate, H, I, B, dtype);
  a.w2 = (const u32x4*)wup;
  a.zt_out = out;
  a.flag_out = flag_out;
  a.t = round_through(dtype, threshold);
  if (joined_takes(dtype, a)) return do_joined_gate_up(a, (hipStream_t)stream);
  return wide ? rows_wide(a, dtype, stream) : do_rows(kGateUp, dtype, a, (hipStream_t)stream);
}

static int mlp_pass(const void* x, const void* wgate, const void* wup, const void* wdown_t, void* y_out, float* y_f32,
             uint8_t* flag_out, int32_t* count_out, int B, int H, int I, int dtype, float threshold, void* ws,
             size_t ws_bytes, void* stream, int stage = 0) {
  int st = check_common(B, H, I, dtype);
  if (st) return st;
  if (!x || !wgate || !wup || !wdown_t || ((y_f32 == nullptr) == (y_out == nullptr))) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(wgate) || !aligned16(wup) || !aligned16(wdown_t)) return CATS_ERR_ALIGN;
  WsLayout l;
  st = check_ws(ws, ws_bytes, H, I, l);
  if (st) return st;
  FusedArgs f;
  int grid = 0;
  RowsArgs a;
  fill_rows(a, x, wgate, H, I, B, dtype);
  a.w2 = (const u32x4*)wup;
  a.flag_out = flag_out;
  a.t = round_through(dtype, threshold);
  bool mma = false;
  if (small_takes(a, dtype, l.room(), mma, grid))
    return do_small(a, mma, grid, stage, wdown_t, y_out, nullptr, y_f32, count_out, dtype, (char*)ws, l, (hipStream_t)stream);
  if (fused_eligible(B, H, I, dtype, f, grid)) {
    f.x = (const u32x4*)x;
    f.wg = (const u32x4*)wgate;
    f.wu = (const u32x4*)wup;
    f.wd = (const u32x4*)wdown_t;
    f.flag_out = flag_out;
    f.t = a.t;
    return do_fused(f, grid, stage, y_out, nullptr, count_out, dtype, (char*)ws, l, (hipStream_t)stream, y_f32);
  }
  a.z32_out = (float*)((char*)ws + l.z32);
  a.mask_out = (uint8_t*)ws + l.mask;
  a.ubytes_out = (uint8_t*)ws + l.ubytes;
  const bool joined = joined_takes(dtype, a);
  l.mask_bytes = joined || rows_mask_is_bytes(kGateUp, dtype, a);
  if (stage != 2) {
    st = joined ? do_joined(a, (float*)((char*)ws + l.zt), a.z32_out, (hipStream_t)stream) : do_rows(kGateUp, dtype, a, (hipStream_t)stream);
    if (st) return st;
  }
  if (stage == 1) return CATS_OK;
  float* acc = y_f32;
  return do_down(a.z32_out, true, wdown_t, acc, y_out, count_out, B, H, I, dtype, (char*)ws, l, (hipStream_t)stream);
}


// Whole MLP for 9..16 rows with W_gate and W_up read once: one matrix-core gate + up launch over all rows (two groups of
// eight), then the sparse down pass per group of eight rows over the union mask of all rows.  Returns kNotTaken when the
// row length rules the one-pass kernel out (two x operands have to fit in LDS), or the A/B knob.
// norm_weight / residual / next: the layer-tail variants (x is then h); all optional.
static int mlp_wide(const void* x, const void* norm_weight, float eps, const void* wgate, const void* wup, const void* wdown_t, void* y_out,
                    float* y_f32, uint8_t* flag_out, int32_t* count_out, bool residual, const NextNorm& next, int B, int H, int I, int dtype,
                    float threshold, void* ws, size_t ws_bytes, void* stream) {
  if (B <= kKernelBatch || B > CATS_MAX_BATCH) return kNotTaken;
  int st = check_common(kKernelBatch, H, I, dtype);
  if (st) return st;
  if (!x || !wgate || !wup || !wdown_t || ((y_f32 == nullptr) == (y_out == nullptr))) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(wgate) || !aligned16(wup) || !aligned16(wdown_t)) return CATS_ERR_ALIGN;
  WsLayout l;
  st = check_ws(ws, ws_bytes, H, I, l);
  if (st) return st;
  RowsArgs a;
  fill_rows(a, x, wgate, H, I, B, dtype);
  a.w2 = (const u32x4*)wup;
  a.flag_out = flag_out;
  a.t = round_through(dtype, threshold);
  a.norm_w = (const u32x4*)norm_weight;
  a.norm_eps = eps;
  bool mma = false;
  int grid = 0;
  if (small_takes(a, dtype, l.room(), mma, grid))
    return do_small(a, mma, grid, 0, wdown_t, y_out, residual ? x : nullptr, y_f32, count_out, dtype, (char*)ws, l, (hipStream_t)stream, next);
  a.z32_out = (float*)((char*)ws + l.z32);
  a.mask_out = (uint8_t*)ws + l.mask;
  a.ubytes_out = (uint8_t*)ws + l.ubytes;
  l.mask_bytes = true;  // the matrix-core kernel or nothing
  st = joined_takes(dtype, a) ? do_joined(a, (float*)((char*)ws + l.zt), a.z32_out, (hipStream_t)stream) : rows_wide(a, dtype, stream);
  if (st) return st;  // an error, or kNotTaken
  // all rows in one pass over W_down^T where the matrix-core down kernel takes the shape, else a pass per eight rows
  st = do_down(a.z32_out, true, wdown_t, y_f32, y_out, count_out, B, H, I, dtype, (char*)ws, l, (hipStream_t)stream, residual ? x : nullptr,
               nullptr, nullptr, 0, nullptr, next);
  if (st != kNotTaken) return st;
  const size_t sz = esz(dtype);
  for (int b0 = 0; b0 < B; b0 += kKernelBatch) {
    const int nb = B - b0 < kKernelBatch ? B - b0 : kKernelBatch;
    NextNorm nx = next;
    if (nx.out) nx.out = at_bytes(nx.out, (size_t)b0 * H * sz);
    st = do_down(a.z32_out + (size_t)b0 * I, true, wdown_t, (float*)at_bytes((void*)y_f32, (size_t)b0 * H * 4), at_bytes(y_out, (size_t)b0 * H * sz),
                 b0 == 0 ? count_out : nullptr, nb, H, I, dtype, (char*)ws, l, (hipStream_t)stream,
                 residual ? at_cbytes(x, (size_t)b0 * H * sz) : nullptr, nullptr, nullptr, 0, nullptr, nx);
    if (st) return st;
  }
  return CATS_OK;
}

// B above kKernelBatch: all rows in one pass over both matrices where the matrix-core kernels take the call, else kNotTaken.
static int up_down_pass(const void* x, const void* a_in, const void* wup, const void* wdown_t, void* y_out, int B, int H, int I,
                        int dtype, float threshold, void* ws, size_t ws_bytes, void* stream) {
  const bool wide = B > kKernelBatch;
  if (wide && (B > CATS_MAX_BATCH || dtype == CATS_F32)) return kNotTaken;
  int st = check_common(wide ? kKernelBatch : B, H, I, dtype);
  if (st) return st;
  if (!x || !a_in || !wup || !wdown_t || !y_out) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(wup) || !aligned16(wdown_t)) return CATS_ERR_ALIGN;
  WsLayout l;
  st = check_ws(ws, ws_bytes, H, I, l);
  if (st) return st;
  FusedArgs f;
  int grid = 0;
  if (fused_eligible(B, H, I, dtype, f, grid)) {
    f.x = (const u32x4*)x;
    f.a_in = a_in;
    f.wu = (const u32x4*)wup;
    f.wd = (const u32x4*)wdown_t;
    f.t = round_through(dtype, threshold);
    return do_fused(f, grid, 0, y_out, nullptr, nullptr, dtype, (char*)ws, l, (hipStream_t)stream);
  }
  RowsArgs a;
  fill_rows(a, x, wup, H, I, B, dtype);
  a.a_in = a_in;
  a.flag_in = nullptr;  // flags = |a| > t, computed where a is read
  a.t = round_through(dtype, threshold);
  a.z32_out = (float*)((char*)ws + l.z32);
  a.mask_out = (uint8_t*)ws + l.mask;
  a.ubytes_out = (uint8_t*)ws + l.ubytes;
  l.mask_bytes = rows_mask_is_bytes(kUp, dtype, a);
  if (wide && !l.mask_bytes) return kNotTaken;  // only the matrix-core up kernel takes more than eight rows
  st = do_rows(kUp, dtype, a, (hipStream_t)stream);
  if (st) return st;
  st = do_down(a.z32_out, true, wdown_t, nullptr, y_out, nullptr, B, H, I, dtype, (char*)ws, l, (hipStream_t)stream);
  if (st != kNotTaken) return st;
  // z of all rows is there: the down pass per group of eight rows over the union of all flags
  const size_t sz = esz(dtype);
  for (int b0 = 0; b0 < B; b0 += kKernelBatch) {
    const int nb = B - b0 < kKernelBatch ? B - b0 : kKernelBatch;
    st = do_down(a.z32_out + (size_t)b0 * I, true, wdown_t, nullptr, at_bytes(y_out, (size_t)b0 * H * sz), nullptr, nb, H, I, dtype, (char*)ws, l,
                 (hipStream_t)stream);
    if (st) return st;
  }
  return CATS_OK;
}

static int mlp_norm_residual_pass(const void* h, const void* norm_weight, float eps, const void* wgate, const void* wup,
                           const void* wdown_t, void* out, int B, int H, int I, int dtype, float threshold, void* ws,
                           size_t ws_bytes, void* stream, const NextNorm& next = NextNorm()) {
  int st = check_common(B, H, I, dtype);
  if (st) return st;
  if (!h || !norm_weight || !wgate || !wup || !wdown_t || !out) return CATS_ERR_NULL;
  if (!aligned16(h) || !aligned16(norm_weight) || !aligned16(wgate) || !aligned16(wup) || !aligned16(wdown_t)) return CATS_ERR_ALIGN;
  // the norm works on the LDS copy of h: same bound as the kernels' own x staging
  if ((size_t)batch_template(B) * (((size_t)H * elem_size(dtype) + 8191) / 8192 * 8192) > kStagedMaxBytes) return CATS_ERR_SHAPE;
  WsLayout l;
  st = check_ws(ws, ws_bytes, H, I, l);
  if (st) return st;
  RowsArgs a;
  fill_rows(a, h, wgate, H, I, B, dtype);
  a.w2 = (const u32x4*)wup;
  a.t = round_through(dtype, threshold);
  a.norm_w = (const u32x4*)norm_weight;
  a.norm_eps = eps;
  FusedArgs f;
  int grid = 0;
  bool mma = false;
  if (small_takes(a, dtype, l.room(), mma, grid))
    return do_small(a, mma, grid, 0, wdown_t, out, h, nullptr, nullptr, dtype, (char*)ws, l, (hipStream_t)stream, next);
  if (fused_eligible(B, H, I, dtype, f, grid)) {
    f.x = (const u32x4*)h;
    f.wg = (const u32x4*)wgate;
    f.wu = (const u32x4*)wup;
    f.wd = (const u32x4*)wdown_t;
    f.t = a.t;
    f.norm_w = (const u32x4*)norm_weight;
    f.norm_eps = eps;
    return do_fused(f, grid, 0, out, h, nullptr, dtype, (char*)ws, l, (hipStream_t)stream, nullptr, next);
  }
  a.z32_out = (float*)((char*)ws + l.z32);
  a.mask_out = (uint8_t*)ws + l.mask;
  a.ubytes_out = (uint8_t*)ws + l.ubytes;
  l.mask_bytes = rows_mask_is_bytes(kGateUp, dtype, a);
  st = do_rows(kGateUp, dtype, a, (hipStream_t)stream);
  if (st) return st;
  return do_down(a.z32_out, true, wdown_t, nullptr, out, nullptr, B, H, I, dtype, (char*)ws, l, (hipStream_t)stream, h, nullptr, nullptr, 0,
                 nullptr, next);
}

static int mlp_rowmajor_down_pass(const void* x, const void* wgate, const void* wup, const void* wdown, void* y_out, int B, int H,
                           int I, int dtype, float threshold, void* ws, size_t ws_bytes, void* stream) {
  int st = check_common(B, H, I, dtype);
  if (st) return st;
  if (!x || !wgate || !wup || !wdown || !y_out) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(wgate) || !aligned16(wup) || !aligned16(wdown)) return CATS_ERR_ALIGN;
  if (((size_t)I * elem_size(dtype)) % 16 != 0) return CATS_ERR_ALIGN;
  WsLayout l;
  st = check_ws(ws, ws_bytes, H, I, l);
  if (st) return st;
  RowsArgs a;
  fill_rows(a, x, wgate, H, I, B, dtype);
  a.w2 = (const u32x4*)wup;
  a.zt_out = (char*)ws + l.zt;
  a.t = round_through(dtype, threshold);
  st = joined_takes(dtype, a) ? do_joined(a, (float*)((char*)ws + l.z32), (float*)a.zt_out, (hipStream_t)stream) : do_rows(kGateUp, dtype, a, (hipStream_t)stream);
  if (st) return st;
  RowsArgs g;
  fill_rows(g, (char*)ws + l.zt, wdown, I, H, B, dtype);
  g.zt_out = y_out;
  return do_rows(kGemv, dtype, g, (hipStream_t)stream);
}

// The same for 9..16 rows with every matrix read once: the matrix-core gate + up launch over all rows, then the matrix-core
// GEMV over all rows.  kNotTaken when the type or the shape rules either kernel out.
static int mlp_rowmajor_down_wide(const void* x, const void* wgate, const void* wup, const void* wdown, void* y_out, int B, int H,
                                  int I, int dtype, float threshold, void* ws, size_t ws_bytes, void* stream) {
  if (B <= kKernelBatch || B > CATS_MAX_BATCH) return kNotTaken;
  int st = check_common(kKernelBatch, H, I, dtype);
  if (st) return st;
  if (!x || !wgate || !wup || !wdown || !y_out) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(wgate) || !aligned16(wup) || !aligned16(wdown)) return CATS_ERR_ALIGN;
  if (((size_t)I * elem_size(dtype)) % 16 != 0) return CATS_ERR_ALIGN;
  WsLayout l;
  st = check_ws(ws, ws_bytes, H, I, l);
  if (st) return st;
  char* z = (char*)ws + (dtype == CATS_F32 ? l.z32 : l.zt);  // 16 rows of a 16-bit type fill the region of 8 rows of fp32
  RowsArgs a;
  fill_rows(a, x, wgate, H, I, B, dtype);
  a.w2 = (const u32x4*)wup;
  a.zt_out = z;
  a.t = round_through(dtype, threshold);
  RowsArgs g;
  fill_rows(g, z, wdown, I, H, B, dtype);
  g.zt_out = y_out;
  g.mma = g_tuning.gate_variant >= 0;
  // the GEMV first: nothing may have been launched when the call falls back to two passes
  if (!rows_take_mma(kGemv, dtype, kKernelBatch, g)) return kNotTaken;
  st = joined_takes(dtype, a) ? do_joined(a, (float*)((char*)ws + l.zt), (float*)z, (hipStream_t)stream) : rows_wide(a, dtype, stream);
  if (st) return st;  // an error, or kNotTaken
  return do_rows(kGemv, dtype, g, (hipStream_t)stream);
}

// ---- public entry points: up to CATS_MAX_BATCH rows, in passes of kKernelBatch rows over the weights --------------
// Decode batches of 1..8 rows are one pass.  Larger ones (the reference's kernels go to 16) re-read the weights per
// pass; at that size the union of the masks is dense anyway and the path has nothing left to skip.


int cats_gate_flag(const void* x, const void* wgate, void* a_out, uint8_t* flag_out, int B, int H, int I, int dtype,
                   float threshold, void* stream) {
  const size_t sz = esz(dtype);
  if (B > kKernelBatch)
    if (const int st = gate_flag_pass(x, wgate, a_out, flag_out, B, H, I, dtype, threshold, stream); st != kNotTaken) return st;
  return in_passes(B, [&](size_t b0, int nb) {
    return gate_flag_pass(at_cbytes(x, b0 * H * sz), wgate, at_bytes(a_out, b0 * I * sz), (uint8_t*)at_bytes((void*)flag_out, b0 * I), nb, H, I,
                          dtype, threshold, stream);
  });
}

int cats_up_flag(const void* x, const void* wup, const void* a_in, const uint8_t* flag, void* out, int out_is_f32, int B,
                 int H, int I, int dtype, void* stream) {
  const size_t sz = esz(dtype);
  if (B > kKernelBatch)
    if (const int st = up_flag_pass(x, wup, a_in, flag, out, out_is_f32, B, H, I, dtype, stream); st != kNotTaken) return st;
  return in_passes(B, [&](size_t b0, int nb) {
    return up_flag_pass(at_cbytes(x, b0 * H * sz), wup, at_cbytes(a_in, b0 * I * sz), (const uint8_t*)at_cbytes((const void*)flag, b0 * I),
                        at_bytes(out, b0 * I * (out_is_f32 ? 4 : sz)), out_is_f32, nb, H, I, dtype, stream);
  });
}

int cats_down_flag(const void* z, const void* wdown_t, const uint8_t* flag, float* y_f32, void* y_out, int B, int H, int I,
                   int dtype, void* ws, size_t ws_bytes, void* stream) {
  const size_t sz = esz(dtype);
  if (B > kKernelBatch)
    if (const int st = down_flag_pass(z, wdown_t, flag, y_f32, y_out, B, H, I, dtype, ws, ws_bytes, stream); st != kNotTaken) return st;
  return in_passes(B, [&](size_t b0, int nb) {
    return down_flag_pass(at_cbytes(z, b0 * I * sz), wdown_t, (const uint8_t*)at_cbytes((const void*)flag, b0 * I),
                          (float*)at_bytes((void*)y_f32, b0 * H * 4), at_bytes(y_out, b0 * H * sz), nb, H, I, dtype, ws, ws_bytes, stream);
  });
}

int cats_gate_up(const void* x, const void* wgate, const void* wup, void* out, uint8_t* flag_out, int B, int H, int I,
                 int dtype, float threshold, void* stream) {
  const size_t sz = esz(dtype);
  if (B > kKernelBatch)
    if (const int st = gate_up_pass(x, wgate, wup, out, flag_out, B, H, I, dtype, threshold, stream); st != kNotTaken) return st;
  return in_passes(B, [&](size_t b0, int nb) {
    return gate_up_pass(at_cbytes(x, b0 * H * sz), wgate, wup, at_bytes(out, b0 * I * sz), (uint8_t*)at_bytes((void*)flag_out, b0 * I), nb, H, I,
                        dtype, threshold, stream);
  });
}

int cats_mlp(const void* x, const void* wgate, const void* wup, const void* wdown_t, void* y_out, float* y_f32,
             uint8_t* flag_out, int32_t* count_out, int B, int H, int I, int dtype, float threshold, void* ws,
             size_t ws_bytes, void* stream) {
  const size_t sz = esz(dtype);
  if (const int st = mlp_wide(x, nullptr, 0.f, wgate, wup, wdown_t, y_out, y_f32, flag_out, count_out, false, NextNorm(), B, H, I, dtype, threshold,
                              ws, ws_bytes, stream);
      st != kNotTaken)
    return st;
  const bool union_count = count_out && B > kKernelBatch;  // a pass counts its own rows only: count the union of the flags instead
  if (union_count && !flag_out) {
    // no flags asked for: the passes write them into `atmp`, which no pass of at most kKernelBatch rows uses (do_joined's sums of
    // eight rows fill `zt`; those of more rows go on into `atmp`, but then there are no passes)
    WsLayout l;
    if (int st = check_common(kKernelBatch, H, I, dtype)) return st;
    if (int st = check_ws(ws, ws_bytes, H, I, l)) return st;
    flag_out = (uint8_t*)ws + l.atmp;  // 8 * I * 4 bytes hold CATS_MAX_BATCH * I flags
  }
  int st = in_passes(B, [&](size_t b0, int nb) {
    return mlp_pass(at_cbytes(x, b0 * H * sz), wgate, wup, wdown_t, at_bytes(y_out, b0 * H * sz), (float*)at_bytes((void*)y_f32, b0 * H * 4),
                    (uint8_t*)at_bytes((void*)flag_out, b0 * I), union_count ? nullptr : count_out, nb, H, I, dtype, threshold, ws, ws_bytes,
                    stream);
  });
  if (st || !union_count) return st;
  return launch_kernel(union_count_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, (const uint8_t*)flag_out, B, I, count_out) == hipSuccess
             ? CATS_OK
             : CATS_ERR_LAUNCH;
}

int cats_mlp_stage(int stage, const void* x, const void* wgate, const void* wup, const void* wdown_t, void* y_out, int B, int H, int I,
                   int dtype, float threshold, void* ws, size_t ws_bytes, void* stream) {
  if (stage != 1 && stage != 2) return CATS_ERR_SHAPE;
  if (B > kKernelBatch) return CATS_ERR_BATCH;
  return mlp_pass(x, wgate, wup, wdown_t, y_out, nullptr, nullptr, nullptr, B, H, I, dtype, threshold, ws, ws_bytes, stream, stage);
}

int cats_up_index(const void* x, const void* w, const int64_t* idx, int M, const void* bias, const void* scale, int activation,
                  void* out, int B, int H, int Z, int dtype, void* stream) {
  if (M == 0) return (B >= 1 && B <= kKernelBatch) ? CATS_OK : CATS_ERR_BATCH;
  int st = check_common(B, H, Z, dtype);
  if (st) return st;
  if (M < 0 || activation < 0 || activation > 3) return CATS_ERR_SHAPE;
  if (!x || !w || !idx || !out) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(w)) return CATS_ERR_ALIGN;
  RowsArgs a;
  fill_rows(a, x, w, H, M, B, dtype);
  a.row_idx = idx;
  a.w_rows = Z;
  a.bias = bias;
  a.scale = scale;
  a.activation = activation;
  a.zt_out = out;
  return do_rows(kUpIndex, dtype, a, (hipStream_t)stream);
}

int cats_down_index(const void* z, const void* wdown_t, const int64_t* idx, int M, const void* bias, void* y_out, int B, int H, int Z,
                    int dtype, void* ws, size_t ws_bytes, void* stream) {
  int st = check_common(B, H, Z, dtype);
  if (st) return st;
  if (M < 0) return CATS_ERR_SHAPE;
  if (!wdown_t || !y_out || (M > 0 && (!z || !idx))) return CATS_ERR_NULL;
  if (!aligned16(wdown_t)) return CATS_ERR_ALIGN;
  WsLayout l;
  st = check_ws(ws, ws_bytes, H, Z, l);
  if (st) return st;
  if (M == 0) {
    // an empty list: y = bias or 0, written by the reduction over zero partials
    ReduceArgs r;
    memset(&r, 0, sizeof(r));
    r.partial = (float*)((char*)ws + l.partial);
    r.y_out = y_out;
    r.bias = bias;
    r.H = H;
    r.G = 0;
    r.BH = B * H;
    return do_reduce(r, dtype, (hipStream_t)stream);
  }
  return do_down(z, false, wdown_t, nullptr, y_out, nullptr, B, H, Z, dtype, (char*)ws, l, (hipStream_t)stream, nullptr, nullptr, idx, M, bias);
}

int cats_mlp_noalloc(const void* x, const void* wgate, const void* wup, const void* wdown_t, void* y_out, int B, int H, int I,
                     int dtype, float threshold, void* stream) {
  int st = check_common(B, H, I, dtype);
  if (st) return st;
  if (!x || !wgate || !wup || !wdown_t || !y_out) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(wgate) || !aligned16(wup) || !aligned16(wdown_t)) return CATS_ERR_ALIGN;
  FusedArgs f;
  int grid = 0;
  RowsArgs a;
  fill_rows(a, x, wgate, H, I, B, dtype);
  a.w2 = (const u32x4*)wup;
  a.t = round_through(dtype, threshold);
  bool mma = false;
  // Two launches, never one: calls that overlap on this GPU may spoil each other's sums, but a counter they left off zero would spoil
  // every call after them.
  if (B <= 2 && (size_t)B * H <= 8192 && small_takes(a, dtype, kScratchPartialBytes, mma, grid) && (size_t)grid * 4 <= kScratchCountBytes) {
    void* sp = nullptr;
    if (int e = scratch_address(&sp)) return e;
    return do_small(a, mma, grid, 0, wdown_t, y_out, nullptr, nullptr, nullptr, dtype, nullptr, WsLayout(), (hipStream_t)stream, NextNorm(), (float*)sp,
                    (int32_t*)((char*)sp + kScratchPartialBytes));
  }
  const bool ok = fused_eligible(B, H, I, dtype, f, grid, true);  // this entry point is the single-pass kernel or nothing
  // the stated limit (B * H <= 8192) whatever the grid turns out to be, and the actual footprint as a second check
  if (!ok || (size_t)B * H > 8192 || (size_t)grid * B * H * 4 > kScratchPartialBytes || (size_t)grid * 4 > kScratchCountBytes)
    return CATS_ERR_SCRATCH;
  void* sp = nullptr;
  st = scratch_address(&sp);
  if (st) return st;
  f.x = (const u32x4*)x;
  f.wg = (const u32x4*)wgate;
  f.wu = (const u32x4*)wup;
  f.wd = (const u32x4*)wdown_t;
  f.t = round_through(dtype, threshold);
  f.partial = (float*)sp;
  f.counts = (int32_t*)((char*)sp + kScratchPartialBytes);
  fused_enable_pool(f, grid, dtype, (int32_t*)((char*)sp + kScratchPartialBytes + kScratchCountBytes), kScratchPoolBytes);
  ReduceArgs r;
  memset(&r, 0, sizeof(r));
  r.partial = f.partial;
  r.counts = f.counts;
  r.y_out = y_out;
  r.H = H;
  r.G = grid;
  r.BH = B * H;
  const int bt = batch_template(B);
  hipError_t e;
  if (dtype == CATS_F16) e = launch_fused<F16>(bt, grid, 0, f, r, (hipStream_t)stream);
  else if (dtype == CATS_BF16) e = launch_fused<BF16>(bt, grid, 0, f, r, (hipStream_t)stream);
  else e = launch_fused<F32>(bt, grid, 0, f, r, (hipStream_t)stream);
  return e == hipSuccess ? CATS_OK : CATS_ERR_LAUNCH;
}

int cats_up_down(const void* x, const void* a, const void* wup, const void* wdown_t, void* y_out, int B, int H, int I,
                 int dtype, float threshold, void* ws, size_t ws_bytes, void* stream) {
  const size_t sz = esz(dtype);
  if (B > kKernelBatch)
    if (const int st = up_down_pass(x, a, wup, wdown_t, y_out, B, H, I, dtype, threshold, ws, ws_bytes, stream); st != kNotTaken) return st;
  return in_passes(B, [&](size_t b0, int nb) {
    return up_down_pass(at_cbytes(x, b0 * H * sz), at_cbytes(a, b0 * I * sz), wup, wdown_t, at_bytes(y_out, b0 * H * sz), nb, H, I, dtype,
                        threshold, ws, ws_bytes, stream);
  });
}

int cats_mlp_norm_residual(const void* h, const void* norm_weight, float eps, const void* wgate, const void* wup,
                           const void* wdown_t, void* out, int B, int H, int I, int dtype, float threshold, void* ws,
                           size_t ws_bytes, void* stream) {
  const size_t sz = esz(dtype);
  if (B > kKernelBatch && norm_weight && aligned16(norm_weight)) {
    // in place (out == h) is fine here too: the gate + up launch has read all of h before the down passes write any row
    if (const int st = mlp_wide(h, norm_weight, eps, wgate, wup, wdown_t, out, nullptr, nullptr, nullptr, true, NextNorm(), B, H, I, dtype,
                                threshold, ws, ws_bytes, stream);
        st != kNotTaken)
      return st;
  }
  return in_passes(B, [&](size_t b0, int nb) {
    return mlp_norm_residual_pass(at_cbytes(h, b0 * H * sz), norm_weight, eps, wgate, wup, wdown_t, at_bytes(out, b0 * H * sz), nb, H, I, dtype,
                                  threshold, ws, ws_bytes, stream);
  });
}

int cats_mlp_norm_residual_norm(const void* h, const void* norm_weight, float eps, const void* wgate, const void* wup,
                                const void* wdown_t, void* out, const void* next_norm_weight, float next_eps, void* next_out, int B,
                                int H, int I, int dtype, float threshold, void* ws, size_t ws_bytes, void* stream) {
  if (!next_norm_weight || !next_out) return CATS_ERR_NULL;
  if (!aligned16(next_norm_weight) || !aligned16(next_out)) return CATS_ERR_ALIGN;
  if (H % kReduceCols != 0) return CATS_ERR_SHAPE;
  const size_t sz = esz(dtype);
  if (B > kKernelBatch && norm_weight && aligned16(norm_weight)) {
    NextNorm next;
    next.w = next_norm_weight;
    next.eps = next_eps;
    next.out = next_out;
    if (const int st = mlp_wide(h, norm_weight, eps, wgate, wup, wdown_t, out, nullptr, nullptr, nullptr, true, next, B, H, I, dtype, threshold,
                                ws, ws_bytes, stream);
        st != kNotTaken)
      return st;
  }
  return in_passes(B, [&](size_t b0, int nb) {
    NextNorm next;
    next.w = next_norm_weight;
    next.eps = next_eps;
    next.out = at_bytes(next_out, b0 * H * sz);
    return mlp_norm_residual_pass(at_cbytes(h, b0 * H * sz), norm_weight, eps, wgate, wup, wdown_t, at_bytes(out, b0 * H * sz), nb, H, I, dtype,
                                  threshold, ws, ws_bytes, stream, next);
  });
}

int cats_mlp_rowmajor_down(const void* x, const void* wgate, const void* wup, const void* wdown, void* y_out, int B, int H,
                           int I, int dtype, float threshold, void* ws, size_t ws_bytes, void* stream) {
  const size_t sz = esz(dtype);
  if (const int st = mlp_rowmajor_down_wide(x, wgate, wup, wdown, y_out, B, H, I, dtype, threshold, ws, ws_bytes, stream); st != kNotTaken) return st;
  return in_passes(B, [&](size_t b0, int nb) {
    return mlp_rowmajor_down_pass(at_cbytes(x, b0 * H * sz), wgate, wup, wdown, at_bytes(y_out, b0 * H * sz), nb, H, I, dtype, threshold, ws,
                                  ws_bytes, stream);
  });
}

int cats_mlp_gate_cols(const void* x, const void* wgate_hi, const void* wup, const void* wdown_t, void* y_out, int H, int I, int dtype,
                       float threshold, void* ws, size_t ws_bytes, void* stream) {
  int st = check_common(1, H, I, dtype);
  if (st) return st;
  if (I < vec_elems(dtype)) return CATS_ERR_SHAPE;
  if (!x || !wgate_hi || !wup || !wdown_t || !y_out) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(wup) || !aligned16(wdown_t) || ((uintptr_t)wgate_hi & (esz(dtype) - 1)) != 0) return CATS_ERR_ALIGN;
  WsLayout l;
  st = check_ws(ws, ws_bytes, H, I, l);
  if (st) return st;
  FusedArgs f;
  int grid = 0;
  const bool single_pass = fused_eligible(1, H, I, dtype, f, grid);
  if (!single_pass) {  // the separate kernels, checked before anything is launched
    const int nslab = (H / vec_elems(dtype) + kWave - 1) / kWave;
    if (nslab > kMaxSlabs || down_chunk(I, nslab, 1) == 0 || (size_t)I * esz(dtype) > l.mask - l.partial) return CATS_ERR_SHAPE;
  }
  GateColsArgs g;
  g.x = x;
  g.w = wgate_hi;
  g.partial = (float*)((char*)ws + l.zt);  // that region and the next, 16 * I floats: nothing else of this call uses them
  g.H = H;
  g.I = I;
  const int slab = kWave * vec_elems(dtype);
  g.nslab = (I + slab - 1) / slab;
  int groups = current_device_cus() / g.nslab;  // one workgroup of sixteen waves per CU, all at once
  if (groups > kGateColsMaxGroups) groups = kGateColsMaxGroups;
  if (groups > (H + kGateColsWaves - 1) / kGateColsWaves) groups = (H + kGateColsWaves - 1) / kGateColsWaves;
  if (groups < 1) groups = 1;
  g.rows_per = (H + groups - 1) / groups;
  groups = (H + g.rows_per - 1) / g.rows_per;
  hipStream_t s = (hipStream_t)stream;
  hipError_t e = dtype == CATS_F16    ? launch_gate_cols<F16>(g, groups, s)
                 : dtype == CATS_BF16 ? launch_gate_cols<BF16>(g, groups, s)
                                      : launch_gate_cols<F32>(g, groups, s);
  if (e != hipSuccess) return CATS_ERR_LAUNCH;
  if (single_pass) {
    f.x = (const u32x4*)x;
    f.a_part = g.partial;
    f.a_groups = groups;
    f.wu = (const u32x4*)wup;
    f.wd = (const u32x4*)wdown_t;
    f.t = round_through(dtype, threshold);
    return do_fused(f, grid, 0, y_out, nullptr, nullptr, dtype, (char*)ws, l, s);
  }
  // Rows too long for the single-pass kernel: the activations as the separate kernels take them.  They lie where the down
  // pass, which runs after their last reader, will leave its partial sums.
  void* a = (char*)ws + l.partial;
  e = dtype == CATS_F16    ? launch_gate_cols_finish<F16>(g, groups, a, s)
      : dtype == CATS_BF16 ? launch_gate_cols_finish<BF16>(g, groups, a, s)
                           : launch_gate_cols_finish<F32>(g, groups, a, s);
  if (e != hipSuccess) return CATS_ERR_LAUNCH;
  return up_down_pass(x, a, wup, wdown_t, y_out, 1, H, I, dtype, threshold, ws, ws_bytes, stream);
}

int cats_silu_mask_mul(const void* gate, const void* up, void* z, size_t n, int dtype, float threshold, void* stream) {
  if (dtype != CATS_F16 && dtype != CATS_BF16 && dtype != CATS_F32) return CATS_ERR_DTYPE;
  if (n == 0) return CATS_OK;
  if (!gate || !up || !z) return CATS_ERR_NULL;
  if (!aligned16(gate) || !aligned16(up) || !aligned16(z)) return CATS_ERR_ALIGN;
  SiluMaskMulArgs a = {gate, up, z, n, round_through(dtype, threshold)};
  const hipError_t e = dtype == CATS_F16    ? launch_silu_mask_mul<F16>(a, (hipStream_t)stream)
                       : dtype == CATS_BF16 ? launch_silu_mask_mul<BF16>(a, (hipStream_t)stream)
                                            : launch_silu_mask_mul<F32>(a, (hipStream_t)stream);
  return e == hipSuccess ? CATS_OK : CATS_ERR_LAUNCH;
}

// The plan of the second product: what it needs in the scratch decides its size.
static PromptPlan prompt_up_plan(int M, int H, int I) { return prompt_plan(true, M, prompt_pitch(I), H, current_device_cus()); }
static PromptPlan prompt_down_plan(int M, int H, int I) { return prompt_plan(false, M, prompt_sum_pitch(H), I, current_device_cus()); }
static size_t prompt_z_bytes(int M, int I) { return ((size_t)M * prompt_pitch(I) * 2 + 255) / 256 * 256; }

static size_t prompt_bytes(const PromptPlan& down, int M, int H, int I) {
  return prompt_z_bytes(M, I) + (down.splits > 1 ? (size_t)down.splits * M * prompt_sum_pitch(H) * sizeof(float) : 0);
}

size_t cats_prompt_scratch_bytes(int M, int H, int I) {
  if (M < 1 || M > CATS_PROMPT_MAX_TOKENS || H < 8 || I < 8 || H > (1 << 28) || I > (1 << 28)) return 0;
  return prompt_bytes(prompt_down_plan(M, H, I), M, H, I);
}

int cats_prompt_plan(int product, int M, int H, int I, int* plan) {
  if (!plan) return CATS_ERR_NULL;
  if ((product != 1 && product != 2) || M < 1 || M > CATS_PROMPT_MAX_TOKENS || H < 8 || I < 8 || H > (1 << 28) || I > (1 << 28)) return CATS_ERR_SHAPE;
  const PromptPlan p = product == 1 ? prompt_up_plan(M, H, I) : prompt_down_plan(M, H, I);
  const int v[6] = {p.tile, p.mblocks, p.nblocks, p.steps, p.splits, prompt_steps_ahead(p, current_device_cus())};
  memcpy(plan, v, sizeof(v));
  return CATS_OK;
}

int cats_prompt_mlp(const void* x, const void* wgate, const void* wup, const void* wdown, void* y_out, int M, int H, int I, int dtype,
                    float threshold, void* scratch, size_t scratch_bytes, void* stream) {
  if (dtype != CATS_F16 && dtype != CATS_BF16) return CATS_ERR_DTYPE;
  // the kernels count a matrix's bytes in 32 bits; the tiles' rounding must not overflow either
  const long long limit = 0xffffffffll;
  if (M < 1 || H < 8 || I < 8 || M > CATS_PROMPT_MAX_TOKENS || I > (1 << 28) || H > (1 << 28) || 2ll * H * prompt_pitch(I) > limit ||
      2ll * M * H > limit || 2ll * M * prompt_pitch(I) > limit)
    return CATS_ERR_SHAPE;
  if (!x || !wgate || !wup || !wdown || !y_out) return CATS_ERR_NULL;
  for (const void* p : {x, wgate, wup, wdown})
    if ((uintptr_t)p & 1u) return CATS_ERR_ALIGN;
  if ((uintptr_t)y_out & 7u) return CATS_ERR_ALIGN;
  const PromptPlan second = prompt_down_plan(M, H, I);
  if (!scratch || ((uintptr_t)scratch & 255u) || scratch_bytes < prompt_bytes(second, M, H, I)) return CATS_ERR_WORKSPACE;
  const hipStream_t s = (hipStream_t)stream;
  const int pitch = prompt_pitch(I);
  PromptArgs a;
  memset(&a, 0, sizeof(a));
  a.x = x;
  a.w = wgate;
  a.w2 = wup;
  a.out = scratch;
  a.M = M; a.N = I; a.K = H;
  a.ldx = H; a.ldo = pitch;
  a.t = round_through(dtype, threshold);
  const PromptPlan first = prompt_up_plan(M, H, I);
  hipError_t e = dtype == CATS_F16 ? launch_prompt<F16>(true, first, a, s) : launch_prompt<BF16>(true, first, a, s);
  if (e != hipSuccess) return CATS_ERR_LAUNCH;
  float* partial = (float*)((char*)scratch + prompt_z_bytes(M, I));
  a.x = scratch;
  a.w = wdown;
  a.w2 = nullptr;
  a.N = H; a.K = I;
  a.ldx = pitch;
  a.out = second.splits > 1 ? (void*)partial : y_out;
  a.ldo = second.splits > 1 ? prompt_sum_pitch(H) : H;
  e = dtype == CATS_F16 ? launch_prompt<F16>(false, second, a, s) : launch_prompt<BF16>(false, second, a, s);
  if (e != hipSuccess) return CATS_ERR_LAUNCH;
  if (second.splits == 1) return CATS_OK;
  const PromptSumArgs r = {partial, y_out, M, H, prompt_sum_pitch(H), second.splits};
  e = dtype == CATS_F16 ? launch_prompt_sum<F16>(r, s) : launch_prompt_sum<BF16>(r, s);
  return e == hipSuccess ? CATS_OK : CATS_ERR_LAUNCH;
}

static int do_proj(int mode, int dtype, const ProjArgs& a, hipStream_t s) {
  const int bt = batch_template(a.r.nb);
  const hipError_t e = dtype == CATS_F16    ? launch_proj<F16>(mode, bt, a, s)
                       : dtype == CATS_BF16 ? launch_proj<BF16>(mode, bt, a, s)
                                            : launch_proj<F32>(mode, bt, a, s);
  return e == hipSuccess ? CATS_OK : CATS_ERR_LAUNCH;
}

// x of all rows is staged on chip whole
static int check_proj(int B, int K, int N, int dtype) {
  if (int st = check_common(B, K, N, dtype)) return st;
  const int vecs = K / vec_elems(dtype);
  return proj_lds_bytes(batch_template(B), (vecs + kWave - 1) / kWave) <= kStagedMaxBytes ? CATS_OK : CATS_ERR_SHAPE;
}

int cats_linear(const void* x, const void* norm_weight, float eps, const void* w, const void* residual, void* out, int B, int K, int N,
                int dtype, void* stream) {
  if (int st = check_proj(B, K, N, dtype)) return st;
  if (!x || !w || !out) return CATS_ERR_NULL;
  if (!aligned16(x) || !aligned16(w) || !aligned16(norm_weight)) return CATS_ERR_ALIGN;
  ProjArgs a;
  memset(&a, 0, sizeof(a));
  fill_rows(a.r, x, w, K, N, B, dtype);
  a.r.norm_w = (const u32x4*)norm_weight;
  a.r.norm_eps = eps;
  a.r.zt_out = out;
  a.residual = residual;
  return do_proj(residual ? kProjAdd : kProjPlain, dtype, a, (hipStream_t)stream);
}

int cats_attention_step(const void* h, const void* x, const void* norm_weight, float eps, const void* wq, const void* wk, const void* wv,
                        const void* wo, void* k_cache, void* v_cache, const void* cos_table, const void* sin_table, const int64_t* position,
                        float* q_scratch, void* attn_scratch, void* out, int B, int H, int heads, int max_len, int dtype, void* stream) {
  if (int st = check_proj(B, H, H, dtype)) return st;
  if (heads < 1 || max_len < 1 || H % heads != 0) return CATS_ERR_SHAPE;
  const int hd = H / heads, lanes = hd / vec_elems(dtype);  // of a cache slot: a power of two, so that lane groups tile a wave
  if (hd % vec_elems(dtype) != 0 || lanes < 2 || lanes > 32 || (lanes & (lanes - 1)) != 0) return CATS_ERR_SHAPE;
  if (!h || !x || !wq || !wk || !wv || !wo || !k_cache || !v_cache || !cos_table || !sin_table || !position || !q_scratch || !attn_scratch || !out)
    return CATS_ERR_NULL;
  for (const void* p : {x, norm_weight, wq, wk, wv, wo, (const void*)k_cache, (const void*)v_cache, (const void*)attn_scratch})
    if (!aligned16(p)) return CATS_ERR_ALIGN;
  ProjArgs a;
  memset(&a, 0, sizeof(a));
  fill_rows(a.r, x, wq, H, H, B, dtype);
  a.r.norm_w = (const u32x4*)norm_weight;
  a.r.norm_eps = eps;
  a.wk = (const u32x4*)wk;
  a.wv = (const u32x4*)wv;
  a.q_out = q_scratch;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.cos_t = cos_table;
  a.sin_t = sin_table;
  a.pos = position;
  a.half = hd / 2;
  a.heads = heads;
  a.max_len = max_len;
  if (int st = do_proj(kProjQkv, dtype, a, (hipStream_t)stream)) return st;
  AttnArgs t;
  t.q = q_scratch;
  t.k = (const u32x4*)k_cache;
  t.v = (const u32x4*)v_cache;
  t.pos = position;
  t.out = attn_scratch;
  t.scale = 1.44269504088896341f / sqrtf((float)hd);
  t.max_len = max_len;
  t.pairs = B * heads;
  t.next = (const u32x4*)wo;
  t.piece_vecs = H / vec_elems(dtype);
  const size_t vecs = (size_t)H * t.piece_vecs;
  t.next_vecs = (unsigned)(vecs < kAttnAheadVecs ? vecs : kAttnAheadVecs);
  const hipError_t e = dtype == CATS_F16    ? launch_attn<F16>(hd, B, t, (hipStream_t)stream)
                       : dtype == CATS_BF16 ? launch_attn<BF16>(hd, B, t, (hipStream_t)stream)
                                            : launch_attn<F32>(hd, B, t, (hipStream_t)stream);
  if (e != hipSuccess) return CATS_ERR_LAUNCH;
  return cats_linear(attn_scratch, nullptr, 0.f, wo, h, out, B, H, H, dtype, stream);
}

}  // extern "C"

// Kernel instantiations for one dtype.  Compiled three times (-DCATS_DT=F16 / BF16 / F32) so the
// translation units build in parallel.
#include "cats_launch.h"
#include "cats_proj_mma.h"
#include "cats_rows_mma.h"

#ifndef CATS_DT
#error "compile with -DCATS_DT=F16|BF16|F32"
#endif

namespace cats {

namespace {

constexpr int kR = 2;    // rows per wave per pass
constexpr int kCB = 8;   // 64-lane chunks whose loads are issued together: 8 x 16 B per lane per row
constexpr int kDownU = 8;  // rows in flight per lane in the down kernel

// Workgroup width by batch: x is staged per workgroup, so wider batches share it across more waves.
template <int B> struct WavesFor { static constexpr int value = B <= 2 ? 4 : 8; };

template <class DT, int B, bool FULL, int MODE, bool XLDS>
hipError_t launch_rows_one(const RowsArgs& a, hipStream_t stream) {
  constexpr int WAVES = WavesFor<B>::value;
  auto kern = rows_kernel<DT, B, kR, kCB, FULL, MODE, XLDS, WAVES, true>;
  if constexpr (rows_norm_apart(MODE, B, XLDS))
    if (!a.norm_w && (sizeof(typename DT::st) == 4 || a.K <= 4096)) kern = rows_kernel<DT, B, kR, kCB, FULL, MODE, XLDS, WAVES, false>;
  const int rows_per_block = WAVES * kR;
  const int grid = (a.N + rows_per_block - 1) / rows_per_block;
  size_t lds = XLDS ? (size_t)B * ((a.nch + kCB - 1) / kCB * kCB) * kWave * sizeof(u32x4) : 0;
  if ((size_t)a.lds_floor > lds) lds = (size_t)a.lds_floor;
  if (hipError_t e = ensure_dynamic_lds((const void*)kern, lds); e != hipSuccess) return e;
  return launch_kernel(kern, dim3(grid), dim3(WAVES * kWave), lds, stream, a);
}

// Matrix-core passes over weight rows: one persistent workgroup per CU.
template <class DT>
struct MmaLaunch {
  static constexpr bool kHasUp = sizeof(typename DT::st) == 2;  // the up pass alone takes 16-bit types
  typedef void (*Kernel)(RowsArgs);
  enum Which { kGateOnly, kGateAndUp, kNormGateAndUp, kUpOnly };
  template <int STEPS, int CH, int NG>
  static Kernel kernel(Which w) {
    if constexpr (kHasUp)
      if (w == kUpOnly) return rows_mma_up_kernel<DT, STEPS, CH, NG>;
    if (w == kGateOnly) return rows_mma_kernel<DT, STEPS, CH, false, NG, false>;
    return w == kNormGateAndUp ? rows_mma_kernel<DT, STEPS, CH, true, NG, CH == 2> : rows_mma_kernel<DT, STEPS, CH, true, NG, false>;
  }
  // One instance per number of steps, so that no load or MFMA sits behind a branch on the row length.
  template <int NG>
  static Kernel kernel_for(Which w, MmaSplit sp) {
    if (sp.chunks == 2) {
      if constexpr (NG == 1) {  // two groups of x operands of such rows do not fit in LDS
        switch (sp.steps) {
          case 5: return kernel<5, 2, NG>(w);
          case 6: return kernel<6, 2, NG>(w);
          case 7: return kernel<7, 2, NG>(w);
          case 8: return kernel<8, 2, NG>(w);
          case 9: return kernel<9, 2, NG>(w);
        }
      }
      return nullptr;
    }
    switch (sp.steps) {
      case 1: return kernel<1, 1, NG>(w);
      case 2: return kernel<2, 1, NG>(w);
      case 3: return kernel<3, 1, NG>(w);
      case 4: return kernel<4, 1, NG>(w);
      case 5: return kernel<5, 1, NG>(w);
      case 6: return kernel<6, 1, NG>(w);
      case 7: return kernel<7, 1, NG>(w);
      case 8: return kernel<8, 1, NG>(w);
      case 9: return kernel<9, 1, NG>(w);
    }
    return nullptr;
  }
  static bool supported(const RowsArgs& a, int ng = 1) {
    const MmaSplit sp = rows_mma_split(a);
    if (a.mask_out && !a.ubytes_out) return false;  // this kernel writes the union of the flags as bytes only
    if (a.norm_w && !a.w2) return false;            // ... and has no norm in the gate pass alone
    return sp.steps > 0 && (ng == 1 || sp.chunks == 1) && rows_mma_lds_bytes(a, ng) <= kMmaMaxLds;
  }
  static constexpr size_t kMmaMaxLds = 160 * 1024 - 256;  // the kernels' static LDS takes the rest
  static hipError_t launch(Which w, const RowsArgs& a_in, int ng, size_t lds, hipStream_t stream) {
    RowsArgs a = a_in;
    const int grid = rows_mma_layout(a, current_device_cus());
    const MmaSplit sp = rows_mma_split(a);
    Kernel kern = ng == 2 ? kernel_for<2>(w, sp) : kernel_for<1>(w, sp);
    if (!kern) return hipErrorInvalidValue;
    a.mma_front = sp.front;
    a.mma_slots = sp.slots;
    if (hipError_t e = ensure_dynamic_lds((const void*)kern, lds); e != hipSuccess) return e;
    return launch_kernel(kern, dim3(grid), dim3(kMmaThreads), lds, stream, a);
  }
  // one persistent workgroup per CU, or per tile where there are fewer tiles
  static int up_grid(const RowsArgs& a) {
    const int cus = current_device_cus();
    const int ntiles = (a.N + kMmaTileRows - 1) / kMmaTileRows;
    return ntiles < cus ? ntiles : cus;
  }
  static Which gate_kernel(const RowsArgs& a, bool up) { return !up ? kGateOnly : a.norm_w ? kNormGateAndUp : kGateAndUp; }
  static hipError_t run(const RowsArgs& a, bool up, hipStream_t stream) {
    return launch(gate_kernel(a, up), a, 1, rows_mma_lds_bytes(a), stream);
  }
  // gate + up (a.w2 set) or the gate pass alone for 9..16 batch rows in one pass over the weights
  static hipError_t run16(const RowsArgs& a, hipStream_t stream) {
    return launch(gate_kernel(a, a.w2 != nullptr), a, 2, rows_mma_lds_bytes(a, 2), stream);
  }
  // the up pass alone, gate activations given (kUp)
  static int up_rows_pad(const RowsArgs& a) {
    const int grid = up_grid(a);
    return ((a.N + grid - 1) / grid + kMmaTileRows - 1) / kMmaTileRows * kMmaTileRows;
  }
  static bool supported_up(const RowsArgs& a) {
    const int ng = a.nb > 8 ? 2 : 1;
    return kHasUp && supported(a, ng) && a.a_in && (a.z32_out || a.zt_out) && !a.norm_w && a.nb <= 16 &&
           rows_mma_up_lds_bytes(a, up_rows_pad(a), ng) <= kMmaMaxLds;
  }
  static hipError_t run_up(const RowsArgs& a, hipStream_t stream) {
    const int ng = a.nb > 8 ? 2 : 1;
    return launch(kUpOnly, a, ng, rows_mma_up_lds_bytes(a, up_rows_pad(a), ng), stream);
  }
  // dense GEMV out = x . w^T (kGemv): any row length, 3..16 batch rows, up to 64 rows of w per workgroup (32 in fp32, whose sums take
  // four times the registers)
  static constexpr int kGemvTiles = kHasUp ? 8 : 4;
  static bool supported_gemv(const RowsArgs& a) {
    return (a.zt_out || (!kHasUp && (a.a_out || a.flag_out))) && !a.norm_w && !a.bias && !a.scale && a.nb <= 16 && a.K % DT::VEC == 0 && up_rows_pad(a) <= kGemvTiles * kMmaTileRows;
  }
  template <int NG>
  static hipError_t run_gemv_ng(const RowsArgs& a, hipStream_t stream) {
    const int tiles = up_rows_pad(a) / kMmaTileRows;
    auto kern = tiles <= 2 ? gemv_mma_kernel<DT, NG, 2> : tiles <= 4 ? gemv_mma_kernel<DT, NG, 4> : gemv_mma_kernel<DT, NG, kGemvTiles>;
    const size_t lds = gemv_mma_lds_bytes();
    if (hipError_t e = ensure_dynamic_lds((const void*)kern, lds); e != hipSuccess) return e;
    return launch_kernel(kern, dim3(up_grid(a)), dim3(kMmaThreads), lds, stream, a);
  }
  static hipError_t run_gemv(const RowsArgs& a, hipStream_t stream) { return a.nb > 8 ? run_gemv_ng<2>(a, stream) : run_gemv_ng<1>(a, stream); }
};

// Whether a call goes to the matrix-core kernel.  16-bit types, measured on Llama-7B shapes: at 2 batch rows the wave-per-row kernel is
// still the faster one (28.4 vs 29.4 us).  From three rows on it wins at every row length (gate + up, wave-per-row against
// matrix cores: 255 against 129 us for 28672 rows of 8192 elements at 8 batch rows; whole MLP calls: 22.0 against 15.7 us for 3000
// rows of 1024 at 4, 162 against 75 us for 13824 rows of 5120 at 8, 57 against 21 us for 3931 rows of 1264 at 11, where the
// other way is two passes).  The plain gate pass goes the same way as gate + up -- in fp32 beyond this kernel's rows too, see
// joined_takes -- so a gate call and a fused call produce the same activations bit for bit.  (Where an up matrix that starts at
// another place of a cache line than the gate matrix takes the fused call past the last row length that fits on chip, the two differ
// in the order of their sums; so do a layer tail and a call without its norm at 9..16 fp32 rows of more than 2180 elements.)
template <class DT>
bool takes_mma(int mode, int bt, const RowsArgs& a) {
  if (bt < 4 || !a.mma) return false;
  // fp32 up to four rows: the wave-per-row kernel keeps up with the weights (gate + up of 4096 / 11008 at 4 rows: 17 us less), as long
  // as it finds x in LDS (dense down, K = 12936: 11 us more).  At eight rows it spends 256 fused multiply-adds a lane on 32 vectors
  // and the matrix cores win (5632 rows of 2048: 54 against 42 us a call, 11008 of 4096: 128 against 115, with a dense down 258 against 120).
  if (std::is_same<DT, F32>::value && bt == 4 && (mode != kGemv || (size_t)bt * a.K * 4 <= kStagedMaxBytes)) return false;
  if (mode == kUp) return MmaLaunch<DT>::supported_up(a);
  if (mode == kGemv) return MmaLaunch<DT>::supported_gemv(a);
  return (mode == kGateUp || mode == kGate) && MmaLaunch<DT>::supported(a);
}

template <class DT, int B>
hipError_t launch_rows_b(int mode, const RowsArgs& a, hipStream_t stream) {
  if (takes_mma<DT>(mode, B, a))
    return mode == kUp ? MmaLaunch<DT>::run_up(a, stream) : mode == kGemv ? MmaLaunch<DT>::run_gemv(a, stream) : MmaLaunch<DT>::run(a, mode == kGateUp, stream);
  const size_t lds = (size_t)B * ((a.nch + kCB - 1) / kCB * kCB) * kWave * sizeof(u32x4);
  const bool xlds = lds <= kStagedMaxBytes;
  const bool full = xlds && (a.K % (kWave * DT::VEC * kCB) == 0);
  switch (mode) {
    case kGate:
      if (full) return launch_rows_one<DT, B, true, kGate, true>(a, stream);
      if (xlds) return launch_rows_one<DT, B, false, kGate, true>(a, stream);
      return launch_rows_one<DT, B, false, kGate, false>(a, stream);
    case kGateUp:
      if (full) return launch_rows_one<DT, B, true, kGateUp, true>(a, stream);
      if (xlds) return launch_rows_one<DT, B, false, kGateUp, true>(a, stream);
      return launch_rows_one<DT, B, false, kGateUp, false>(a, stream);
    case kUp:
      if (xlds) return launch_rows_one<DT, B, false, kUp, true>(a, stream);
      return launch_rows_one<DT, B, false, kUp, false>(a, stream);
    case kGemv:
      if (xlds) return launch_rows_one<DT, B, false, kGemv, true>(a, stream);
      return launch_rows_one<DT, B, false, kGemv, false>(a, stream);
    case kUpIndex:
      if (xlds) return launch_rows_one<DT, B, false, kUpIndex, true>(a, stream);
      return launch_rows_one<DT, B, false, kUpIndex, false>(a, stream);
  }
  return hipErrorInvalidValue;
}

template <class DT, int B, bool ZF32>
hipError_t launch_down_one(const DownArgs& a, int block, hipStream_t stream) {
  auto kern = down_kernel<DT, B, ZF32, kDownU>;
  const int nwaves = block / kWave;
  // streaming phase: index list + z of the range; fold phase (same bytes): half the waves' partial sums
  // (index list, z, and for 16-bit types the packed z pairs)
  const size_t zbytes = (size_t)B * a.chunk * sizeof(typename DT::st);
  const size_t lds_stream = (size_t)a.chunk * sizeof(int) + (zbytes + 3) / 4 * 4 + (sizeof(typename DT::st) == 2 ? zbytes + 4 * B : 0);
  const size_t lds_fold = (size_t)nwaves * (B < 4 ? B : 4) * kWave * DT::VEC * sizeof(float);  // up to four batch rows per pass
  const size_t lds = (lds_stream > lds_fold ? lds_stream : lds_fold) + 64;
  if (hipError_t e = ensure_dynamic_lds((const void*)kern, lds); e != hipSuccess) return e;
  return launch_kernel(kern, dim3(a.nslab * a.ngroup), dim3(block), lds, stream, a);
}

#ifndef CATS_DOWN_MMA_DEPTH
#define CATS_DOWN_MMA_DEPTH 2
#endif
constexpr int kDownMmaDepth = CATS_DOWN_MMA_DEPTH;  // steps of loads a wave of the matrix-core down kernel keeps in flight

template <class DT>
struct DownMmaLaunch {
  static bool supported(const DownArgs&) { return false; }
  static hipError_t run(bool, const DownArgs&, hipStream_t) { return hipErrorInvalidValue; }
};
template <class DT>
struct DownMmaLaunch16 {
  static bool supported(const DownArgs& a) {
    return a.partial_out && a.nb >= 1 && a.nb <= 16 && down_mma_lds_bytes(a.chunk, a.nb, kDownMmaDepth) <= 150 * 1024;
  }
  static hipError_t run(bool zf32, const DownArgs& a_in, hipStream_t stream) {
    DownArgs a = a_in;
    // slabs of equal width, in whole cache lines: 385 vectors are seven of 56, the last one 49, not six of 64 and one of 1
    a.slab_vecs = ((a.row_vecs + a.nslab - 1) / a.nslab + 7) / 8 * 8;
    const size_t lds = down_mma_lds_bytes(a.chunk, a.nb, kDownMmaDepth);
    // Early rows save the trip in which the memory idles, 0.6 to 1.2 us, and cost 64 rows of every range, up to 16.8 MB in all whatever the matrix,
    // times their dead share.  Without, with them in us at 30 / 60 / 90 % sparsity:
    //   3 rows   3080 / 8191 36.0, 35.1 / 33.3, 33.0 / 27.4, 27.9 (75 % 29.6, 30.8)   2304 / 6144 24.1, 23.5 / 23.1, 22.8 / 20.9, 21.1
    //            2048 / 5461 21.8, 21.1 / 20.8, 20.6 / 19.1, 19.6   4096 / 11008 51.1, 50.5 / - / 35.6, 37.5
    //   8 rows   4096 / 11008 54.6, 53.6 / 52.0, 51.2 / 42.1, 42.2
    //            3080 / 8191 38.4, 37.5 / 37.4, 36.8 / 30.8, 32.1   2560 / 6912 31.2, 30.3 / 31.0, 30.3 / 26.4, 26.6   1024 / 10000 23.1, 22.5 / 23.3, 22.6 / 20.2, 20.0
    //   16 rows  4096 / 14336 71.5, 70.0 / 69.6, 68.2 / 58.6, 58.4   4096 / 11008 60.7, 59.4 / 59.7, 58.6 / 51.3, 50.7   2560 / 6912 34.3, 33.4 / 34.6, 33.8 / 30.4, 31.1
    // So they pay up to 60 to 75 %, and beyond cost up to what they gave; which it will be the host cannot see.  They are left out where the loss is the
    // larger: up to eight rows of large matrices (for the few rows among them), and ranges that are half early and
    // start a multiple of 512 KiB apart, whose early rows all lie on the same part of the memory (2048 / 8192 at 3 rows 26.7, 26.8 / 25.3, 25.8 / 21.9,
    // 23.1, at 8 28.6, 28.9 / 28.3, 28.6 / 24.8, 25.7; 2048 / 7168 at 3 rows 24.9, 24.1 / 23.6, 23.3, 1920 / 8192 25.3, 24.4 / 24.0, 23.6).
    const bool alike = a.chunk <= 2 * kDownMmaEarly && ((size_t)a.chunk * a.row_vecs * 16) % (512 << 10) == 0;
    const bool early = a.mask_bytes && !a.flags && !a.idx && (a.nb > 8 || ((size_t)a.I * a.row_vecs * 16 <= (56u << 20) && !alike));
    auto kern = early ? (zf32 ? down_mma_kernel<DT, true, kDownMmaDepth, true> : down_mma_kernel<DT, false, kDownMmaDepth, true>)
                      : (zf32 ? down_mma_kernel<DT, true, kDownMmaDepth, false> : down_mma_kernel<DT, false, kDownMmaDepth, false>);
    if (hipError_t e = ensure_dynamic_lds((const void*)kern, lds); e != hipSuccess) return e;
    return launch_kernel(kern, dim3(a.nslab * a.ngroup), dim3(kDownMmaThreads), lds, stream, a);
  }
};
template <> struct DownMmaLaunch<F16> : DownMmaLaunch16<F16> {};
template <> struct DownMmaLaunch<BF16> : DownMmaLaunch16<BF16> {};

template <class DT, int B, bool FULL, int KV, int DW>
hipError_t launch_fused_one(int grid, const FusedArgs& a, hipStream_t stream) {
  auto kern = mlp_fused_kernel<DT, B, FULL, KV, DW>;
  const size_t lds = fused_lds_bytes(B, a.nch, a.cap, DT::VEC, DW);
  if (hipError_t e = ensure_dynamic_lds((const void*)kern, lds); e != hipSuccess) return e;
  return launch_kernel(kern, dim3(grid), dim3(kFusedThreads), lds, stream, a);
}

template <class DT, int B>
hipError_t launch_fused_b(int grid, const FusedArgs& a, hipStream_t stream) {
  const bool full = a.H % (kWave * DT::VEC * kFusedCB) == 0;
  constexpr int DW = fused_down_waves(B);
  const int kv = (a.row_vecs + DW * kWave - 1) / (DW * kWave);
#define CATS_FUSED_KV(KVV)                                                                \
  if (kv <= KVV) return full ? launch_fused_one<DT, B, true, KVV, DW>(grid, a, stream)    \
                             : launch_fused_one<DT, B, false, KVV, DW>(grid, a, stream);
  CATS_FUSED_KV(1)
  CATS_FUSED_KV(2)
  CATS_FUSED_KV(4)
#undef CATS_FUSED_KV
  return hipErrorInvalidValue;
}

template <class DT, int B, int MODE, int CB>
hipError_t launch_proj_cb(const ProjArgs& a, hipStream_t stream) {
  constexpr int WAVES = WavesFor<B>::value, R = MODE == kProjPlain ? 2 * kProjCB / CB : 2;
  const bool full = a.r.K % (kWave * DT::VEC * CB) == 0;
  auto kern = full ? proj_kernel<DT, B, CB, R, true, MODE, WAVES> : proj_kernel<DT, B, CB, R, false, MODE, WAVES>;
  const int items = MODE == kProjQkv ? a.r.N / 2 * 3 : (a.r.N + R - 1) / R;
  const size_t lds = proj_lds_bytes(B, a.r.nch, CB);
  if (hipError_t e = ensure_dynamic_lds((const void*)kern, lds); e != hipSuccess) return e;
  return launch_kernel(kern, dim3((items + WAVES - 1) / WAVES), dim3(WAVES * kWave), lds, stream, a);
}
// Rows of up to two or four chunks of 64 vectors have instances of their own at one and two rows; batches of such rows are the matrix cores'.
template <class DT, int B, int MODE>
hipError_t launch_proj_one(const ProjArgs& a, hipStream_t stream) {
  if constexpr (B <= 2) {
    if (a.r.nch <= 2) return launch_proj_cb<DT, B, MODE, 2>(a, stream);
    if (a.r.nch <= 4) return launch_proj_cb<DT, B, MODE, 4>(a, stream);
  }
  return launch_proj_cb<DT, B, MODE, kProjCB>(a, stream);
}

// Projections of 3..8 rows on the matrix cores: 16-bit types, rows and matrices on whole cache lines, head halves in fours, x operands in LDS.
// Products in fp16 with the weights from memory, a wave a row / matrix cores in us:
//   2 rows   32000 x 512 8.5, 9.5   32000 x 2048 23.3, 24.9   4096 x 4096 7.5, 8.7   3072 x 1024 4.4, 5.3
//   3 rows   32000 x 512 26.0, 9.5   32000 x 2048 30.5, 25.0   32000 x 4096 42.5, 43.5   4096 x 4096 8.8, 8.8   3072 x 1024 5.9, 5.3   5120 x 5120 17.8, 13.2
//   4 rows   32000 x 512 26.1, 9.4   32000 x 2048 31.8, 24.9   32000 x 4096 43.6, 43.6   4096 x 4096 9.1, 8.9   8000 x 2048 9.8, 8.6   32000 x 8192 87.2, 83.4
//   8 rows   32000 x 512 46.0, 9.4   32000 x 2048 50.5, 24.7   32000 x 4096 63.4, 41.9   4096 x 4096 13.1, 9.0   8000 x 8192 40.2, 28.2
// So they are taken from three rows on.  At three and four rows 8192 x 8192 alone loses, 25.5, 27.8; 1024 x 8192 10.2, 9.4 and 7168 x 7168 20.5, 19.7 do not.
template <class DT>
struct ProjMma {
  template <int MODE, int STEPS, int CH>
  static hipError_t run(const ProjArgs& a, int grid, size_t lds, hipStream_t stream) {
    if constexpr (sizeof(typename DT::st) == 2) {
      auto kern = proj_mma_kernel<DT, STEPS, CH, MODE>;
      if (hipError_t e = ensure_dynamic_lds((const void*)kern, lds); e != hipSuccess) return e;
      return launch_kernel(kern, dim3(grid), dim3(kMmaThreads), lds, stream, a);
    } else {
      return hipErrorInvalidValue;
    }
  }
  static bool takes(int mode, const ProjArgs& a) {
    if (sizeof(typename DT::st) != 2 || a.r.nb < 3 || a.r.nb > 8 || a.r.row_vecs % 8 != 0) return false;
    uintptr_t w = (uintptr_t)a.r.w;
    if (mode == kProjQkv) {
      w |= (uintptr_t)a.wk | (uintptr_t)a.wv;
      if (a.half % 4 != 0 || 2 * a.half > kProjMaxHeadDim || a.r.N % 8 != 0) return false;
    }
    const MmaSplit sp = rows_mma_split(a.r);
    return w % 128 == 0 && sp.steps > 0 && proj_mma_lds_bytes(sp) <= MmaLaunch<DT>::kMmaMaxLds;
  }
  template <int MODE>
  static hipError_t launch(const ProjArgs& a_in, hipStream_t stream) {
    ProjArgs a = a_in;
    const MmaSplit sp = rows_mma_split(a.r);
    const int ntiles = proj_mma_ntiles(a, MODE), cus = current_device_cus();
    a.r.rows_per = (ntiles + cus - 1) / cus;
    a.r.mma_slots = sp.slots;
    const int grid = (ntiles + a.r.rows_per - 1) / a.r.rows_per;
    const size_t lds = proj_mma_lds_bytes(sp);
#define CATS_PROJ_CASE(STEPS, CH) \
  if (sp.steps == STEPS && sp.chunks == CH) return run<MODE, STEPS, CH>(a, grid, lds, stream);
    CATS_PROJ_CASE(1, 1) CATS_PROJ_CASE(2, 1) CATS_PROJ_CASE(3, 1) CATS_PROJ_CASE(4, 1) CATS_PROJ_CASE(5, 1) CATS_PROJ_CASE(6, 1) CATS_PROJ_CASE(7, 1)
    CATS_PROJ_CASE(8, 1) CATS_PROJ_CASE(9, 1) CATS_PROJ_CASE(5, 2) CATS_PROJ_CASE(6, 2) CATS_PROJ_CASE(7, 2) CATS_PROJ_CASE(8, 2) CATS_PROJ_CASE(9, 2)
#undef CATS_PROJ_CASE
    return hipErrorInvalidValue;
  }
};

template <class DT, int B>
hipError_t launch_proj_b(int mode, const ProjArgs& a, hipStream_t stream) {
  if (B >= 4 && ProjMma<DT>::takes(mode, a)) {
    if (mode == kProjPlain) return ProjMma<DT>::template launch<kProjPlain>(a, stream);
    if (mode == kProjAdd) return ProjMma<DT>::template launch<kProjAdd>(a, stream);
    return ProjMma<DT>::template launch<kProjQkv>(a, stream);
  }
  switch (mode) {
    case kProjPlain: return launch_proj_one<DT, B, kProjPlain>(a, stream);
    case kProjAdd: return launch_proj_one<DT, B, kProjAdd>(a, stream);
    case kProjQkv: return launch_proj_one<DT, B, kProjQkv>(a, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace

template <>
hipError_t launch_proj<CATS_DT>(int mode, int bt, const ProjArgs& a, hipStream_t stream) {
  switch (bt) {
    case 1: return launch_proj_b<CATS_DT, 1>(mode, a, stream);
    case 2: return launch_proj_b<CATS_DT, 2>(mode, a, stream);
    case 4: return launch_proj_b<CATS_DT, 4>(mode, a, stream);
    case 8: return launch_proj_b<CATS_DT, 8>(mode, a, stream);
  }
  return hipErrorInvalidValue;
}

typedef void (*AttnKernel)(AttnArgs);
template <int LPS>
static AttnKernel attn_for(bool ahead) { return ahead ? attn_decode_kernel<CATS_DT, LPS, true> : attn_decode_kernel<CATS_DT, LPS, false>; }

template <>
hipError_t launch_attn<CATS_DT>(int head_dim, int bt, AttnArgs a, hipStream_t stream) {
  AttnKernel kern = nullptr;
  const int cus = current_device_cus();
  const bool spare = a.pairs <= cus / 4;
  switch (head_dim / CATS_DT::VEC) {  // lanes per cache slot
    case 2: kern = attn_for<2>(spare); break;
    case 4: kern = attn_for<4>(spare); break;
    case 8: kern = attn_for<8>(spare); break;
    case 16: kern = attn_for<16>(spare); break;
    case 32: kern = attn_for<32>(spare); break;
  }
  if (!kern) return hipErrorInvalidValue;
  // the CUs that attention leaves free fetch the next projection's weights, where they are at least three quarters of the chip (half of
  // it: steps of two layers 4096 / 11008, 4 rows of 32 heads, 228.7 / 231.2 us)
  const int ahead = spare ? (cus - a.pairs) / 8 * 8 : 0;
  // from vectors of a row to those of a workgroup of the projection
  const int rows = a.pairs / bt * head_dim;
  if (sizeof(CATS_DT::st) == 2 && bt >= 3 && a.piece_vecs % 8 == 0) a.piece_vecs *= ((rows + 7) / 8 + cus - 1) / cus * 8;
  else a.piece_vecs *= kR * (bt <= 2 ? WavesFor<1>::value : WavesFor<8>::value);
  return launch_kernel(kern, dim3(a.pairs + ahead), dim3(1024), 0, stream, a);
}

template <>
hipError_t launch_silu_mask_mul<CATS_DT>(const SiluMaskMulArgs& a, hipStream_t stream) {
  const size_t blocks = (a.n / CATS_DT::VEC + 1 + 255) / 256;  // one thread more than vectors: it takes what is left
  if (blocks > 0x7fffffffu) return hipErrorInvalidValue;
  return launch_kernel(silu_mask_mul_kernel<CATS_DT>, dim3((unsigned)blocks), dim3(256), 0, stream, a);
}

template <class DT>
struct PromptLaunch {
  template <class T, bool GATE_UP>
  static hipError_t tile(const PromptArgs& a, hipStream_t stream) {
    auto kern = prompt_kernel<DT, T, GATE_UP>;
    if (hipError_t e = ensure_dynamic_lds((const void*)kern, T::LDS); e != hipSuccess) return e;
    const int grid = 8 * a.mblocks * ((a.nblocks * a.splits + 7) / 8);
    return launch_kernel(kern, dim3(grid), dim3(T::THREADS), T::LDS, stream, a);
  }
  template <bool GATE_UP>
  static hipError_t run(const PromptPlan& plan, const PromptArgs& a, hipStream_t stream) {
    const bool two = prompt_steps_ahead(plan, current_device_cus()) == 2;
    switch (plan.tile) {
      case 0: return two ? tile<PromptTile0<2>, GATE_UP>(a, stream) : tile<PromptTile0<1>, GATE_UP>(a, stream);
      case 1: return tile<PromptTile1, GATE_UP>(a, stream);
      case 2: return two ? tile<PromptTile2<2>, GATE_UP>(a, stream) : tile<PromptTile2<1>, GATE_UP>(a, stream);
      case 3: return tile<PromptTile3, GATE_UP>(a, stream);
      case 4: return tile<PromptTile4, GATE_UP>(a, stream);
      case 5: return tile<PromptTile5, GATE_UP>(a, stream);
    }
    return hipErrorInvalidValue;
  }
  static hipError_t sum(const PromptSumArgs& a, hipStream_t stream) {
    const size_t threads = (size_t)a.M * (a.ldp / 4);
    return launch_kernel(prompt_sum_kernel<DT>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, a);
  }
};
template <>
struct PromptLaunch<F32> {
  template <bool GATE_UP>
  static hipError_t run(const PromptPlan&, const PromptArgs&, hipStream_t) { return hipErrorInvalidValue; }
  static hipError_t sum(const PromptSumArgs&, hipStream_t) { return hipErrorInvalidValue; }
};
template <>
hipError_t launch_prompt<CATS_DT>(bool gate_up, const PromptPlan& plan, PromptArgs a, hipStream_t stream) {
  a.mblocks = plan.mblocks;
  a.nblocks = plan.nblocks;
  a.steps = plan.steps;
  a.splits = plan.splits;
  return gate_up ? PromptLaunch<CATS_DT>::run<true>(plan, a, stream) : PromptLaunch<CATS_DT>::run<false>(plan, a, stream);
}
template <>
hipError_t launch_prompt_sum<CATS_DT>(const PromptSumArgs& a, hipStream_t stream) {
  return PromptLaunch<CATS_DT>::sum(a, stream);
}

template <>
hipError_t launch_gate_cols<CATS_DT>(const GateColsArgs& a, int groups, hipStream_t stream) {
  return launch_kernel(gate_cols_kernel<CATS_DT>, dim3(a.nslab * groups), dim3(kGateColsWaves * kWave), 0, stream, a);
}

template <>
hipError_t launch_gate_cols_finish<CATS_DT>(const GateColsArgs& a, int groups, void* a_out, hipStream_t stream) {
  return launch_kernel(gate_cols_finish_kernel<CATS_DT>, dim3((a.I + 255) / 256), dim3(256), 0, stream, (const float*)a.partial, groups, a.I, a_out);
}

template <>
hipError_t launch_reduce<CATS_DT>(const ReduceArgs& r, hipStream_t stream) {
  const int rgrid = (r.BH + kReduceCols - 1) / kReduceCols;  // BH == 0: only the count is wanted
  return launch_kernel(reduce_partials_kernel<CATS_DT>, dim3(rgrid > 0 ? rgrid : 1), dim3(256), 0, stream, r);
}

template <>
hipError_t launch_fused<CATS_DT>(int bt, int grid, int stage, const FusedArgs& a, const ReduceArgs& r, hipStream_t stream) {
  if (stage != 2) {
    hipError_t e = bt == 1 ? launch_fused_b<CATS_DT, 1>(grid, a, stream) : launch_fused_b<CATS_DT, 2>(grid, a, stream);
    if (e != hipSuccess) return e;
  }
  return stage != 1 ? launch_reduce<CATS_DT>(r, stream) : hipSuccess;
}

template <>
bool rows_takes_mma<CATS_DT>(int mode, int bt, const RowsArgs& a) { return takes_mma<CATS_DT>(mode, bt, a); }

template <>
bool down_mma_supported<CATS_DT>(const DownArgs& a) { return DownMmaLaunch<CATS_DT>::supported(a); }

template <>
hipError_t launch_down_mma<CATS_DT>(bool zf32, const DownArgs& a, hipStream_t stream) { return DownMmaLaunch<CATS_DT>::run(zf32, a, stream); }

template <>
bool rows_mma16_supported<CATS_DT>(const RowsArgs& a) { return a.mma && MmaLaunch<CATS_DT>::supported(a, 2); }

template <>
hipError_t launch_rows_mma16<CATS_DT>(const RowsArgs& a, hipStream_t stream) { return MmaLaunch<CATS_DT>::run16(a, stream); }

template <>
hipError_t launch_rows<CATS_DT>(int mode, int bt, const RowsArgs& a, hipStream_t stream) {
  switch (bt) {
    case 1: return launch_rows_b<CATS_DT, 1>(mode, a, stream);
    case 2: return launch_rows_b<CATS_DT, 2>(mode, a, stream);
    case 4: return launch_rows_b<CATS_DT, 4>(mode, a, stream);
    case 8: return launch_rows_b<CATS_DT, 8>(mode, a, stream);
  }
  return hipErrorInvalidValue;
}

template <>
hipError_t launch_down<CATS_DT>(int bt, bool zf32, const DownArgs& a, int block, hipStream_t stream) {
#define CATS_DOWN_CASE(BB)                                                         \
  case BB:                                                                         \
    return zf32 ? launch_down_one<CATS_DT, BB, true>(a, block, stream)             \
                : launch_down_one<CATS_DT, BB, false>(a, block, stream);
  switch (bt) {
    CATS_DOWN_CASE(1)
    CATS_DOWN_CASE(2)
    CATS_DOWN_CASE(4)
    CATS_DOWN_CASE(8)
  }
#undef CATS_DOWN_CASE
  return hipErrorInvalidValue;
}

}  // namespace cats

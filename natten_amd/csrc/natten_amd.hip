// C ABI of the MI355X fused neighborhood attention forward path (see include/natten_amd.h).
// Host-side argument validation, kernel selection and launches; no framework types.

#include "../../include/natten_amd.h"

#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <mutex>
#include <type_traits>

#include "fna_bwd.hpp"
#include "fna_fwd.hpp"
#include "fna_fwd_f32.hpp"
#include "fna_fwd_fp8.hpp"
#include "linear.hpp"
#include "merge.hpp"
#include "mfma_probe.hpp"
#include "na_math.hpp"
#include "tokperm.hpp"

using namespace natten_amd;

// Queue counters of natten_amd_fna_forward_fused_static, the entry point for callers that cannot
// allocate: every GPU the library runs on holds this array (512 bytes) until the process ends.
// The name is a host-side stand-in, not a device address: host code only ever uses the
// per-device address hipGetSymbolAddress returns for it (static_scratch()).  No `used`
// attribute: the compiler gives the device-side symbol external binding because host code names
// it, and with the attribute it stays local, where the runtime's lookup by name cannot find it.
static __device__ __align__(256) uint32_t scratch[kQueueWords];

namespace {

thread_local char g_error[512] = "";

int fail(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
  return 1;
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail("%s: launch failed: %s", what, hipGetErrorString(e));
  return 0;
}

int prod3(const int* x) { return x[0] * x[1] * x[2]; }

struct TileConfig {
  int q_tile, kv_tile;
};

// (Q tile, KV tile) sizes in tokens that have a kernel instance.
const TileConfig kTileConfigs[] = {{128, 64}, {256, 64}, {64, 64}};
constexpr int kNumTileConfigs = sizeof(kTileConfigs) / sizeof(kTileConfigs[0]);

// Workgroups a work-queue launch starts: `per_cu` per compute unit (what the kernel's LDS and register
// use keep resident), a multiple of the XCD count; the device's figure is read once.
int resident_workgroups(int per_cu = 2) {
  static std::atomic<int> cached[64] = {};  // (threads that race here compute the same value)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256 * per_cu;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) cus = 256;
    n = cus;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  n = (per_cu * n / kNumXcd) * kNumXcd;
  return n < kNumXcd ? kNumXcd : n;
}

// Head dims whose rows the 128 x 64 forward instances take as they are, besides 32, 64 and 128
bool narrow_rows(int head_dim) { return head_dim > 32 && head_dim < 128 && head_dim != 64 && head_dim % 8 == 0; }

// The counters of a work-queue launch (null: one workgroup per Q tile).  Every work-queue kernel
// leaves the counters at zero when its last workgroup ends; `clear_first` clears them by a kernel
// before the launch, for memory whose contents are not known.
struct WorkQueue {
  uint32_t* counters = nullptr;
  bool clear_first = true;
  bool paired = false;  // no queue: a workgroup of two groups of waves for each Q tile
};

// DC != 0: rows of p.row_dim elements, DC columns multiplied (no work-queue launch)
template <typename T, int D, int NWAVES, bool RAGGED, int KVT, bool NOMASK = false, int DC = 0, bool CTX = false>
int launch_fna(const FnaParams& p, hipStream_t stream, WorkQueue queues = {}) {
  constexpr int QT = NWAVES * 32;
  if (!fna_tiles_are_powers_of_two(p)) return fail("fna_forward: tile extents must be powers of two");
  if ((p.seqlen_q + QT - 1) / QT != p.num_q_tiles) return fail("fna_forward: internal tile count mismatch");
  const long long wgs = (long long)((p.total_groups + kNumXcd - 1) / kNumXcd) * kNumXcd * p.wg_group;
  if (wgs > 0x7fffffffLL) return fail("fna_forward: problem needs more than 2^31 workgroups");
  if constexpr (DC == 0 && (NWAVES == 4 || !CTX)) {
    if (queues.counters != nullptr) {
      const long long resident = resident_workgroups();
      if (queues.clear_first) hipLaunchKernelGGL(fna_queue_clear_kernel, dim3(1), dim3(kQueueWords), 0, stream, queues.counters);
      hipLaunchKernelGGL((fna_fwd_queue_kernel<T, D, NWAVES, RAGGED, KVT, NOMASK, CTX>),
                         dim3((unsigned)(wgs < resident ? wgs : resident)), dim3(NWAVES * 64), 0, stream, p, queues.counters,
                         int(wgs / kNumXcd));
      return check_launch("fna_forward (work queue)");
    }
  }
  if (p.kv_splits > 1) {
    // kv_splits workgroups per Q-tile position, split slowest (positions keep their XCDs: wgs is a multiple of 8)
    if constexpr (NWAVES == 4 && KVT == 64 && !CTX) {
      if (wgs * p.kv_splits > 0x7fffffffLL) return fail("fna_forward: problem needs more than 2^31 workgroups");
      FnaParams ps = p;
      if (p.split_first < 0) {
        ps.split_grid = int(wgs);
        hipLaunchKernelGGL((fna_fwd_split_kernel<T, D, NWAVES, RAGGED, KVT, DC>), dim3((unsigned)(wgs * p.kv_splits)),
                           dim3(NWAVES * 64), 0, stream, ps);
        return check_launch("fna_forward (split)");
      }
      // the last split_grid positions (a multiple of 8: positions keep their XCDs)
      if (p.split_grid < kNumXcd || p.split_grid % kNumXcd != 0 || p.split_grid > wgs)
        return fail("fna_forward: the split positions must be a multiple of %d up to %lld, got %d", kNumXcd, wgs, p.split_grid);
      ps.split_first = int(wgs) - p.split_grid;
      hipLaunchKernelGGL((fna_fwd_split_kernel<T, D, NWAVES, RAGGED, KVT, DC>),
                         dim3((unsigned)(ps.split_first + p.split_grid * p.kv_splits)), dim3(NWAVES * 64), 0, stream, ps);
      if (int rc = check_launch("fna_forward (split)")) return rc;
      hipLaunchKernelGGL((merge_tail_kernel<T>), dim3((unsigned)p.split_grid * 8), dim3(256), 0, stream, ps);
      return check_launch("fna_forward (merge)");
    } else {
      return fail("fna_forward: KV splits exist for Q tiles of 128 and KV tiles of 64 tokens");
    }
  }
  FnaParams pk = p;
  long long clearing = 0;
  if (RAGGED && p.cu_q != nullptr) {
    clearing = p.split_first != 0 ? na_ceil_div(p.total_q, packed_clear_rows(p.batch)) : 0;
    pk.split_first = int(wgs);
    if (wgs + clearing > 0x7fffffffLL) return fail("fna_forward: problem needs more than 2^31 workgroups");
  }
  // Launches whose tiles mostly need the mask take the maxima late (LATE_MAX; the same bits).  A tile with a mask gains about twice
  // what one without loses, hence the line at half of them.  Us before / after, bf16: 2 x 96 x 96, 7 x 7, H 8, D 128 48.0 / 46.7; 100
  // x 90, 31 x 17, H 12 78.9 / 76.5; 16 x 32 x 32, 5 x 9 x 9, H 8 98.2 / 95.4; 96 x 96, 21 x 21, H 8, D 64 43.3 / 41.6.
  if constexpr (NWAVES == 4 && D >= 64 && !RAGGED && !NOMASK && DC == 0 && !CTX) {
    if (p.mostly_masked) {
      hipLaunchKernelGGL((fna_fwd_kernel<T, D, 4, false, KVT, false, 0, false, true>), dim3((unsigned)wgs), dim3(256), 0, stream, pk);
      return check_launch("fna_forward");
    }
  }
  hipLaunchKernelGGL((fna_fwd_kernel<T, D, NWAVES, RAGGED, KVT, NOMASK, DC, CTX>), dim3((unsigned)(wgs + clearing)),
                     dim3(NWAVES * 64), 0, stream, pk);
  return check_launch("fna_forward");
}

template <typename T, int D>
int launch_paired(const FnaParams& p, hipStream_t stream) {
  if (!fna_tiles_are_powers_of_two(p)) return fail("fna_forward: tile extents must be powers of two");
  if ((p.seqlen_q + 127) / 128 != p.num_q_tiles) return fail("fna_forward: internal tile count mismatch");
  const long long wgs = (long long)((p.total_groups + kNumXcd - 1) / kNumXcd) * kNumXcd * p.wg_group;
  if (wgs > 0x7fffffffLL) return fail("fna_forward: problem needs more than 2^31 workgroups");
  hipLaunchKernelGGL((fna_fwd_paired_kernel<T, D>), dim3((unsigned)wgs), dim3(512), 0, stream, p);
  return check_launch("fna_forward (paired)");
}

// Whether the launch is fully block-sparse: every Q tile is whole (no padding queries), all its
// queries share one window in every dimension, and the KV tiles laid out for it cover that window
// exactly, so that every (Q tile, KV tile) pair the kernel visits is attended in full and the
// instance without any mask code gives the same bits.  The role of the reference's
// fully_block_sparse (csrc/include/natten/cuda/fna_blackwell/collective/fna_fusion.hpp:503-593),
// evaluated from the kernel's own window and box arithmetic.  Needs set_wg_layout() to have run.
bool fully_block_sparse(const FnaParams& p) {
  if (p.cu_q != nullptr || p.edge != 0 || p.kv_splits > 1) return false;
  for (int a = 0; a < 3; ++a) {
    // dilation groups come in at most two extents
    for (int ext = p.ext_base[a] + (p.ext_rem[a] > 0 ? 1 : 0); ext >= p.ext_base[a]; --ext) {
      if (ext < 1 || ext % p.q_tile[a] != 0) return false;
      const bool c = p.causal[a] != 0;
      for (int qf = 0; qf < ext; qf += p.q_tile[a]) {
        const int ql = qf + p.q_tile[a] - 1;
        const int st_f = na_window_start(qf, p.ksize[a], p.stride[a], p.d_stride[a], ext, c);
        const int st_l = na_window_start(ql, p.ksize[a], p.stride[a], p.d_stride[a], ext, c);
        const int en_f = na_window_end(qf, st_f, p.ksize[a], ext, c);
        const int en_l = na_window_end(ql, st_l, p.ksize[a], ext, c);
        // (start and end are monotone in the query: equal at both ends means equal throughout)
        if (st_f != st_l || en_f != en_l) return false;
        const int org = p.anchor ? st_f : ((st_f >> p.kv_tile_lg[a]) << p.kv_tile_lg[a]);
        if (org != st_f || (en_l - org) % p.kv_tile[a] != 0) return false;
      }
    }
  }
  return true;
}

template <bool E5M2, int D, bool NOMASK>
int launch_fna_fp8_instance(const FnaParams& p, hipStream_t stream, WorkQueue queues) {
  constexpr int QT = 128;
  if (!fna_tiles_are_powers_of_two(p)) return fail("fna_forward: tile extents must be powers of two");
  if ((p.seqlen_q + QT - 1) / QT != p.num_q_tiles) return fail("fna_forward: internal tile count mismatch");
  const long long wgs = (long long)((p.total_groups + kNumXcd - 1) / kNumXcd) * kNumXcd * p.wg_group;
  if (wgs > 0x7fffffffLL) return fail("fna_forward: problem needs more than 2^31 workgroups");
  if (queues.counters != nullptr) {
    const long long resident = resident_workgroups(fp8_waves_per_simd(D));
    if (queues.clear_first) hipLaunchKernelGGL(fna_queue_clear_kernel, dim3(1), dim3(kQueueWords), 0, stream, queues.counters);
    hipLaunchKernelGGL((fna_fwd_fp8_queue_kernel<E5M2, D, 4, NOMASK>), dim3((unsigned)(wgs < resident ? wgs : resident)),
                       dim3(256), 0, stream, p, queues.counters, int(wgs / kNumXcd));
    return check_launch("fna_forward (work queue)");
  }
  hipLaunchKernelGGL((fna_fwd_fp8_kernel<E5M2, D, 4, NOMASK>), dim3((unsigned)wgs), dim3(256), 0, stream, p);
  return check_launch("fna_forward");
}

template <bool E5M2, int D>
int launch_fna_fp8(const FnaParams& p, hipStream_t stream, WorkQueue queues) {
  if (fully_block_sparse(p)) return launch_fna_fp8_instance<E5M2, D, true>(p, stream, queues);
  return launch_fna_fp8_instance<E5M2, D, false>(p, stream, queues);
}

// Key sequences that end inside a tile, where the tile cannot be moved back to end with them: packed
// sequences, dense ones shorter than a tile, dilation groups narrower than a tile.  All others move it back: the
// instance that clamps has the registers of each tile's end to hold (2 x 4097 tokens, H 16, D 64: 218 us there when it
// also issued its copies at the top of an iteration, 203 with the last tile moved back).
bool needs_clamped_rows(const FnaParams& p, int kvt) {
  return p.cu_q != nullptr || p.edge == 2 || (p.seqlen_kv % kvt != 0 && p.edge != 1);
}

// Launches whose queries also attend to a context: masked instances.
bool context_launch_fits(const FnaParams& p, int kvt) { return kvt == 64 && !needs_clamped_rows(p, kvt); }

template <typename T, int D>
int dispatch_tiles(const FnaParams& p, int qt, int kvt, hipStream_t stream, WorkQueue queues) {
  if (p.has_context()) {
    if (context_launch_fits(p, kvt)) {
      if (qt == 128) return launch_fna<T, D, 4, false, 64, false, 0, true>(p, stream, queues);
      if constexpr (D <= 64) {
        if (qt == 64 && queues.counters == nullptr) return launch_fna<T, D, 2, false, 64, false, 0, true>(p, stream);
      }
    }
    return fail("fna_forward: no kernel with a context for these tiles and extents (Q tile %d, KV tile %d, head_dim %d)", qt, kvt, D);
  }
  if (needs_clamped_rows(p, kvt)) {
    if (qt == 128 && kvt == 64) return launch_fna<T, D, 4, true, 64>(p, stream);
    return fail("fna_forward: seqlen_kv (%d) must be a multiple of the KV tile (%d tokens)", p.seqlen_kv, kvt);
  }
  // (A fully block-sparse launch of head dim 128 keeps its mask-free instance, one group a Q tile: 16 x 32 x 32, 8 x 16 x 16
  // blocked, H 2: 37.1 us there, 37.9 as pairs with masks; 8192 tokens blocked by 128, windows of 8, 12 and 16 KV tiles, us in one
  // group / split in two and merged / as pairs, 64 Q tiles 12.1 / 15.2 / 13.5, 15.0 / 16.6 / 16.0, 18.0 / 18.3 / 18.2, 128
  // Q tiles 12.5 / 18.3 / 13.9, 15.3 / 20.2 / 16.4, 18.2 / 22.0 / 18.6.  Head dim 64: 32768 tokens, 2048 blocked by
  // 128, H 1: 24.0 and 22.5; the 8192 tokens with 64 Q tiles 9.1 / 11.8 / 9.5, 11.4 / 13.0 / 11.1, 13.4 / 14.1 / 12.6.)
  if (queues.paired && !(D == 128 && qt == 128 && kvt == 64 && fully_block_sparse(p))) {
    if constexpr (D >= 64) {
      if (qt == 128 && kvt == 64) return launch_paired<T, D>(p, stream);
    }
    return fail("fna_forward: pairs of groups exist for Q tiles of 128 and KV tiles of 64 tokens and head dims 64 and 128");
  }
  // the work-queue launch exists for the default tile pair; the others launch a workgroup per Q tile
  if (qt == 128 && kvt == 64) {
    if (fully_block_sparse(p)) return launch_fna<T, D, 4, false, 64, true>(p, stream, queues);
    return launch_fna<T, D, 4, false, 64>(p, stream, queues);
  }
  if (qt == 256 && kvt == 64) return launch_fna<T, D, 8, false, 64>(p, stream);
  if (qt == 64 && kvt == 64) return launch_fna<T, D, 2, false, 64>(p, stream);
  return fail("fna_forward: no kernel for Q tile of %d and KV tile of %d tokens", qt, kvt);
}

// Head dims between the native ones (multiples of 8 above 32).  Up to 96 of 128 columns are multiplied as
// 96: a quarter of the matrix work and of the LDS reads less.
template <typename T, bool RAGGED, bool CTX = false>
int dispatch_narrow_rows(const FnaParams& p, int head_dim, hipStream_t stream) {
  if (head_dim < 64) return launch_fna<T, 64, 4, RAGGED, 64, false, 64, CTX>(p, stream);
  if (head_dim <= 96) return launch_fna<T, 128, 4, RAGGED, 64, false, 96, CTX>(p, stream);
  return launch_fna<T, 128, 4, RAGGED, 64, false, 128, CTX>(p, stream);
}

template <typename T>
int dispatch_head_dim(const FnaParams& p, int head_dim, int qt, int kvt, hipStream_t stream, WorkQueue queues) {
  switch (head_dim) {
    case 32: return dispatch_tiles<T, 32>(p, qt, kvt, stream, queues);
    case 64: return dispatch_tiles<T, 64>(p, qt, kvt, stream, queues);
    case 128: return dispatch_tiles<T, 128>(p, qt, kvt, stream, queues);
  }
  if (!narrow_rows(head_dim)) return fail("fna_forward: head_dim must be 32, 64 or 128, got %d", head_dim);
  if (qt != 128 || kvt != 64 || queues.counters != nullptr || p.cu_q != nullptr || p.row_dim != head_dim)
    return fail("fna_forward: head_dim %d needs tiles of 128 x 64 tokens and no work queue", head_dim);
  if (p.has_context()) {
    if (!context_launch_fits(p, kvt)) return fail("fna_forward: no kernel with a context for these extents (head_dim %d)", head_dim);
    return dispatch_narrow_rows<T, false, true>(p, head_dim, stream);
  }
  if (needs_clamped_rows(p, kvt)) return dispatch_narrow_rows<T, true>(p, head_dim, stream);
  return dispatch_narrow_rows<T, false>(p, head_dim, stream);
}

int dispatch_dtype(const FnaParams& p, int dtype, int head_dim, int qt, int kvt, hipStream_t stream,
                   WorkQueue queues = {}) {
  switch (dtype) {
    case NATTEN_AMD_F16: return dispatch_head_dim<_Float16>(p, head_dim, qt, kvt, stream, queues);
    case NATTEN_AMD_BF16: return dispatch_head_dim<__bf16>(p, head_dim, qt, kvt, stream, queues);
  }
  if (p.kv_splits > 1) return fail("fna_forward: KV splits need fp16 / bf16 operands, got dtype code %d", dtype);
  if (dtype == NATTEN_AMD_F8E4M3 || dtype == NATTEN_AMD_F8E5M2) {
    // 8-bit float operands, bf16 output: one kernel configuration
    if (qt != 128 || kvt != 64)
      return fail("fna_forward: 8-bit float operands need a Q tile of 128 and a KV tile of 64 tokens, got %d and %d", qt,
                  kvt);
    if (p.seqlen_kv % kvt != 0)
      return fail("fna_forward: seqlen_kv (%d) must be a multiple of the KV tile (%d tokens)", p.seqlen_kv, kvt);
    if (head_dim != 64 && head_dim != 128)
      return fail("fna_forward: 8-bit float operands need head_dim 64 or 128, got %d", head_dim);
    const bool e5m2 = dtype == NATTEN_AMD_F8E5M2;
    if (head_dim == 128)
      return e5m2 ? launch_fna_fp8<true, 128>(p, stream, queues) : launch_fna_fp8<false, 128>(p, stream, queues);
    return e5m2 ? launch_fna_fp8<true, 64>(p, stream, queues) : launch_fna_fp8<false, 64>(p, stream, queues);
  }
  if (dtype == NATTEN_AMD_F32) {
    // float32 operands and output: one plain kernel configuration on token-permuted sequences
    if (qt != 128 || kvt != 64)
      return fail("fna_forward: float32 operands need a Q tile of 128 and a KV tile of 64 tokens, got %d and %d", qt, kvt);
    if (p.fused || p.cu_q != nullptr) return fail("fna_forward: float32 operands run on token-permuted sequences only");
    if (p.seqlen_kv % kvt != 0)
      return fail("fna_forward: seqlen_kv (%d) must be a multiple of the KV tile (%d tokens)", p.seqlen_kv, kvt);
    if (p.q_scale || p.k_scale || p.v_scale) return fail("fna_forward: float32 operands take no dequantisation scales");
    if ((p.seqlen_q + qt - 1) / qt != p.num_q_tiles) return fail("fna_forward: internal tile count mismatch");
    const long long wgs = (long long)p.num_q_tiles * p.heads_q * p.batch;
    if (wgs > 0x7fffffffLL) return fail("fna_forward: problem needs more than 2^31 workgroups");
    switch (head_dim) {
      case 32: hipLaunchKernelGGL((fna_fwd_f32_kernel<32>), dim3((unsigned)wgs), dim3(256), 0, stream, p); break;
      case 64: hipLaunchKernelGGL((fna_fwd_f32_kernel<64>), dim3((unsigned)wgs), dim3(256), 0, stream, p); break;
      case 128: hipLaunchKernelGGL((fna_fwd_f32_kernel<128>), dim3((unsigned)wgs), dim3(256), 0, stream, p); break;
      default: return fail("fna_forward: unsupported head_dim %d", head_dim);
    }
    return check_launch("fna_forward (float32)");
  }
  return fail("fna_forward: unsupported dtype code %d", dtype);
}

int check_common(const char* what, const void* q, const void* k, const void* v, const void* out, const float* lse,
                 int batch, int seqlen_q, int seqlen_kv, int heads_q, int heads_kv, int head_dim, bool narrow_ok = false) {
  if (!q || !k || !v || !out || !lse) return fail("%s: null pointer argument", what);
  if (batch < 1 || seqlen_q < 1 || seqlen_kv < 1 || heads_q < 1 || heads_kv < 1)
    return fail("%s: batch, sequence lengths and head counts must be positive", what);
  if (heads_q % heads_kv != 0)
    return fail("%s: heads_kv (%d) must divide heads_q (%d)", what, heads_kv, heads_q);
  if (head_dim != 32 && head_dim != 64 && head_dim != 128 && !(narrow_ok && narrow_rows(head_dim)))
    return fail("%s: head_dim must be 32, 64 or 128, got %d", what, head_dim);
  if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
       reinterpret_cast<uintptr_t>(out)) & 15)
    return fail("%s: q, k, v and out must be 16-byte aligned", what);
  return 0;
}

// Shared by the permuted and the fused entry points: checks the neighborhood parameters and fills
// everything but the operand layout.  q_shape / kv_shape: padded per-group token layouts.
int fill_fna_params(const char* what, FnaParams& p, int na_dim, const int* q_shape, const int* kv_shape,
                    const int32_t* qkv_shape, const int32_t* kernel_size, const int32_t* stride,
                    const int32_t* dilation, const int32_t* is_causal, const int32_t* q_tile_shape,
                    const int32_t* kv_tile_shape) {
  memset(&p, 0, sizeof(p));
  p.num_groups = 1;
  for (int a = 0; a < 3; ++a) {
    const bool used = a < na_dim;
    p.qkv_shape[a] = used ? qkv_shape[a] : 1;
    p.ksize[a] = used ? kernel_size[a] : 1;
    p.stride[a] = used ? stride[a] : 1;
    p.dil[a] = used ? dilation[a] : 1;
    p.causal[a] = used ? (is_causal[a] != 0) : 0;
    p.q_tile[a] = used ? q_tile_shape[a] : 1;
    p.kv_tile[a] = used ? kv_tile_shape[a] : 1;
    const int qs = used ? q_shape[a] : 1, ks = used ? kv_shape[a] : 1;
    if (p.qkv_shape[a] < 1 || p.dil[a] < 1 || p.stride[a] < 1 || p.q_tile[a] < 1 || p.kv_tile[a] < 1 ||
        (used && p.ksize[a] < 2))
      return fail("%s: invalid parameter along dimension %d", what, a);
    if (p.ksize[a] * p.dil[a] > p.qkv_shape[a])
      return fail("%s: kernel_size * dilation exceeds the input along dimension %d (%d * %d > %d)", what, a,
                  p.ksize[a], p.dil[a], p.qkv_shape[a]);
    if (p.stride[a] > p.ksize[a])
      return fail("%s: stride exceeds kernel_size along dimension %d (%d > %d)", what, a, p.stride[a], p.ksize[a]);
    if (qs % p.q_tile[a] != 0 || ks % p.kv_tile[a] != 0)
      return fail("%s: padded layouts must be multiples of the tile shapes (dimension %d)", what, a);
    const int need = na_ceil_div(p.qkv_shape[a], p.dil[a]);
    if (qs < need || ks < need)
      return fail("%s: q_shape / kv_shape smaller than the dilation group extent along dimension %d", what, a);
    if (p.kv_tile[a] > 512) return fail("%s: KV tile extent above 512 along dimension %d", what, a);
    p.q_tiled[a] = qs / p.q_tile[a];
    p.kv_tiled[a] = ks / p.kv_tile[a];
    p.num_groups *= p.dil[a];
  }
  p.tok_stride[2] = 1;
  p.tok_stride[1] = p.qkv_shape[2];
  p.tok_stride[0] = p.qkv_shape[2] * p.qkv_shape[1];
  return 0;
}

// The queue counters of a work-queue launch inside the caller's workspace (nullptr: launch a
// workgroup per Q tile).  rc != 0 on a workspace that cannot hold them.
int queue_workspace(const char* what, int run_persistent, void* workspace, uint64_t workspace_bytes, WorkQueue* queues) {
  *queues = WorkQueue{};
  if (!run_persistent) return 0;
  if (run_persistent != 1 && run_persistent != 2) return fail("%s: run_persistent must be 0, 1 or 2, got %d", what, run_persistent);
  if (!workspace || workspace_bytes < uint64_t(kQueueWords) * 4 || (reinterpret_cast<uintptr_t>(workspace) & 63))
    return fail("%s: run_persistent needs a 64-byte aligned device workspace of at least %d bytes (got %p, %llu bytes)", what,
                kQueueWords * 4, workspace, (unsigned long long)workspace_bytes);
  queues->counters = static_cast<uint32_t*>(workspace);
  queues->clear_first = run_persistent == 1;  // 2: the caller vouches for zeros (what every launch leaves behind)
  return 0;
}

int fused_geometry(const char* what, FnaParams& p, bool sixteen_bit, int na_dim, int heads_kv, int head_dim,
                   const int32_t* qkv_shape, const int32_t* kernel_size, const int32_t* stride, const int32_t* dilation,
                   const int32_t* is_causal, const int32_t* q_tile_shape, const int32_t* kv_tile_shape, int anchor_kv_tiles,
                   long long* tokens_out);
}  // namespace

extern "C" {

int natten_amd_abi_version(void) { return 22; }

uint64_t natten_amd_fna_forward_workspace_bytes(void) { return uint64_t(kQueueWords) * 4; }

const char* natten_amd_last_error(void) { return g_error; }

int natten_amd_window(int query, int kernel_size, int stride, int extent, int is_causal, int32_t* start, int32_t* end) {
  g_error[0] = 0;
  if (!start || !end) return fail("window: null pointer argument");
  if (query < 0 || kernel_size < 1 || stride < 1 || extent < 1)
    return fail("window: query >= 0, kernel_size, stride and extent >= 1 expected");
  // the arithmetic the kernels' set-up runs: stride division by multiply and shift
  *start = na_window_start(query, kernel_size, stride, na_make_div(stride), extent, is_causal != 0);
  *end = na_window_end(query, *start, kernel_size, extent, is_causal != 0);
  return 0;
}

int natten_amd_tile_key_mask(const int32_t* kv_tile_shape, const int32_t* lo, const int32_t* hi, uint64_t* mask) {
  g_error[0] = 0;
  if (!kv_tile_shape || !lo || !hi || !mask) return fail("tile_key_mask: null pointer argument");
  int lg[3], keys = 1;
  for (int a = 0; a < 3; ++a) {
    lg[a] = 0;
    while ((1 << lg[a]) < kv_tile_shape[a]) ++lg[a];
    if (kv_tile_shape[a] < 1 || (1 << lg[a]) != kv_tile_shape[a])
      return fail("tile_key_mask: tile extents must be powers of two, got %d", kv_tile_shape[a]);
    if (lo[a] < 0 || hi[a] < 0 || lo[a] > kv_tile_shape[a] || hi[a] > kv_tile_shape[a])
      return fail("tile_key_mask: bounds must lie in 0 .. extent along dimension %d", a);
    keys *= kv_tile_shape[a];
  }
  if (keys != 64) return fail("tile_key_mask: the tile must hold 64 keys, got %d", keys);
  // the rows the kernels keep in LDS (per half of the wave: the bits its lanes hold logits for) and
  // how their element mask combines them
  uint32_t half[2] = {~uint32_t(0), ~uint32_t(0)};
  int lg_stride = 0;
  for (int a = 0; a < 3; ++a) {
    for (int g = 0; g < 2; ++g)
      half[g] &= na_lane_half_bits(na_keys_at_or_after(lo[a], lg_stride, lg[a]), g) &
                 ~na_lane_half_bits(na_keys_at_or_after(hi[a], lg_stride, lg[a]), g);
    lg_stride += lg[a];
  }
  *mask = na_keys_of_lane_halves(half[0], half[1]);
  return 0;
}

int natten_amd_fna_fully_block_sparse(int na_dim, const int32_t* qkv_shape, const int32_t* kernel_size,
                                      const int32_t* stride, const int32_t* dilation, const int32_t* is_causal,
                                      const int32_t* q_tile_shape, const int32_t* kv_tile_shape, int anchor_kv_tiles,
                                      int32_t* result) {
  g_error[0] = 0;
  if (na_dim < 1 || na_dim > 3) return fail("fna_fully_block_sparse: na_dim must be 1, 2 or 3, got %d", na_dim);
  if (!result) return fail("fna_fully_block_sparse: null pointer argument");
  FnaParams p;
  long long tokens = 0;
  if (int rc = fused_geometry("fna_fully_block_sparse", p, true, na_dim, 1, 32, qkv_shape, kernel_size, stride, dilation,
                              is_causal, q_tile_shape, kv_tile_shape, anchor_kv_tiles, &tokens))
    return rc;
  p.batch = p.num_groups;
  p.heads_q = p.heads_kv = 1;
  set_wg_layout(p, 1);
  *result = fully_block_sparse(p) ? 1 : 0;
  return 0;
}

int natten_amd_fna_wave_box(int na_dim, const int32_t* qkv_shape, const int32_t* kernel_size, const int32_t* stride,
                            const int32_t* dilation, const int32_t* is_causal, const int32_t* q_tile_shape,
                            const int32_t* kv_tile_shape, int anchor_kv_tiles, int32_t* box) {
  g_error[0] = 0;
  if (na_dim < 1 || na_dim > 3) return fail("fna_wave_box: na_dim must be 1, 2 or 3, got %d", na_dim);
  if (!box) return fail("fna_wave_box: null pointer argument");
  FnaParams p;
  long long tokens = 0;
  if (int rc = fused_geometry("fna_wave_box", p, true, na_dim, 1, 32, qkv_shape, kernel_size, stride, dilation, is_causal,
                              q_tile_shape, kv_tile_shape, anchor_kv_tiles, &tokens))
    return rc;
  p.batch = p.num_groups;
  p.heads_q = p.heads_kv = 1;
  set_wg_layout(p, 1);
  for (int a = 0; a < na_dim; ++a) box[a] = 1 << p.wave_box_lg[a];
  return 0;
}

int natten_amd_fna_supported_tiles(int dtype, int head_dim, int32_t* q_sizes, int32_t* kv_sizes, int capacity) {
  if (dtype == NATTEN_AMD_F8E4M3 || dtype == NATTEN_AMD_F8E5M2) {
    if (head_dim != 64 && head_dim != 128) return 0;
    if (capacity > 0 && q_sizes) q_sizes[0] = 128;
    if (capacity > 0 && kv_sizes) kv_sizes[0] = 64;
    return 1;
  }
  if (dtype == NATTEN_AMD_F32) {
    if (head_dim != 32 && head_dim != 64 && head_dim != 128) return 0;
    if (capacity > 0 && q_sizes) q_sizes[0] = 128;
    if (capacity > 0 && kv_sizes) kv_sizes[0] = 64;
    return 1;
  }
  if (dtype != NATTEN_AMD_F16 && dtype != NATTEN_AMD_BF16) return 0;
  if (head_dim != 32 && head_dim != 64 && head_dim != 128) return 0;
  for (int i = 0; i < kNumTileConfigs && i < capacity; ++i) {
    if (q_sizes) q_sizes[i] = kTileConfigs[i].q_tile;
    if (kv_sizes) kv_sizes[i] = kTileConfigs[i].kv_tile;
  }
  return kNumTileConfigs;
}

int natten_amd_fna_forward(const void* q, const void* k, const void* v, void* out, float* lse, int dtype, int na_dim,
                           int batch, int seqlen_q, int seqlen_kv, int heads_q, int heads_kv, int head_dim,
                           const int32_t* q_shape, const int32_t* kv_shape, const int32_t* qkv_shape,
                           const int32_t* kernel_size, const int32_t* stride, const int32_t* dilation,
                           const int32_t* is_causal, const int32_t* q_tile_shape, const int32_t* kv_tile_shape,
                           float scale, const float* q_scale, const float* k_scale, const float* v_scale,
                           int run_persistent, void* workspace, uint64_t workspace_bytes, void* stream) {
  g_error[0] = 0;
  if (na_dim < 1 || na_dim > 3) return fail("fna_forward: na_dim must be 1, 2 or 3, got %d", na_dim);
  WorkQueue queues;
  if (int rc = queue_workspace("fna_forward", run_persistent, workspace, workspace_bytes, &queues)) return rc;
  if (int rc = check_common("fna_forward", q, k, v, out, lse, batch, seqlen_q, seqlen_kv, heads_q, heads_kv, head_dim))
    return rc;
  if (!q_shape || !kv_shape || !qkv_shape || !kernel_size || !stride || !dilation || !is_causal || !q_tile_shape ||
      !kv_tile_shape)
    return fail("fna_forward: null shape argument");
  FnaParams p;
  if (int rc = fill_fna_params("fna_forward", p, na_dim, q_shape, kv_shape, qkv_shape, kernel_size, stride, dilation,
                               is_causal, q_tile_shape, kv_tile_shape))
    return rc;
  int qs[3] = {1, 1, 1}, ks[3] = {1, 1, 1};
  for (int a = 0; a < na_dim; ++a) {
    qs[a] = q_shape[a];
    ks[a] = kv_shape[a];
  }
  if (prod3(qs) != seqlen_q || prod3(ks) != seqlen_kv)
    return fail("fna_forward: seqlen_q / seqlen_kv do not match q_shape / kv_shape (%d vs %d, %d vs %d)", prod3(qs),
                seqlen_q, prod3(ks), seqlen_kv);
  if (batch % p.num_groups != 0)
    return fail("fna_forward: batch (%d) is not a multiple of the number of dilation groups (%d)", batch, p.num_groups);
  p.q = q;
  p.k = k;
  p.v = v;
  p.o = out;
  p.lse = lse;
  p.batch = batch;
  p.heads_q = heads_q;
  p.heads_kv = heads_kv;
  p.seqlen_q = seqlen_q;
  p.seqlen_kv = seqlen_kv;
  p.scale = scale;
  p.q_scale = q_scale;
  p.k_scale = k_scale;
  p.v_scale = v_scale;
  set_wg_layout(p, 1);
  return dispatch_dtype(p, dtype, head_dim, prod3(p.q_tile), prod3(p.kv_tile), static_cast<hipStream_t>(stream), queues);
}

namespace {
// The part of natten_amd_fna_forward_fused that needs no operands: checks the shapes and fills the
// launch geometry of the one-launch route (`sixteen_bit`: fp16 / bf16 operands, which take any extent).
int fused_geometry(const char* what, FnaParams& p, bool sixteen_bit, int na_dim, int heads_kv, int head_dim,
                   const int32_t* qkv_shape, const int32_t* kernel_size, const int32_t* stride, const int32_t* dilation,
                   const int32_t* is_causal, const int32_t* q_tile_shape, const int32_t* kv_tile_shape, int anchor_kv_tiles,
                   long long* tokens_out) {
  if (!qkv_shape || !kernel_size || !stride || !dilation || !is_causal || !q_tile_shape || !kv_tile_shape)
    return fail("%s: null shape argument", what);
  int qs[3] = {1, 1, 1}, ks[3] = {1, 1, 1};
  long long tokens = 1;
  // Extents that are not multiples of dilation x KV tile: some KV tile would reach past its
  // dilation group.  1: every group is at least a KV tile wide everywhere, any kernel instance will
  // do (such tiles are gathered from one tile extent before the group's end).  2: a group is
  // narrower than the KV tile somewhere, only the instance that clamps its gathers will do.
  int edge = 0;
  for (int a = 0; a < na_dim; ++a) {
    if (qkv_shape[a] < 1 || dilation[a] < 1 || q_tile_shape[a] < 1 || kv_tile_shape[a] < 1)
      return fail("%s: invalid parameter along dimension %d", what, a);
    // dilation groups may differ in extent by one; the padded per-group layouts cover the largest
    const int ext = na_ceil_div(qkv_shape[a], dilation[a]);
    if (qkv_shape[a] % dilation[a] != 0 || ext % kv_tile_shape[a] != 0) edge = edge > 1 ? edge : 1;
    if (qkv_shape[a] / dilation[a] < kv_tile_shape[a]) edge = 2;
    qs[a] = na_ceil_div(ext, q_tile_shape[a]) * q_tile_shape[a];
    ks[a] = na_ceil_div(ext, kv_tile_shape[a]) * kv_tile_shape[a];
    tokens *= qkv_shape[a];
  }
  if (edge != 0) {
    long long qt = 1, kvt = 1;
    for (int a = 0; a < na_dim; ++a) {
      qt *= q_tile_shape[a];
      kvt *= kv_tile_shape[a];
    }
    if (edge == 2 && !sixteen_bit)
      return fail("%s: a dilation group narrower than the KV tile needs fp16 / bf16 operands; use the token-permuted "
                  "entry point", what);
    if (edge == 2 && (qt != 128 || kvt != 64))
      return fail("%s: a dilation group narrower than the KV tile needs tiles of 128 x 64 tokens (got %lld x %lld); use "
                  "the token-permuted entry point", what, qt, kvt);
  }
  if (tokens > 0x7fffffffLL) return fail("%s: more than 2^31 tokens per batch", what);
  if (int rc = fill_fna_params(what, p, na_dim, qs, ks, qkv_shape, kernel_size, stride, dilation, is_causal, q_tile_shape,
                               kv_tile_shape))
    return rc;
  // per-lane byte offsets inside a KV tile are 32-bit
  long long span = 0;
  for (int a = 0; a < 3; ++a) span += (long long)(p.kv_tile[a] - 1) * p.dil[a] * p.tok_stride[a];
  if ((span + 1) * heads_kv * head_dim * 2 + 8192 >= 0x7fffffffLL)  // (16-bit rows; 8-bit ones are shorter)
    return fail("%s: a KV tile spans more than 2^31 bytes of the input; use the token-permuted entry point", what);
  p.seqlen_q = prod3(qs);
  p.seqlen_kv = prod3(ks);
  p.fused = p.token_rows = 1;
  p.edge = edge;
  // tiles laid out from the window's first key: needs every dilation group at least a KV tile wide
  p.anchor = (anchor_kv_tiles != 0 && edge != 2) ? 1 : 0;
  for (int a = 0; a < na_dim; ++a)
    if (qkv_shape[a] / dilation[a] < kv_tile_shape[a]) p.anchor = 0;
  p.tokens = int(tokens);
  *tokens_out = tokens;
  return 0;
}

// natten_amd_fna_forward_fused after its workspace has been resolved (`queues` == nullptr: a workgroup per Q tile)
int fna_forward_fused_impl(const void* q, const void* k, const void* v, void* out, float* lse, int dtype, int na_dim,
                           int batch, int heads_q, int heads_kv, int head_dim, const int32_t* qkv_shape,
                           const int32_t* kernel_size, const int32_t* stride, const int32_t* dilation,
                           const int32_t* is_causal, const int32_t* q_tile_shape, const int32_t* kv_tile_shape,
                           float scale, const float* q_scale, const float* k_scale, const float* v_scale,
                           int anchor_kv_tiles, WorkQueue queues, void* stream, int kv_splits = 1,
                           const void* ctx_k = nullptr, const void* ctx_v = nullptr, int ctx_len = 0) {
  FnaParams p;
  long long tokens = 0;
  if (heads_kv < 1 || head_dim < 1) return fail("fna_forward_fused: head counts and head_dim must be positive");
  if (int rc = fused_geometry("fna_forward_fused", p, dtype == NATTEN_AMD_F16 || dtype == NATTEN_AMD_BF16, na_dim, heads_kv,
                              head_dim, qkv_shape, kernel_size, stride, dilation, is_causal, q_tile_shape, kv_tile_shape,
                              anchor_kv_tiles, &tokens))
    return rc;
  if (int rc = check_common("fna_forward_fused", q, k, v, out, lse, batch, p.seqlen_q, p.seqlen_kv, heads_q, heads_kv,
                            head_dim, dtype == NATTEN_AMD_F16 || dtype == NATTEN_AMD_BF16))
    return rc;
  p.q = q;
  p.k = k;
  p.v = v;
  p.o = out;
  p.lse = lse;
  p.batch = batch * p.num_groups;
  p.heads_q = heads_q;
  p.heads_kv = heads_kv;
  p.row_dim = head_dim;
  p.scale = scale;
  p.q_scale = q_scale;
  p.k_scale = k_scale;
  p.v_scale = v_scale;
  if (ctx_len > 0) {
    p.ctx_k = ctx_k;
    p.ctx_v = ctx_v;
    p.ctx_len = ctx_len;
  }
  if (kv_splits > 1) {
    // out and lse hold kv_splits results of the full shape, one after the other
    p.kv_splits = kv_splits;
    p.split_first = -1;
    p.o_split_stride = (int64_t)batch * tokens * heads_q * head_dim;
    p.lse_split_stride = (int64_t)batch * tokens * heads_q;
  }
  set_wg_layout(p, 1);
  return dispatch_dtype(p, dtype, head_dim, prod3(p.q_tile), prod3(p.kv_tile), static_cast<hipStream_t>(stream), queues);
}
}  // namespace

int natten_amd_fna_forward_fused(const void* q, const void* k, const void* v, void* out, float* lse, int dtype,
                                 int na_dim, int batch, int heads_q, int heads_kv, int head_dim,
                                 const int32_t* qkv_shape, const int32_t* kernel_size, const int32_t* stride,
                                 const int32_t* dilation, const int32_t* is_causal, const int32_t* q_tile_shape,
                                 const int32_t* kv_tile_shape, float scale, const float* q_scale,
                                 const float* k_scale, const float* v_scale, int anchor_kv_tiles, int run_persistent,
                                 void* workspace, uint64_t workspace_bytes, void* stream) {
  g_error[0] = 0;
  if (na_dim < 1 || na_dim > 3) return fail("fna_forward_fused: na_dim must be 1, 2 or 3, got %d", na_dim);
  WorkQueue queues;
  if (int rc = queue_workspace("fna_forward_fused", run_persistent, workspace, workspace_bytes, &queues)) return rc;
  return fna_forward_fused_impl(q, k, v, out, lse, dtype, na_dim, batch, heads_q, heads_kv, head_dim, qkv_shape,
                                kernel_size, stride, dilation, is_causal, q_tile_shape, kv_tile_shape, scale, q_scale,
                                k_scale, v_scale, anchor_kv_tiles, queues, stream);
}

extern "C++" {
template <bool WIDE>
static void launch_f32_direct(const FnaF32Params& p, dim3 grid, hipStream_t s) {
  switch (p.head_dim) {
    case 32: hipLaunchKernelGGL((fna_fwd_f32_direct_kernel<32, false, WIDE>), grid, dim3(256), 0, s, p); break;
    case 64: hipLaunchKernelGGL((fna_fwd_f32_direct_kernel<64, false, WIDE>), grid, dim3(256), 0, s, p); break;
    case 128: hipLaunchKernelGGL((fna_fwd_f32_direct_kernel<128, false, WIDE>), grid, dim3(256), 0, s, p); break;
    default:
      if (p.head_dim < 32)
        hipLaunchKernelGGL((fna_fwd_f32_direct_kernel<32, true, WIDE>), grid, dim3(256), 0, s, p);
      else if (p.head_dim < 64)
        hipLaunchKernelGGL((fna_fwd_f32_direct_kernel<64, true, WIDE>), grid, dim3(256), 0, s, p);
      else
        hipLaunchKernelGGL((fna_fwd_f32_direct_kernel<128, true, WIDE>), grid, dim3(256), 0, s, p);
  }
}
}  // extern "C++"

int natten_amd_fna_forward_f32(const void* q, const void* k, const void* v, void* out, float* lse, int na_dim, int batch,
                               int heads_q, int heads_kv, int head_dim, const int32_t* qkv_shape,
                               const int32_t* kernel_size, const int32_t* stride, const int32_t* dilation,
                               const int32_t* is_causal, float scale, void* stream) {
  g_error[0] = 0;
  const char* what = "fna_forward_f32";
  if (na_dim < 1 || na_dim > 3) return fail("%s: na_dim must be 1, 2 or 3, got %d", what, na_dim);
  if (!qkv_shape || !kernel_size || !stride || !dilation || !is_causal) return fail("%s: null shape argument", what);
  if (head_dim < 8 || head_dim > 128 || head_dim % 8 != 0)
    return fail("%s: head_dim must be a multiple of 8 from 8 to 128, got %d", what, head_dim);
  if (int rc = check_common(what, q, k, v, out, lse, batch, 1, 1, heads_q, heads_kv, 32)) return rc;
  FnaF32Params p;
  memset(&p, 0, sizeof(p));
  p.num_groups = 1;
  p.dims = na_dim;
  long long tokens = 1;
  for (int a = 0; a < 3; ++a) {
    const bool used = a < na_dim;
    const int X = used ? qkv_shape[a] : 1;
    p.ksize[a] = used ? kernel_size[a] : 1;
    p.stride[a] = used ? stride[a] : 1;
    p.dil[a] = used ? dilation[a] : 1;
    p.causal[a] = used ? (is_causal[a] != 0) : 0;
    if (X < 1 || p.dil[a] < 1 || p.stride[a] < 1 || (used && p.ksize[a] < 2))
      return fail("%s: invalid parameter along dimension %d", what, a);
    if ((long long)p.ksize[a] * p.dil[a] > X)
      return fail("%s: kernel_size * dilation exceeds the input along dimension %d (%d * %d > %d)", what, a, p.ksize[a],
                  p.dil[a], X);
    if (p.stride[a] > p.ksize[a])
      return fail("%s: stride exceeds kernel_size along dimension %d (%d > %d)", what, a, p.stride[a], p.ksize[a]);
    p.ext_base[a] = X / p.dil[a];
    p.ext_rem[a] = X % p.dil[a];
    p.num_groups *= p.dil[a];
    tokens *= X;
    if (tokens > 0x7fffffffLL) return fail("%s: more than 2^31 tokens per batch", what);
    p.d_stride[a] = na_make_div(p.stride[a]);
    p.d_dil[a] = na_make_div(p.dil[a]);
  }
  p.tok_stride[2] = 1;
  p.tok_stride[1] = na_dim > 2 ? qkv_shape[2] : 1;
  p.tok_stride[0] = (na_dim > 1 ? qkv_shape[1] : 1) * p.tok_stride[1];
  p.tokens = int(tokens);
  p.q = static_cast<const float*>(q);
  p.k = static_cast<const float*>(k);
  p.v = static_cast<const float*>(v);
  p.o = static_cast<float*>(out);
  p.lse = lse;
  p.heads_q = heads_q;
  p.heads_kv = heads_kv;
  p.head_dim = head_dim;
  p.scale = scale;
  choose_f32_boxes(p);
  long long waves = (long long)batch * heads_q * p.num_groups;
  p.num_boxes = 1;
  for (int a = 0; a < 3; ++a) {
    const int ext = p.ext_base[a] + (p.ext_rem[a] > 0);
    p.q_boxes[a] = (ext + (1 << p.q_lg[a]) - 1) >> p.q_lg[a];
    p.d_q_boxes[a] = na_make_div(p.q_boxes[a]);
    p.num_boxes *= p.q_boxes[a];  // (at most the tokens of a batch entry)
  }
  waves *= p.num_boxes;
  const long long wgs_per_xcd = (waves + 4 * kNumXcd - 1) / (4 * kNumXcd);
  if (waves > 0x7fffff00LL) return fail("%s: problem needs more than 2^31 waves", what);
  p.waves = int(waves);
  p.wgs_per_xcd = int(wgs_per_xcd);
  p.d_boxes = na_make_div(p.num_boxes);
  p.d_heads_q = na_make_div(heads_q);
  p.d_q_per_kv = na_make_div(heads_q / heads_kv);
  p.d_num_groups = na_make_div(p.num_groups);
  const dim3 grid((unsigned)(wgs_per_xcd * kNumXcd));
  hipStream_t s = static_cast<hipStream_t>(stream);
  // A block's rows lie within 32-bit byte offsets of its first one, or the launch takes the instances that form 64-bit ones
  long long span = 0;
  for (int a = 0; a < 3; ++a)
    span += (long long)(na_min(1 << p.kv_lg[a], p.ext_base[a] + (p.ext_rem[a] > 0)) - 1) * p.dil[a] * p.tok_stride[a];
  if ((span + 1) * heads_kv * head_dim * 4 < (1LL << 32)) launch_f32_direct<false>(p, grid, s);
  else launch_f32_direct<true>(p, grid, s);
  return check_launch(what);
}

int natten_amd_fna_forward_fused_split(const void* q, const void* k, const void* v, void* out_parts, float* lse_parts,
                                       int dtype, int na_dim, int batch, int heads_q, int heads_kv, int head_dim,
                                       const int32_t* qkv_shape, const int32_t* kernel_size, const int32_t* stride,
                                       const int32_t* dilation, const int32_t* is_causal,
                                       const int32_t* q_tile_shape, const int32_t* kv_tile_shape, float scale,
                                       int anchor_kv_tiles, int kv_splits, void* stream) {
  g_error[0] = 0;
  const char* what = "fna_forward_fused_split";
  if (na_dim < 1 || na_dim > 3) return fail("%s: na_dim must be 1, 2 or 3, got %d", what, na_dim);
  if (kv_splits < 2 || kv_splits > 8) return fail("%s: kv_splits must be 2 .. 8, got %d", what, kv_splits);
  if (dtype != NATTEN_AMD_F16 && dtype != NATTEN_AMD_BF16)
    return fail("%s: KV splits need fp16 / bf16 operands, got dtype code %d", what, dtype);
  if (!q_tile_shape || !kv_tile_shape) return fail("%s: null shape argument", what);
  long long qt = 1, kvt = 1;
  for (int a = 0; a < na_dim; ++a) {
    qt *= q_tile_shape[a];
    kvt *= kv_tile_shape[a];
  }
  if (qt != 128 || kvt != 64)
    return fail("%s: KV splits exist for Q tiles of 128 and KV tiles of 64 tokens, got %lld and %lld", what, qt, kvt);
  return fna_forward_fused_impl(q, k, v, out_parts, lse_parts, dtype, na_dim, batch, heads_q, heads_kv, head_dim, qkv_shape,
                                kernel_size, stride, dilation, is_causal, q_tile_shape, kv_tile_shape, scale, nullptr,
                                nullptr, nullptr, anchor_kv_tiles, WorkQueue{}, stream, kv_splits);
}

int natten_amd_fna_forward_fused_paired(const void* q, const void* k, const void* v, void* out, float* lse, int dtype,
                                        int na_dim, int batch, int heads_q, int heads_kv, int head_dim,
                                        const int32_t* qkv_shape, const int32_t* kernel_size, const int32_t* stride,
                                        const int32_t* dilation, const int32_t* is_causal, const int32_t* q_tile_shape,
                                        const int32_t* kv_tile_shape, float scale, int anchor_kv_tiles, void* stream) {
  g_error[0] = 0;
  const char* what = "fna_forward_fused_paired";
  if (na_dim < 1 || na_dim > 3) return fail("%s: na_dim must be 1, 2 or 3, got %d", what, na_dim);
  if (dtype != NATTEN_AMD_F16 && dtype != NATTEN_AMD_BF16) return fail("%s: fp16 / bf16 operands, got dtype code %d", what, dtype);
  if (head_dim != 64 && head_dim != 128) return fail("%s: head_dim must be 64 or 128, got %d", what, head_dim);
  WorkQueue launch;
  launch.paired = true;
  return fna_forward_fused_impl(q, k, v, out, lse, dtype, na_dim, batch, heads_q, heads_kv, head_dim, qkv_shape, kernel_size,
                                stride, dilation, is_causal, q_tile_shape, kv_tile_shape, scale, nullptr, nullptr, nullptr,
                                anchor_kv_tiles, launch, stream);
}

int natten_amd_fna_forward_fused_context(const void* q, const void* k, const void* v, const void* context_k,
                                         const void* context_v, void* out, float* lse, int dtype, int na_dim, int batch,
                                         int context_len, int heads_q, int heads_kv, int head_dim, const int32_t* qkv_shape,
                                         const int32_t* kernel_size, const int32_t* stride, const int32_t* dilation,
                                         const int32_t* is_causal, const int32_t* q_tile_shape,
                                         const int32_t* kv_tile_shape, float scale, int run_persistent, void* workspace,
                                         uint64_t workspace_bytes, void* stream) {
  g_error[0] = 0;
  const char* what = "fna_forward_fused_context";
  if (na_dim < 1 || na_dim > 3) return fail("%s: na_dim must be 1, 2 or 3, got %d", what, na_dim);
  WorkQueue queues;
  if (int rc = queue_workspace(what, run_persistent, workspace, workspace_bytes, &queues)) return rc;
  if (!context_k || !context_v) return fail("%s: null pointer argument", what);
  if ((reinterpret_cast<uintptr_t>(context_k) | reinterpret_cast<uintptr_t>(context_v)) & 15)
    return fail("%s: context_k and context_v must be 16-byte aligned", what);
  if (context_len < 64) return fail("%s: the context must hold at least a KV tile (64 keys), got %d", what, context_len);
  if (dtype != NATTEN_AMD_F16 && dtype != NATTEN_AMD_BF16)
    return fail("%s: fp16 / bf16 operands expected, got dtype code %d", what, dtype);
  return fna_forward_fused_impl(q, k, v, out, lse, dtype, na_dim, batch, heads_q, heads_kv, head_dim, qkv_shape,
                                kernel_size, stride, dilation, is_causal, q_tile_shape, kv_tile_shape, scale, nullptr,
                                nullptr, nullptr, /*anchor_kv_tiles=*/1, queues, stream, 1, context_k, context_v, context_len);
}

namespace {
// Device address of `scratch` on the current device, looked up once per device (each GPU holds
// its own copy of the array at its own address); nullptr + error message on failure.
uint32_t* static_scratch(const char* what) {
  constexpr int kMaxDevices = 64;
  static uint32_t* ptrs[kMaxDevices] = {};
  static std::mutex lock;
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    fail("%s: cannot identify the current device (%s, device %d)", what, hipGetErrorString(e), dev);
    return nullptr;
  }
  std::lock_guard<std::mutex> guard(lock);
  if (ptrs[dev] == nullptr) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr) {
      fail("%s: hipGetSymbolAddress(scratch) failed on device %d: %s", what, dev, hipGetErrorString(e));
      return nullptr;
    }
    ptrs[dev] = static_cast<uint32_t*>(ptr);
  }
  return ptrs[dev];
}
}  // namespace

int natten_amd_fna_forward_fused_static(const void* q, const void* k, const void* v, void* out, float* lse, int dtype,
                                        int na_dim, int batch, int heads_q, int heads_kv, int head_dim,
                                        const int32_t* qkv_shape, const int32_t* kernel_size, const int32_t* stride,
                                        const int32_t* dilation, const int32_t* is_causal,
                                        const int32_t* q_tile_shape, const int32_t* kv_tile_shape, float scale,
                                        const float* q_scale, const float* k_scale, const float* v_scale,
                                        void* stream) {
  g_error[0] = 0;
  const char* what = "fna_forward_fused_static";
  if (na_dim < 1 || na_dim > 3) return fail("%s: na_dim must be 1, 2 or 3, got %d", what, na_dim);
  if (!qkv_shape || !q_tile_shape || !kv_tile_shape) return fail("%s: null shape argument", what);
  // only the work-queue kernel uses the scratch array: 16-bit operands, 128 x 64 token tiles
  if (dtype != NATTEN_AMD_F16 && dtype != NATTEN_AMD_BF16)
    return fail("%s: the work-queue kernel takes fp16 / bf16 operands, got dtype code %d", what, dtype);
  long long qt = 1, kvt = 1, q_tiles = 1;
  for (int a = 0; a < na_dim; ++a) {
    if (q_tile_shape[a] < 1 || kv_tile_shape[a] < 1 || qkv_shape[a] < 1 || !dilation || dilation[a] < 1)
      return fail("%s: invalid parameter along dimension %d", what, a);
    qt *= q_tile_shape[a];
    kvt *= kv_tile_shape[a];
    const long long ext = (qkv_shape[a] + dilation[a] - 1) / dilation[a];
    q_tiles *= (ext + q_tile_shape[a] - 1) / q_tile_shape[a] * dilation[a];
  }
  if (qt != 128 || kvt != 64)
    return fail("%s: the work-queue kernel exists for Q tiles of 128 and KV tiles of 64 tokens, got %lld and %lld", what, qt,
                kvt);
  // the queues hold 32-bit positions: at most 2^28 Q tiles per queue (2^31 in all); the array itself never grows
  if (batch < 1 || heads_q < 1 || q_tiles * batch * heads_q > (1LL << 31) - 4096)
    return fail("%s: %lld Q tiles x %d x %d exceed the 2^31 positions the static queues can count", what, q_tiles, batch,
                heads_q);
  WorkQueue queues;  // (cleared by a kernel before every launch: the array is shared by all callers on this GPU)
  queues.counters = static_scratch(what);
  if (queues.counters == nullptr) return 1;
  return fna_forward_fused_impl(q, k, v, out, lse, dtype, na_dim, batch, heads_q, heads_kv, head_dim, qkv_shape,
                                kernel_size, stride, dilation, is_causal, q_tile_shape, kv_tile_shape, scale, q_scale,
                                k_scale, v_scale, /*anchor_kv_tiles=*/1, queues, stream);
}

// Dense attention is the 1-D neighborhood problem whose window is the whole key sequence:
// non-causal windows are [0, seqlen_kv), causal ones [0, min(i + 1, seqlen_kv)).
static void fill_dense_fwd(FnaParams& p, int batch, int seqlen_q, int seqlen_kv, int heads_q, int heads_kv, int is_causal) {
  constexpr int QT = 128, KVT = 64;
  memset(&p, 0, sizeof(p));
  for (int a = 0; a < 3; ++a) {
    p.qkv_shape[a] = p.ksize[a] = p.stride[a] = p.dil[a] = p.q_tile[a] = p.kv_tile[a] = p.q_tiled[a] = p.kv_tiled[a] = 1;
  }
  p.ksize[0] = seqlen_kv;  // (a one-key window is the unused-dimension case of the window arithmetic)
  p.qkv_shape[0] = seqlen_kv;
  p.causal[0] = is_causal != 0;
  p.q_tile[0] = QT;
  p.kv_tile[0] = KVT;
  p.q_tiled[0] = na_ceil_div(seqlen_q, QT);
  p.kv_tiled[0] = na_ceil_div(seqlen_kv, KVT);
  p.edge = (seqlen_kv % KVT != 0 && seqlen_kv >= KVT) ? 1 : 0;
  p.token_rows = p.tok_stride[0] = 1;
  p.num_groups = 1;
  p.batch = batch;
  p.heads_q = heads_q;
  p.heads_kv = heads_kv;
  p.seqlen_q = seqlen_q;
  p.seqlen_kv = seqlen_kv;
  set_wg_layout(p, 1);
}

static int attention_forward(const void* q, const void* k, const void* v, void* out, float* lse, int dtype, int batch,
                             int seqlen_q, int seqlen_kv, int heads_q, int heads_kv, int head_dim, int is_causal, float scale,
                             const float* q_scale, const float* k_scale, const float* v_scale, void* stream, int split_positions,
                             int kv_splits, float* parts, float* lse_parts) {
  g_error[0] = 0;
  if (int rc = check_common("attention_forward", q, k, v, out, lse, batch, seqlen_q, seqlen_kv, heads_q, heads_kv,
                            head_dim, dtype == NATTEN_AMD_F16 || dtype == NATTEN_AMD_BF16))
    return rc;
  FnaParams p;
  fill_dense_fwd(p, batch, seqlen_q, seqlen_kv, heads_q, heads_kv, is_causal);
  p.q = q;
  p.k = k;
  p.v = v;
  p.o = out;
  p.lse = lse;
  p.row_dim = head_dim;
  p.scale = scale;
  p.q_scale = q_scale;
  p.k_scale = k_scale;
  p.v_scale = v_scale;
  if (kv_splits > 1) {
    p.kv_splits = kv_splits;
    p.split_grid = split_positions;
    p.split_parts = parts;
    p.split_lse = lse_parts;
  }
  return dispatch_dtype(p, dtype, head_dim, 128, 64, static_cast<hipStream_t>(stream));
}

int natten_amd_attention_forward(const void* q, const void* k, const void* v, void* out, float* lse, int dtype,
                                 int batch, int seqlen_q, int seqlen_kv, int heads_q, int heads_kv, int head_dim,
                                 int is_causal, float scale, const float* q_scale, const float* k_scale,
                                 const float* v_scale, void* stream) {
  return attention_forward(q, k, v, out, lse, dtype, batch, seqlen_q, seqlen_kv, heads_q, heads_kv, head_dim, is_causal, scale,
                           q_scale, k_scale, v_scale, stream, 0, 1, nullptr, nullptr);
}

int natten_amd_attention_split_plan(int batch, int seqlen_q, int seqlen_kv, int heads_q, int head_dim, int is_causal,
                                    int32_t* split_positions, int32_t* kv_splits) {
  g_error[0] = 0;
  const char* what = "attention_split_plan";
  if (!split_positions || !kv_splits) return fail("%s: null pointer argument", what);
  if (batch < 1 || seqlen_q < 1 || seqlen_kv < 1 || heads_q < 1 || head_dim < 1)
    return fail("%s: batch, sequence lengths, heads and head_dim must be positive", what);
  *split_positions = 0;
  *kv_splits = 1;
  const int kv_tiles = na_ceil_div(seqlen_kv, 64);
  const long long q_tiles = na_ceil_div(seqlen_q, 128), n = q_tiles * heads_q * batch;
  // One batch entry is never split: a packed call promises the bits of a dense call on each of its sequences alone.
  const int slots = resident_workgroups(2) / kNumXcd, cus = resident_workgroups(1) / kNumXcd;
  if (batch < 2 || kv_tiles < 16 || n / (slots * kNumXcd) > 12) return 0;
  FnaParams p;
  fill_dense_fwd(p, batch, seqlen_q, seqlen_kv, heads_q, heads_q, is_causal);
  // Every XCD works off its own launch positions (see fna_fwd_tile): the one with the most sets the time.  In an XCD's
  // positions, where the shares are uneven (5 x 3100 tokens, H 5, D 128: 131 us in one launch; counted over the chip, 113 of 625
  // Q tiles were split four ways, and the fullest XCD still began another round: 149).  Positions without a Q tile, at the end
  // of a short group, count: workgroups go to the compute units in order, and the room that such a one leaves is not
  // refilled out of turn (3 x 3712 tokens, H 6, D 64, 68 Q tiles in 70 positions: with 4 of them split, so that 64 Q tiles
  // are left whole, 105 us, with 6 80, in one launch 82).
  auto position_at = [&](int xcd, int local) {  // 1 where the position belongs to a group
    return local / p.wg_group * kNumXcd + xcd < p.total_groups ? 1 : 0;
  };
  const int positions = na_ceil_div(p.total_groups, kNumXcd) * p.wg_group;  // of an XCD
  int share[kNumXcd] = {}, most = 0;
  for (int x = 0; x < kNumXcd; ++x) {
    for (int i = 0; i < positions; ++i) share[x] += position_at(x, i);
    most = na_max(most, share[x]);
  }
  // An XCD takes `slots` workgroups of the split launch at a time (two waves per SIMD at every head dim).  What does not
  // fill a last round is split so that it does, where that saves a twelfth of the whole and more than the merge takes
  // (2 x 4097 tokens, H 16, D 64, a third round of 4 Q tiles: 176 us, 153 with them split 8 ways; 2 x 9000, H 4, D 64: 226
  // and 177; 2 x 5000, H 8, D 128: 205 and 194).  In KV tiles of a workgroup that shares its compute unit (0.62 us at head
  // dim 64, 1.05 at 128): a workgroup alone on one takes three quarters, the second launch eight.  The second
  // launch and the workspace also take the host 5 us: launches under 40 KV tiles (2 x 1000 tokens, H 4, D 128: 19.6 us, split
  // 23.9; 2 x 2000, H 4, D 32: 21.0 and 26.2) are over by then.
  int round_slots = slots;
  if (most > slots) {
    if (is_causal) return 0;  // rounds even out by themselves: the longest walks start first
    if (fwd_max_waves(head_dim <= 32 ? 32 : head_dim, fully_block_sparse(p)) > 2) {
      // The one launch holds three waves per SIMD, and whatever is split, every Q tile loses the third.
      const int held = resident_workgroups(3) / kNumXcd;
      const int left = most % slots;
      if (head_dim <= 32) {
        // Rounds are those of the one launch.  One and up to an eighth: faster split from some 128 KV tiles on (us, one launch /
        // split: 792 Q tiles of 65 KV tiles 97.5 / 99.5, of 125 179 / 174, of 197 279 / 266; 840 of 80 119 / 119, of 125 180 / 172;
        // 888 of 125 181 / 180); more rounds lose more (1562 of 141 340 / 374).
        if (most / held != 1 || most % held * 8 > held || kv_tiles < 128) return 0;
        round_slots = held;
      } else if (most > held) {
        // Two or three rounds and a sixteenth or less: 1040 Q tiles of 100 KV tiles 238 / 237, of 140 330 / 317, of 200 467 / 441; 1568
        // of 140 482 / 465; 1088 of 100 244 / 242, of 140 337 / 332; 2080 of 140 617 / 615; 2600 of 200 1073 / 1080.
        if (left * 16 > slots || most > 4 * slots || kv_tiles < 128) return 0;
      } else if (left * 4 > slots || kv_tiles < 40 + 256 * left / slots) {
        // One round there, two here: the walk has to be long for what is left over to be worth the third wave (528 Q tiles of 48
        // KV tiles 69.8 / 65.4; 544 of 48 69.8 / 71.0, of 72 101.9 / 98.5; 576 of 48 71.7 / 73.8, of 72 103.3 / 99.1, of 144
        // 200 / 183; 640 of 40 64 / 68, of 72 106.2 / 108.6, of 100 145.7 / 144.7; 704 of 176 258 / 272).
        return 0;
      }
    }
  }
  const int full = most / round_slots;
  if (most % round_slots == 0) return 0;
  // the fewest positions at the end of every XCD's that leave no XCD more than whole rounds
  int last = 0;
  for (bool over = true; over;) {
    ++last;
    over = false;
    for (int x = 0; x < kNumXcd; ++x) {
      share[x] -= position_at(x, positions - last);
      over = over || share[x] > full * round_slots;
    }
  }
  const double round = last <= cus ? 0.75 * kv_tiles : kv_tiles;
  // The parts are written and read once, which takes 12 us for 60 of them on every XCD at head dim 128.  Two and three
  // ways, which fill the chip with parts, lost without this (us, one launch / split: 224 Q tiles of 56 KV tiles, head
  // dim 128, two ways 57.5 / 65.4, 204 of 72 69.7 / 76.1, 222 of 74 77.8 / 83.1; head dim 64, 240 of 55 38.1 / 43.0; 630 of 42 at
  // 128, three ways, 117.9 / 125.2).
  const double part = 0.0015 * (head_dim + 1);
  double least = 1e30;
  int best = 1;
  for (int s = 2; s <= 16 && last * s <= slots && kv_tiles / s >= 3; ++s) {
    const double t = (last * s <= cus ? 0.75 : 1.0) * na_ceil_div(kv_tiles, s) + 8 + part * last * s;
    if (t < least) {
      least = t;
      best = s;
    }
  }
  if (best == 1 || full * kv_tiles + round < 40 || least > round - (full * kv_tiles + round) / 12) return 0;
  *split_positions = last * kNumXcd;
  *kv_splits = best;
  return 0;
}

int natten_amd_attention_forward_split(const void* q, const void* k, const void* v, void* out, float* lse, float* parts,
                                       uint64_t parts_floats, int split_positions, int kv_splits, int dtype, int batch,
                                       int seqlen_q, int seqlen_kv, int heads_q, int heads_kv, int head_dim, int is_causal,
                                       float scale, const float* q_scale, const float* k_scale, const float* v_scale,
                                       void* stream) {
  g_error[0] = 0;
  const char* what = "attention_forward_split";
  if (!parts || (reinterpret_cast<uintptr_t>(parts) & 15)) return fail("%s: parts must be a 16-byte aligned workspace", what);
  if (kv_splits < 2 || kv_splits > 16) return fail("%s: kv_splits must be 2 .. 16, got %d", what, kv_splits);
  if (split_positions < kNumXcd || split_positions % kNumXcd != 0)
    return fail("%s: split_positions must be a multiple of %d, got %d", what, kNumXcd, split_positions);
  if (seqlen_kv < 64) return fail("%s: at least 64 keys expected, got %d", what, seqlen_kv);
  if (dtype != NATTEN_AMD_F16 && dtype != NATTEN_AMD_BF16) return fail("%s: fp16 / bf16 operands expected, got dtype code %d", what, dtype);
  const uint64_t rows = uint64_t(split_positions) * uint64_t(kv_splits) * 128;
  if (head_dim < 1 || parts_floats < rows * (uint64_t(head_dim) + 1))
    return fail("%s: parts must hold split_positions * kv_splits * 128 rows of head_dim + 1 floats, got %llu floats", what,
                (unsigned long long)parts_floats);
  return attention_forward(q, k, v, out, lse, dtype, batch, seqlen_q, seqlen_kv, heads_q, heads_kv, head_dim, is_causal, scale,
                           q_scale, k_scale, v_scale, stream, split_positions, kv_splits, parts, parts + rows * uint64_t(head_dim));
}

// clear: rows that belong to no sequence become zeros
static int attention_forward_varlen(const void* q, const void* k, const void* v, void* out, float* lse, int dtype,
                                    int num_seqs, int total_seqlen_q, int total_seqlen_kv, int max_seqlen_q,
                                    int max_seqlen_kv, int heads_q, int heads_kv, int head_dim,
                                    const int32_t* cumulative_seqlen_q, const int32_t* cumulative_seqlen_kv,
                                    int is_causal, float scale, const float* q_scale, const float* k_scale,
                                    const float* v_scale, void* stream, int clear) {
  g_error[0] = 0;
  const char* what = "attention_forward_varlen";
  if (int rc = check_common(what, q, k, v, out, lse, num_seqs, total_seqlen_q, total_seqlen_kv, heads_q, heads_kv,
                            head_dim))
    return rc;
  if (!cumulative_seqlen_q || !cumulative_seqlen_kv) return fail("%s: null cumulative sequence length array", what);
  if (max_seqlen_q < 1 || max_seqlen_kv < 1 || max_seqlen_q > total_seqlen_q || max_seqlen_kv > total_seqlen_kv)
    return fail("%s: maximum sequence lengths (%d, %d) must lie in 1 .. total (%d, %d)", what, max_seqlen_q,
                max_seqlen_kv, total_seqlen_q, total_seqlen_kv);
  if (dtype != NATTEN_AMD_F16 && dtype != NATTEN_AMD_BF16)
    return fail("%s: only 16-bit float operands are supported, got dtype code %d", what, dtype);
  constexpr int QT = 128, KVT = 64;
  FnaParams p;
  memset(&p, 0, sizeof(p));
  for (int a = 0; a < 3; ++a) {
    p.qkv_shape[a] = p.ksize[a] = p.stride[a] = p.dil[a] = p.q_tile[a] = p.kv_tile[a] = p.q_tiled[a] = p.kv_tiled[a] = 1;
  }
  // one batch entry per sequence; the kernel reads every sequence's own lengths (window =
  // its whole key sequence) from the cumulative arrays, the launch is sized for the longest
  p.ksize[0] = max_seqlen_kv;
  p.qkv_shape[0] = max_seqlen_kv;
  p.causal[0] = is_causal != 0;
  p.q_tile[0] = QT;
  p.kv_tile[0] = KVT;
  p.q_tiled[0] = na_ceil_div(max_seqlen_q, QT);
  p.kv_tiled[0] = na_ceil_div(max_seqlen_kv, KVT);
  p.token_rows = p.tok_stride[0] = 1;
  p.split_first = clear;
  p.num_groups = 1;
  p.q = q;
  p.k = k;
  p.v = v;
  p.o = out;
  p.lse = lse;
  p.batch = num_seqs;
  p.heads_q = heads_q;
  p.heads_kv = heads_kv;
  p.seqlen_q = max_seqlen_q;
  p.seqlen_kv = max_seqlen_kv;
  p.scale = scale;
  p.q_scale = q_scale;
  p.k_scale = k_scale;
  p.v_scale = v_scale;
  p.cu_q = cumulative_seqlen_q;
  p.cu_kv = cumulative_seqlen_kv;
  p.total_q = total_seqlen_q;
  p.total_kv = total_seqlen_kv;
  set_wg_layout(p, 1);
  return dispatch_dtype(p, dtype, head_dim, QT, KVT, static_cast<hipStream_t>(stream));
}

int natten_amd_attention_forward_varlen(const void* q, const void* k, const void* v, void* out, float* lse, int dtype,
                                        int num_seqs, int total_seqlen_q, int total_seqlen_kv, int max_seqlen_q,
                                        int max_seqlen_kv, int heads_q, int heads_kv, int head_dim,
                                        const int32_t* cumulative_seqlen_q, const int32_t* cumulative_seqlen_kv,
                                        int is_causal, float scale, const float* q_scale, const float* k_scale,
                                        const float* v_scale, void* stream) {
  return attention_forward_varlen(q, k, v, out, lse, dtype, num_seqs, total_seqlen_q, total_seqlen_kv, max_seqlen_q, max_seqlen_kv,
                                  heads_q, heads_kv, head_dim, cumulative_seqlen_q, cumulative_seqlen_kv, is_causal, scale,
                                  q_scale, k_scale, v_scale, stream, 0);
}

int natten_amd_attention_forward_varlen_all_rows(const void* q, const void* k, const void* v, void* out, float* lse, int dtype,
                                                 int num_seqs, int total_seqlen_q, int total_seqlen_kv, int max_seqlen_q,
                                                 int max_seqlen_kv, int heads_q, int heads_kv, int head_dim,
                                                 const int32_t* cumulative_seqlen_q, const int32_t* cumulative_seqlen_kv,
                                                 int is_causal, float scale, const float* q_scale, const float* k_scale,
                                                 const float* v_scale, void* stream) {
  return attention_forward_varlen(q, k, v, out, lse, dtype, num_seqs, total_seqlen_q, total_seqlen_kv, max_seqlen_q, max_seqlen_kv,
                                  heads_q, heads_kv, head_dim, cumulative_seqlen_q, cumulative_seqlen_kv, is_causal, scale,
                                  q_scale, k_scale, v_scale, stream, 1);
}

// ---- backward ---------------------------------------------------------------------------------

extern "C++" {
// A thread's second stream on a device, and the events that order it behind the caller's stream and that one behind it.
// Made on first use, given back when the thread ends; work on it is joined before the entry point that put it there returns.
// One caller's stream uses it at a time: the work of another one would wait behind the first one's, and with it that stream.
struct SideStream {
  hipStream_t stream = nullptr, user = nullptr;  // user: the stream that forked it last
  hipEvent_t fork = nullptr, join = nullptr;
  void release() {
    if (join) (void)hipEventDestroy(join);
    if (fork) (void)hipEventDestroy(fork);
    if (stream) (void)hipStreamDestroy(stream);
    stream = nullptr;
    fork = join = nullptr;
  }
};
struct SideStreams {
  static constexpr int kDevices = 16;
  SideStream of[kDevices];
  ~SideStreams() {
    for (SideStream& s : of) s.release();
  }
};
// The calling thread's side stream, `stream`'s work so far in front of it; null where there is none: a stream that is
// being captured (the graph would hold the side stream, which eager calls also use), work of another stream on it that is
// not done, or any error.
static SideStream* fork_side_stream(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  int dev = 0;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone || hipGetDevice(&dev) != hipSuccess ||
      dev < 0 || dev >= SideStreams::kDevices) {
    (void)hipGetLastError();
    return nullptr;
  }
  thread_local SideStreams streams;
  SideStream& s = streams.of[dev];
  if (!s.stream && (hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking) != hipSuccess ||
                    hipEventCreateWithFlags(&s.fork, hipEventDisableTiming) != hipSuccess ||
                    hipEventCreateWithFlags(&s.join, hipEventDisableTiming) != hipSuccess)) {
    (void)hipGetLastError();
    s.release();
    return nullptr;
  }
  if ((s.user != stream && hipStreamQuery(s.stream) != hipSuccess) || hipEventRecord(s.fork, stream) != hipSuccess ||
      hipStreamWaitEvent(s.stream, s.fork, 0) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  s.user = stream;
  return &s;
}

// The dQ launch that comes first (see FnaBwdParams::out)
template <typename T, int D>
static int launch_bwd_first(const FnaBwdParams& params, hipStream_t stream) {
  FnaBwdParams p = params;
  const long long wgs = ((long long)p.batch * p.heads_q * prod3(p.q_tiled) + kNumXcd - 1) / kNumXcd * kNumXcd;
  set_bwd_divisions(p);
  if (wgs > 0x7fffffffLL) return fail("fna_backward: problem needs more than 2^31 workgroups");
  hipLaunchKernelGGL((fna_bwd_kernel<T, D, kBwdDQ, false, true>), dim3((unsigned)wgs), dim3(256), 0, stream, p);
  return check_launch("fna_backward (dQ)");
}

template <typename T, int D, bool RAGGED, bool RAW>
static int launch_bwd(const FnaBwdParams& params, hipStream_t stream) {
  FnaBwdParams p = params;
  // grids are padded to a multiple of the 8 XCDs: each XCD takes a contiguous eighth of the tiles
  auto grid = [](long long wgs) { return (wgs + kNumXcd - 1) / kNumXcd * kNumXcd; };
  const long long wg_q = grid((long long)p.batch * p.heads_q * prod3(p.q_tiled));
  long long wg_kv = grid((long long)p.batch * p.heads_kv * prod3(p.kv_tiled));
  if constexpr (D == 128) {
    // paired role (one workgroup per CU, 32 resident per XCD): runs of about 32 key tiles, a whole
    // number of dimension-0 slabs or an even part of one, dealt round-robin to the XCDs
    const int slab = p.kv_tiled[1] * p.kv_tiled[2];
    int run;
    if (slab >= 32) {
      const int parts = (slab + 16) / 32;
      run = (slab + parts - 1) / parts;
    } else {
      int rows = (32 + slab / 2) / slab;
      if (rows > p.kv_tiled[0]) rows = p.kv_tiled[0];
      run = slab * rows;
    }
    p.kv_wg_run = run;
    const long long runs = ((long long)p.batch * p.heads_kv * prod3(p.kv_tiled) + run - 1) / run;
    wg_kv = (runs + kNumXcd - 1) / kNumXcd * kNumXcd * run;
  }
  set_bwd_divisions(p);
  if (wg_q > 0x7fffffffLL || wg_kv > 0x7fffffffLL) return fail("fna_backward: problem needs more than 2^31 workgroups");
  const int roles = p.roles ? p.roles : 3;
  if ((roles & 2) && !(roles & 4)) {
    // The key-stationary launch streams the queries as the forward kernel multiplied them: scaled
    // and rounded once, into the workspace.  It runs before the dQ launch, so that the workspace
    // may be the dq buffer.
    const long long q_rows = p.cu_q ? (long long)p.seqlen_q
                                    : p.fused ? (long long)(p.batch / p.num_groups) * p.tokens : (long long)p.batch * p.seqlen_q;
    const long long chunks = q_rows * p.heads_q * (D / 8);
    const long long blocks = (chunks + 255) / 256;
    if (blocks > 0x7fffffffLL) return fail("fna_backward: problem needs more than 2^31 workgroups");
    hipLaunchKernelGGL((scale_queries_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, stream, static_cast<const T*>(p.q),
                       static_cast<T*>(const_cast<void*>(p.qs)), (int64_t)chunks, p.scale * 1.4426950408889634f);
    if (int rc = check_launch("fna_backward (scaled queries)")) return rc;
  }
  SideStream* side = (roles & kBwdOverlap) ? fork_side_stream(stream) : nullptr;
  int rc_kv = 0, rc_q = 0;
  if (roles & 2) {
    if constexpr (D == 128) {
      // dK and dV by wave pairs (eight waves per workgroup): one wave's registers cannot hold the
      // accumulators, fragments and products of both
      hipLaunchKernelGGL((fna_bwd_kernel<T, D, kBwdPair, RAGGED, RAW>), dim3((unsigned)wg_kv), dim3(512), 0, stream, p);
    } else {
      hipLaunchKernelGGL((fna_bwd_kernel<T, D, kBwdDKV, RAGGED, RAW>), dim3((unsigned)wg_kv), dim3(256), 0, stream, p);
    }
    rc_kv = check_launch("fna_backward (dK, dV)");
  }
  if ((roles & 1) && rc_kv == 0) {
    hipLaunchKernelGGL((fna_bwd_kernel<T, D, kBwdDQ, RAGGED>), dim3((unsigned)wg_q), dim3(256), 0, side ? side->stream : stream, p);
    rc_q = check_launch("fna_backward (dQ)");
  }
  if (side && (hipEventRecord(side->join, side->stream) != hipSuccess || hipStreamWaitEvent(stream, side->join, 0) != hipSuccess)) {
    (void)hipStreamSynchronize(side->stream);  // (the caller may reuse its memory once its own stream is past this call)
    return fail("fna_backward: the dQ launch could not be joined");
  }
  return rc_kv ? rc_kv : rc_q;
}

template <typename T, int D>
static int dispatch_bwd_form(const FnaBwdParams& p, hipStream_t stream, bool ragged) {
  if (p.out != nullptr) return launch_bwd_first<T, D>(p, stream);
  if (ragged) return launch_bwd<T, D, true, false>(p, stream);  // (dense attention: prepared arrays only)
  return p.prepared ? launch_bwd<T, D, false, false>(p, stream) : launch_bwd<T, D, false, true>(p, stream);
}

template <typename T>
static int dispatch_bwd_head_dim(const FnaBwdParams& p, int head_dim, hipStream_t stream, bool ragged) {
  switch (head_dim) {
    case 32: return dispatch_bwd_form<T, 32>(p, stream, ragged);
    case 64: return dispatch_bwd_form<T, 64>(p, stream, ragged);
    case 128: return dispatch_bwd_form<T, 128>(p, stream, ragged);
  }
  return fail("fna_backward: head_dim must be 32, 64 or 128, got %d", head_dim);
}

// ragged: dense attention on sequences that end inside a tile
static int dispatch_bwd(const FnaBwdParams& p, int dtype, int head_dim, hipStream_t stream, bool ragged = false) {
  switch (dtype) {
    case NATTEN_AMD_F16: return dispatch_bwd_head_dim<_Float16>(p, head_dim, stream, ragged);
    case NATTEN_AMD_BF16: return dispatch_bwd_head_dim<__bf16>(p, head_dim, stream, ragged);
  }
  return fail("fna_backward: only 16-bit float operands are supported, got dtype code %d", dtype);
}
}  // extern "C++"

// last dimension of extent > 1 (0 for a one-token tile)
static int split_dim_of(const int* tile) {
  int s = 0;
  for (int a = 0; a < 3; ++a)
    if (tile[a] > 1) s = a;
  return s;
}

static int check_bwd_pointers(const char* what, const void* q, const void* k, const void* v, const void* d_out,
                              const float* lse, const float* delta, void* dq, void* dk, void* dv, void* q_scaled,
                              int roles) {
  if (!q || !k || !v || !d_out || !lse || !delta || !dq || !dk || !dv) return fail("%s: null pointer argument", what);
  if ((roles & 2) && !q_scaled) return fail("%s: the dk / dv launch needs the q_scaled workspace", what);
  if (q_scaled == q) return fail("%s: q_scaled must not be q itself (the dq launch reads the unscaled queries)", what);
  if (reinterpret_cast<uintptr_t>(q_scaled) & 15) return fail("%s: q_scaled must be 16-byte aligned", what);
  const uintptr_t all = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
                        reinterpret_cast<uintptr_t>(d_out) | reinterpret_cast<uintptr_t>(dq) |
                        reinterpret_cast<uintptr_t>(dk) | reinterpret_cast<uintptr_t>(dv);
  if (all & 15) return fail("%s: q, k, v, d_out, dq, dk and dv must be 16-byte aligned", what);
  return 0;
}

int natten_amd_fna_backward(const void* q, const void* k, const void* v, const void* d_out, const float* lse,
                            const float* delta, void* dq, void* dk, void* dv, void* q_scaled, int dtype, int na_dim,
                            int batch, int seqlen_q, int seqlen_kv, int heads_q, int heads_kv, int head_dim,
                            const int32_t* q_shape, const int32_t* kv_shape, const int32_t* qkv_shape,
                            const int32_t* kernel_size, const int32_t* stride, const int32_t* dilation,
                            const int32_t* is_causal, const int32_t* q_tile_shape, const int32_t* kv_tile_shape,
                            float scale, void* stream) {
  g_error[0] = 0;
  const char* what = "fna_backward";
  if (int rc = check_bwd_pointers(what, q, k, v, d_out, lse, delta, dq, dk, dv, q_scaled, 3)) return rc;
  if (int rc = check_common(what, q, k, v, dq, lse, batch, seqlen_q, seqlen_kv, heads_q, heads_kv, head_dim)) return rc;
  if (na_dim < 1 || na_dim > 3) return fail("%s: na_dim must be 1, 2 or 3, got %d", what, na_dim);
  if (!q_shape || !kv_shape || !qkv_shape || !kernel_size || !stride || !dilation || !is_causal || !q_tile_shape ||
      !kv_tile_shape)
    return fail("%s: null shape argument", what);
  FnaParams f;
  if (int rc = fill_fna_params(what, f, na_dim, q_shape, kv_shape, qkv_shape, kernel_size, stride, dilation, is_causal,
                               q_tile_shape, kv_tile_shape))
    return rc;
  if (prod3(f.q_tile) != 128 || prod3(f.kv_tile) != 128)
    return fail("%s: Q and KV tiles must hold 128 tokens each, got %d and %d", what, prod3(f.q_tile), prod3(f.kv_tile));
  FnaBwdParams p;
  memset(&p, 0, sizeof(p));
  p.q_split = split_dim_of(f.q_tile);
  p.kv_split = split_dim_of(f.kv_tile);
  if (f.q_tile[p.q_split] % 2 != 0 || f.kv_tile[p.kv_split] % 2 != 0)
    return fail("%s: the last tile extent above 1 must be even", what);
  int groups = 1;
  for (int a = 0; a < 3; ++a) {
    p.qkv_shape[a] = f.qkv_shape[a];
    p.ksize[a] = f.ksize[a];
    p.stride[a] = f.stride[a];
    p.dil[a] = f.dil[a];
    p.causal[a] = f.causal[a];
    p.q_tile[a] = f.q_tile[a];
    p.kv_tile[a] = f.kv_tile[a];
    p.q_tiled[a] = f.q_tiled[a];
    p.kv_tiled[a] = f.kv_tiled[a];
    groups *= f.dil[a];
  }
  if (batch % groups != 0) return fail("%s: batch (%d) must be a multiple of prod(dilation) (%d)", what, batch, groups);
  if (seqlen_q != prod3(p.q_tiled) * 128 || seqlen_kv != prod3(p.kv_tiled) * 128)
    return fail("%s: sequence lengths (%d, %d) do not match the padded layouts (%d, %d)", what, seqlen_q, seqlen_kv,
                prod3(p.q_tiled) * 128, prod3(p.kv_tiled) * 128);
  p.q = q;
  p.qs = q_scaled;
  p.k = k;
  p.v = v;
  p.d_out = d_out;
  p.lse = lse;
  p.delta = delta;
  p.dq = dq;
  p.dk = dk;
  p.dv = dv;
  p.batch = batch;
  p.heads_q = heads_q;
  p.heads_kv = heads_kv;
  p.seqlen_q = seqlen_q;
  p.seqlen_kv = seqlen_kv;
  p.num_groups = groups;
  p.q_extent0 = 0;
  p.scale = scale;
  return dispatch_bwd(p, dtype, head_dim, static_cast<hipStream_t>(stream));
}

// Launches of the backward on the original tensors.  out, lse_rows: those of the launch that comes first (roles = 1), else null
static int fna_backward_fused_launches(const char* what, const void* q, const void* k, const void* v, const void* out,
                                       const float* lse_rows, const void* d_out, const float* lse, const float* delta, void* dq,
                                       void* dk, void* dv, void* q_scaled, int dtype, int na_dim, int batch, int heads_q,
                                       int heads_kv, int head_dim, const int32_t* qkv_shape, const int32_t* kernel_size,
                                       const int32_t* stride, const int32_t* dilation, const int32_t* is_causal,
                                       const int32_t* q_tile_shape, const int32_t* kv_tile_shape, float scale, int roles,
                                       void* stream) {
  if (roles < 1 || roles > 15 || (roles & 3) == 0)
    return fail("%s: roles must be 1 (dq), 2 (dk and dv) or 3 (all), plus 4 for prepared arrays, plus 8 for key tiles laid out "
                "by the windows, got %d",
                what, roles);
  const bool lay_out_keys = (roles & 8) != 0;
  roles &= 7;
  if (int rc = check_bwd_pointers(what, q, k, v, d_out, lse, delta, dq, dk, dv, q_scaled, roles)) return rc;
  if (na_dim < 1 || na_dim > 3) return fail("%s: na_dim must be 1, 2 or 3, got %d", what, na_dim);
  if (!qkv_shape || !kernel_size || !stride || !dilation || !is_causal || !q_tile_shape || !kv_tile_shape)
    return fail("%s: null shape argument", what);
  // Per-group layouts, padded to whole tiles.  Extents that are not multiples of dilation x tile are
  // taken as long as every dilation group is at least one tile wide (either side's) in every
  // dimension: tiles that would reach past a group are then moved back or clamped by the kernels.
  int q_group_shape[3] = {1, 1, 1}, kv_group_shape[3] = {1, 1, 1}, edge = 0;
  long long tokens = 1;
  for (int a = 0; a < na_dim; ++a) {
    if (qkv_shape[a] < 1 || dilation[a] < 1 || q_tile_shape[a] < 1 || kv_tile_shape[a] < 1)
      return fail("%s: invalid parameter along dimension %d", what, a);
    if (qkv_shape[a] % (dilation[a] * q_tile_shape[a]) != 0 || qkv_shape[a] % (dilation[a] * kv_tile_shape[a]) != 0) edge = 1;
    if (qkv_shape[a] / dilation[a] < q_tile_shape[a] || qkv_shape[a] / dilation[a] < kv_tile_shape[a])
      return fail("%s: a dilation group of dimension %d (%d tokens / dilation %d) is narrower than a tile (%d, %d); use "
                  "the token-permuted entry point",
                  what, a, qkv_shape[a], dilation[a], q_tile_shape[a], kv_tile_shape[a]);
    const int ext = na_ceil_div(qkv_shape[a], dilation[a]);
    q_group_shape[a] = na_ceil_div(ext, q_tile_shape[a]) * q_tile_shape[a];
    kv_group_shape[a] = na_ceil_div(ext, kv_tile_shape[a]) * kv_tile_shape[a];
    tokens *= qkv_shape[a];
  }
  if (tokens > 0x7fffffffLL) return fail("%s: more than 2^31 tokens", what);
  FnaParams f;
  if (int rc = fill_fna_params(what, f, na_dim, q_group_shape, kv_group_shape, qkv_shape, kernel_size, stride, dilation,
                               is_causal, q_tile_shape, kv_tile_shape))
    return rc;
  if (!fna_tiles_are_powers_of_two(f)) return fail("%s: tile extents must be powers of two", what);
  if (int rc = check_common(what, q, k, v, dq, lse, batch, int(tokens), int(tokens), heads_q, heads_kv, head_dim)) return rc;
  // per-lane byte offsets inside a tile are 32-bit
  long long span_q = 0, span_kv = 0;
  for (int a = 0; a < 3; ++a) {
    span_q += (long long)(f.q_tile[a] - 1) * f.dil[a] * f.tok_stride[a];
    span_kv += (long long)(f.kv_tile[a] - 1) * f.dil[a] * f.tok_stride[a];
  }
  if ((span_q + 1) * heads_q * head_dim * 2 + 8192 >= 0x7fffffffLL || (span_kv + 1) * heads_kv * head_dim * 2 + 8192 >= 0x7fffffffLL)
    return fail("%s: a tile spans more than 2^31 bytes of the tensors; use the token-permuted entry point", what);
  if (prod3(f.q_tile) != 128 || prod3(f.kv_tile) != 128)
    return fail("%s: Q and KV tiles must hold 128 tokens each, got %d and %d", what, prod3(f.q_tile), prod3(f.kv_tile));
  FnaBwdParams p;
  memset(&p, 0, sizeof(p));
  p.q_split = split_dim_of(f.q_tile);
  p.kv_split = split_dim_of(f.kv_tile);
  if (f.q_tile[p.q_split] % 2 != 0 || f.kv_tile[p.kv_split] % 2 != 0)
    return fail("%s: the last tile extent above 1 must be even", what);
  int groups = 1;
  for (int a = 0; a < 3; ++a) {
    p.qkv_shape[a] = f.qkv_shape[a];
    p.ksize[a] = f.ksize[a];
    p.stride[a] = f.stride[a];
    p.dil[a] = f.dil[a];
    p.causal[a] = f.causal[a];
    p.q_tile[a] = f.q_tile[a];
    p.kv_tile[a] = f.kv_tile[a];
    p.q_tiled[a] = f.q_tiled[a];
    p.kv_tiled[a] = f.kv_tiled[a];
    if (lay_out_keys && (roles & 2)) {
      const int ext = na_ceil_div(f.qkv_shape[a], f.dil[a]), q_sub = f.q_tile[a] >> (a == p.q_split ? 1 : 0);
      p.kv_shift[a] = choose_kv_shift(ext, f.ksize[a], f.stride[a], f.causal[a] != 0, f.kv_tile[a], q_sub);
      p.kv_tiled[a] = na_ceil_div(ext + p.kv_shift[a], f.kv_tile[a]);
    }
    p.tok_stride[a] = f.tok_stride[a];
    groups *= f.dil[a];
  }
  p.q = q;
  p.qs = q_scaled;
  p.k = k;
  p.v = v;
  p.d_out = d_out;
  p.lse = lse;
  p.delta = delta;
  p.dq = dq;
  p.dk = dk;
  p.dv = dv;
  p.batch = batch * groups;
  p.heads_q = heads_q;
  p.heads_kv = heads_kv;
  p.seqlen_q = prod3(p.q_tiled) * 128;
  p.seqlen_kv = prod3(p.kv_tiled) * 128;
  p.num_groups = groups;
  p.q_extent0 = 0;
  p.scale = scale;
  p.fused = 1;
  p.edge = edge;
  p.tokens = int(tokens);
  p.roles = roles;
  p.prepared = (roles & 4) != 0;
  p.out = out;
  p.lse_rows = lse_rows;
  return dispatch_bwd(p, dtype, head_dim, static_cast<hipStream_t>(stream));
}

int natten_amd_fna_backward_fused(const void* q, const void* k, const void* v, const void* d_out, const float* lse,
                                  const float* delta, void* dq, void* dk, void* dv, void* q_scaled, int dtype, int na_dim,
                                  int batch, int heads_q, int heads_kv, int head_dim, const int32_t* qkv_shape,
                                  const int32_t* kernel_size, const int32_t* stride, const int32_t* dilation,
                                  const int32_t* is_causal, const int32_t* q_tile_shape, const int32_t* kv_tile_shape,
                                  float scale, int roles, void* stream) {
  g_error[0] = 0;
  return fna_backward_fused_launches("fna_backward_fused", q, k, v, nullptr, nullptr, d_out, lse, delta, dq, dk, dv, q_scaled, dtype,
                                     na_dim, batch, heads_q, heads_kv, head_dim, qkv_shape, kernel_size, stride, dilation, is_causal,
                                     q_tile_shape, kv_tile_shape, scale, roles, stream);
}

int natten_amd_fna_backward_from_output(const void* q, const void* k, const void* v, const void* out, const void* d_out,
                                        const float* lse, void* dq, void* dk, void* dv, void* q_scaled, float* neg_lse2,
                                        float* neg_delta, int dtype, int na_dim, int batch, int heads_q, int heads_kv,
                                        int head_dim, const int32_t* qkv_shape, const int32_t* kernel_size, const int32_t* stride,
                                        const int32_t* dilation, const int32_t* is_causal, const int32_t* q_tile_shape,
                                        const int32_t* kv_tile_shape, const int32_t* kv_role_q_tile_shape,
                                        const int32_t* kv_role_kv_tile_shape, float scale, void* stream) {
  g_error[0] = 0;
  const char* what = "fna_backward_from_output";
  if (!out || !lse || !neg_lse2 || !neg_delta || !q_scaled) return fail("%s: null pointer argument", what);
  if (reinterpret_cast<uintptr_t>(out) & 15) return fail("%s: out must be 16-byte aligned", what);
  if (q_scaled == dq) return fail("%s: q_scaled must not be dq (the dq launch comes first)", what);
  if ((kv_role_q_tile_shape == nullptr) != (kv_role_kv_tile_shape == nullptr))
    return fail("%s: the tile shapes of the dk / dv launch must be given together", what);
  if (int rc = fna_backward_fused_launches(what, q, k, v, out, lse, d_out, neg_lse2, neg_delta, dq, dk, dv, q_scaled, dtype, na_dim,
                                           batch, heads_q, heads_kv, head_dim, qkv_shape, kernel_size, stride, dilation, is_causal,
                                           q_tile_shape, kv_tile_shape, scale, 1 + 4, stream))
    return rc;
  const bool own = kv_role_q_tile_shape != nullptr;
  return fna_backward_fused_launches(what, q, k, v, nullptr, nullptr, d_out, neg_lse2, neg_delta, dq, dk, dv, q_scaled, dtype, na_dim,
                                     batch, heads_q, heads_kv, head_dim, qkv_shape, kernel_size, stride, dilation, is_causal,
                                     own ? kv_role_q_tile_shape : q_tile_shape, own ? kv_role_kv_tile_shape : kv_tile_shape, scale,
                                     2 + 4 + (own ? 8 : 0), stream);
}

namespace {
// dense attention backward as the 1-D neighborhood problem whose window is the whole key sequence
void fill_dense_bwd(FnaBwdParams& p, const void* q, const void* k, const void* v, const void* d_out, const float* neg_lse2,
                    const float* neg_delta, void* dq, void* dk, void* dv, void* q_scaled, int batch, int seqlen_q, int seqlen_kv,
                    int heads_q, int heads_kv, int is_causal, float scale, int filled) {
  memset(&p, 0, sizeof(p));
  for (int a = 0; a < 3; ++a) {
    p.qkv_shape[a] = p.ksize[a] = p.stride[a] = p.dil[a] = p.q_tile[a] = p.kv_tile[a] = p.q_tiled[a] = p.kv_tiled[a] = 1;
  }
  p.qkv_shape[0] = p.ksize[0] = seqlen_kv;
  p.q_extent0 = seqlen_q;
  p.causal[0] = is_causal != 0;
  p.q_tile[0] = p.kv_tile[0] = 128;
  p.q_tiled[0] = na_ceil_div(seqlen_q, 128);
  p.kv_tiled[0] = na_ceil_div(seqlen_kv, 128);
  p.q = q;
  p.qs = q_scaled;
  p.k = k;
  p.v = v;
  p.d_out = d_out;
  p.lse = neg_lse2;
  p.delta = neg_delta;
  p.prepared = 1;
  p.dq = dq;
  p.dk = dk;
  p.dv = dv;
  p.batch = batch;
  p.heads_q = heads_q;
  p.heads_kv = heads_kv;
  p.seqlen_q = seqlen_q;
  p.seqlen_kv = seqlen_kv;
  p.num_groups = 1;
  p.scale = scale;
  p.roles = 3 + (filled ? 4 : 0);
}
}  // namespace

int natten_amd_attention_backward(const void* q, const void* k, const void* v, const void* d_out, const float* neg_lse2,
                                  const float* neg_delta, void* dq, void* dk, void* dv, void* q_scaled, int q_scaled_filled,
                                  int dtype, int batch, int seqlen_q, int seqlen_kv, int heads_q, int heads_kv, int head_dim,
                                  int is_causal, float scale, void* stream) {
  g_error[0] = 0;
  const char* what = "attention_backward";
  if (int rc = check_bwd_pointers(what, q, k, v, d_out, neg_lse2, neg_delta, dq, dk, dv, q_scaled, 3)) return rc;
  if (int rc = check_common(what, q, k, v, dq, neg_lse2, batch, seqlen_q, seqlen_kv, heads_q, heads_kv, head_dim)) return rc;
  FnaBwdParams p;
  fill_dense_bwd(p, q, k, v, d_out, neg_lse2, neg_delta, dq, dk, dv, q_scaled, batch, seqlen_q, seqlen_kv, heads_q, heads_kv, is_causal,
                 scale, q_scaled_filled & 1);
  if ((q_scaled_filled & 2) && q_scaled != dq && head_dim == 128) p.roles |= kBwdOverlap;
  // (sequences of whole tiles need no clamping: the instances of neighborhood attention)
  return dispatch_bwd(p, dtype, head_dim, static_cast<hipStream_t>(stream), seqlen_q % 128 != 0 || seqlen_kv % 128 != 0);
}

int natten_amd_attention_backward_varlen(const void* q, const void* k, const void* v, const void* d_out,
                                         const float* neg_lse2, const float* neg_delta, void* dq, void* dk, void* dv,
                                         void* q_scaled, int q_scaled_filled, int dtype, int num_seqs, int rows_q, int rows_kv,
                                         const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_kv,
                                         const int32_t* packed_tiles, int heads_q, int heads_kv, int head_dim, int is_causal,
                                         float scale, void* stream) {
  g_error[0] = 0;
  const char* what = "attention_backward_varlen";
  if (int rc = check_bwd_pointers(what, q, k, v, d_out, neg_lse2, neg_delta, dq, dk, dv, q_scaled, 3)) return rc;
  if (int rc = check_common(what, q, k, v, dq, neg_lse2, num_seqs, rows_q, rows_kv, heads_q, heads_kv, head_dim)) return rc;
  if (!cu_seqlens_q || !cu_seqlens_kv || !packed_tiles) return fail("%s: null cumulative length or packed_tiles argument", what);
  if (reinterpret_cast<uintptr_t>(packed_tiles) & 7) return fail("%s: packed_tiles must be 8-byte aligned", what);
  if (num_seqs > (1 << 28)) return fail("%s: more than 2^28 sequences", what);
  FnaBwdParams p;
  fill_dense_bwd(p, q, k, v, d_out, neg_lse2, neg_delta, dq, dk, dv, q_scaled, 1, rows_q, rows_kv, heads_q, heads_kv, is_causal, scale,
                 q_scaled_filled & 1);
  // lengths and windows are replaced per sequence inside the kernel
  p.q_tiled[0] = rows_q / 128 + num_seqs + 3;
  p.kv_tiled[0] = rows_kv / 128 + num_seqs + 3;
  p.cu_q = cu_seqlens_q;
  p.cu_kv = cu_seqlens_kv;
  p.packed_q = reinterpret_cast<const int2*>(packed_tiles);
  p.packed_kv = p.packed_q + (num_seqs + 2);
  p.num_seqs = num_seqs;
  if ((q_scaled_filled & 2) && q_scaled != dq && head_dim == 128) p.roles |= kBwdOverlap;
  return dispatch_bwd(p, dtype, head_dim, static_cast<hipStream_t>(stream), true);
}

int natten_amd_query_range(int key_first, int key_last, int kernel_size, int stride, int extent, int num_queries,
                           int is_causal, int32_t* first_query, int32_t* last_query) {
  g_error[0] = 0;
  if (!first_query || !last_query) return fail("query_range: null pointer argument");
  if (kernel_size < 1 || stride < 1 || extent < 1 || num_queries < 1 || kernel_size > extent || stride > kernel_size ||
      key_first < 0 || key_last < key_first || key_last >= extent)
    return fail("query_range: invalid argument");
  *first_query = na_first_query_attending(key_first, kernel_size, stride, na_make_div(stride), num_queries, is_causal != 0);
  *last_query = na_last_query_attending(key_last, kernel_size, stride, na_make_div(stride), extent, num_queries, is_causal != 0);
  return 0;
}

int natten_amd_key_tile_shift(int extent, int kernel_size, int stride, int is_causal, int key_tile, int query_tile, int32_t* shift) {
  g_error[0] = 0;
  if (!shift) return fail("key_tile_shift: null pointer argument");
  if (extent < 1 || kernel_size < 1 || kernel_size > extent || stride < 1 || stride > kernel_size || key_tile < 1 || query_tile < 1)
    return fail("key_tile_shift: 1 <= stride <= kernel_size <= extent and positive tile extents expected");
  *shift = choose_kv_shift(extent, kernel_size, stride, is_causal != 0, key_tile, query_tile);
  return 0;
}

// ---- linear maps around the attention of a layer -------------------------------------------------
namespace {
// Shape, type and alignment rules of the three entry points; fills what they share.  `outer`: the tensors of y or dy
int fill_linear(const char* what, LinearParams& p, const void* const* outer, const void* x, const void* w, int dtype, int64_t m, int n,
                int k, int part) {
  memset(&p, 0, sizeof(p));
  if (dtype != NATTEN_AMD_F16 && dtype != NATTEN_AMD_BF16) return fail("%s: only 16-bit float operands are supported, got dtype code %d", what, dtype);
  if (m < 1 || m > 0x7fffffff - 128 || n < 1 || k < 1) return fail("%s: invalid sizes (%lld rows, %d and %d columns)", what, (long long)m, n, k);
  if (part < 1 || n % part != 0 || n / part > 3) return fail("%s: one to three tensors of %d columns do not make %d", what, part, n);
  if (k % 64 != 0 || part % 64 != 0) return fail("%s: columns must be multiples of 64, got %d and tensors of %d", what, k, part);
  if (n > 32768 || k > 32768 || (long long)n * k > 0x3fffffffLL) return fail("%s: more than 32768 columns or 2^30 weights", what);
  uintptr_t bits = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w);
  for (int t = 0; t < n / part; ++t) {
    if (!outer[t]) return fail("%s: null pointer argument", what);
    bits |= reinterpret_cast<uintptr_t>(outer[t]);
  }
  if (bits & 15) return fail("%s: tensors must be 16-byte aligned", what);
  p.m = int(m);
  p.n = n;
  p.k = k;
  p.part = part;
  p.slices = 1;
  p.d_part = na_make_div(part);
  return 0;
}

// Lays `rows` x `cols` of a result out in tiles of rt x ct; the workgroups that makes (a multiple of the XCD count)
long long lay_out_linear(LinearParams& p, int rows, int cols, int rt, int ct) {
  p.row_tiles = na_ceil_div(rows, rt);
  p.col_tiles = cols / ct;
  p.d_row_tiles = na_make_div(p.row_tiles);
  p.d_col_tiles = na_make_div(p.col_tiles);
  return ((long long)p.row_tiles * p.col_tiles * p.slices + kNumXcd - 1) / kNumXcd * kNumXcd;
}

// Result tiles of 128 x 128 where there are four for each compute unit and they divide the columns (`align`), else 128 x 64: forward, us,
// 128 x 128 / 128 x 64: 36864 tokens, 512 -> 1536 (3456 wide tiles) 80 / 90, 256 -> 768 (1728) 26.6 / 28.9, 256 -> 256 (576) 13.9 /
// 12.3; 12544, 256 -> 768 (588) 13.6 / 12.5.  Fewer workgroups than that leave compute units with one to wait on.
bool wide_linear_tiles(int m, int cols, int align) {
  return align % 128 == 0 && (long long)na_ceil_div(m, 128) * (cols / 128) >= 1024;
}

// Tiles of a weight gradient (128 x 128, or 64 x 64 where that does not divide the tensors) and its slices: about one
// workgroup per compute unit, of at least two steps.
int linear_weight_tile(int k, int part) { return (k % 128 == 0 && part % 128 == 0) ? 128 : 64; }
int linear_weight_slices(int64_t m, int n, int k, int part) {
  const int tile = linear_weight_tile(k, part);
  const long long tiles = (long long)(n / tile) * (k / tile);
  const long long blocks = (m + 63) / 64;
  long long slices = (256 + tiles / 2) / tiles;
  if (slices > (blocks + 1) / 2) slices = (blocks + 1) / 2;
  if (slices < 1) slices = 1;
  const long long rows = (blocks + slices - 1) / slices;
  return int((blocks + rows - 1) / rows);
}
}  // namespace

int natten_amd_linear_forward(const void* x, const void* w, const void* bias, void* y0, void* y1, void* y2, int dtype, int64_t rows,
                              int n, int k, int part, void* stream) {
  g_error[0] = 0;
  const char* what = "linear_forward";
  if (!x || !w) return fail("%s: null pointer argument", what);
  LinearParams p;
  void* const outs[3] = {y0, y1, y2};
  if (int rc = fill_linear(what, p, outs, x, w, dtype, rows, n, k, part)) return rc;
  if (reinterpret_cast<uintptr_t>(bias) & 7) return fail("%s: bias must be 8-byte aligned", what);
  p.row[0] = x;
  p.col = w;
  p.bias = bias;
  for (int t = 0; t < 3; ++t) p.out[t] = outs[t];
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool wide = wide_linear_tiles(p.m, n, part);
  const long long blocks = lay_out_linear(p, p.m, n, 128, wide ? 128 : 64);
  if (blocks > 0x7fffffffLL) return fail("%s: problem needs more than 2^31 workgroups", what);
  const dim3 grid((unsigned)blocks), threads(256);
  if (dtype == NATTEN_AMD_F16) {
    if (wide) hipLaunchKernelGGL((linear_forward_kernel<_Float16, 128, 128>), grid, threads, 0, s, p);
    else hipLaunchKernelGGL((linear_forward_kernel<_Float16, 128, 64>), grid, threads, 0, s, p);
  } else {
    if (wide) hipLaunchKernelGGL((linear_forward_kernel<__bf16, 128, 128>), grid, threads, 0, s, p);
    else hipLaunchKernelGGL((linear_forward_kernel<__bf16, 128, 64>), grid, threads, 0, s, p);
  }
  return check_launch(what);
}

int natten_amd_linear_backward_workspace(int64_t rows, int n, int k, int part, uint64_t* bytes) {
  g_error[0] = 0;
  if (!bytes) return fail("linear_backward_workspace: null pointer argument");
  if (rows < 1 || n < 64 || k < 64 || part < 64 || n % part != 0 || k % 64 != 0 || part % 64 != 0)
    return fail("linear_backward_workspace: %lld rows, %d columns in tensors of %d, and %d columns", (long long)rows, n, part, k);
  *bytes = uint64_t(linear_weight_slices(rows, n, k, part)) * uint64_t(n) * (uint64_t(k) + 1) * 4;
  return 0;
}

namespace {
extern "C++" {
template <typename T>
int launch_linear_backward(const char* what, const LinearBackwardParams& p, bool big, bool wide, void* dw, void* db, hipStream_t s) {
  const dim3 grid((unsigned)(p.weight_blocks + p.input_blocks)), threads(256);
  if (big && wide) hipLaunchKernelGGL((linear_backward_kernel<T, 128, 128>), grid, threads, 0, s, p);
  else if (big) hipLaunchKernelGGL((linear_backward_kernel<T, 128, 64>), grid, threads, 0, s, p);
  else if (wide) hipLaunchKernelGGL((linear_backward_kernel<T, 64, 128>), grid, threads, 0, s, p);
  else hipLaunchKernelGGL((linear_backward_kernel<T, 64, 64>), grid, threads, 0, s, p);
  if (int rc = check_launch(what)) return rc;
  if (dw != nullptr) {
    const int elements = p.weight.n * p.weight.k;
    hipLaunchKernelGGL((linear_reduce_kernel<T>), dim3((unsigned)((elements / 4 + p.weight.n / 4 + 255) / 256)), threads, 0, s,
                       p.weight.partial, p.weight.partial_bias, static_cast<T*>(dw), static_cast<T*>(db), elements, p.weight.n,
                       p.weight.slices);
    return check_launch(what);
  }
  return 0;
}
}  // extern "C++"
}  // namespace

int natten_amd_linear_backward(const void* dy0, const void* dy1, const void* dy2, const void* x, const void* w, void* dx, void* dw,
                               void* db, void* workspace, uint64_t workspace_bytes, int dtype, int64_t rows, int n, int k, int part,
                               void* stream) {
  g_error[0] = 0;
  const char* what = "linear_backward";
  if ((!dx && !dw) || (dx && !w) || (dw && (!x || !workspace)) || (db && !dw)) return fail("%s: null pointer argument", what);
  LinearBackwardParams p;
  memset(&p, 0, sizeof(p));
  const void* const outer[3] = {dy0, dy1, dy2};
  bool wide = false;
  if (dx) {
    if (int rc = fill_linear(what, p.input, outer, dx, w, dtype, rows, n, k, part)) return rc;
    for (int t = 0; t < 3; ++t) p.input.row[t] = outer[t];
    p.input.col = w;
    p.input.out[0] = dx;
    wide = wide_linear_tiles(p.input.m, k, k);
    const long long blocks = lay_out_linear(p.input, p.input.m, k, 128, wide ? 128 : 64);
    if (blocks > 0x3fffffffLL) return fail("%s: problem needs more than 2^30 workgroups", what);
    p.input_blocks = int(blocks);
  }
  const int tile = linear_weight_tile(k, part);
  if (dw) {
    if (int rc = fill_linear(what, p.weight, outer, x, dw, dtype, rows, n, k, part)) return rc;
    if ((reinterpret_cast<uintptr_t>(db) & 7) || (reinterpret_cast<uintptr_t>(workspace) & 15))
      return fail("%s: db must be 8-byte and the workspace 16-byte aligned", what);
    p.weight.slices = linear_weight_slices(rows, n, k, part);
    const uint64_t need = uint64_t(p.weight.slices) * uint64_t(n) * (uint64_t(k) + 1) * 4;
    if (workspace_bytes < need)
      return fail("%s: the workspace holds %llu bytes, %llu are needed", what, (unsigned long long)workspace_bytes, (unsigned long long)need);
    p.weight.slice_rows = na_ceil_div(int((rows + 63) / 64), p.weight.slices) * 64;
    for (int t = 0; t < 3; ++t) p.weight.row[t] = outer[t];
    p.weight.col = x;
    p.weight.partial = static_cast<float*>(workspace);
    p.weight.partial_bias = db ? p.weight.partial + int64_t(p.weight.slices) * n * k : nullptr;
    const long long blocks = lay_out_linear(p.weight, n, k, tile, tile);
    if (blocks > 0x3fffffffLL) return fail("%s: problem needs more than 2^30 workgroups", what);
    p.weight_blocks = int(blocks);
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == NATTEN_AMD_F16 ? launch_linear_backward<_Float16>(what, p, tile == 128, wide, dw, db, s)
                                 : launch_linear_backward<__bf16>(what, p, tile == 128, wide, dw, db, s);
}

int natten_amd_compute_delta(const void* out, const void* d_out, float* delta, int dtype, int64_t items, int head_dim,
                             void* stream) {
  g_error[0] = 0;
  if (!out || !d_out || !delta) return fail("compute_delta: null pointer argument");
  if (items < 0) return fail("compute_delta: negative item count");
  if ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(d_out)) & 15)
    return fail("compute_delta: out and d_out must be 16-byte aligned");
  if (items == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define NA_DELTA_LAUNCH(TYPE, DD)                                                                              \
  do {                                                                                                         \
    const int64_t blocks = (items * ((DD) / 8) + 255) / 256;                                                   \
    if (blocks > 0x7fffffffLL) return fail("compute_delta: too many rows");                                    \
    hipLaunchKernelGGL((delta_kernel<TYPE, DD>), dim3((unsigned)blocks), dim3(256), 0, s,                      \
                       static_cast<const TYPE*>(out), static_cast<const TYPE*>(d_out), delta, items);          \
  } while (0)
#define NA_DELTA_DTYPE(DD)                                              \
  do {                                                                  \
    if (dtype == NATTEN_AMD_F16) NA_DELTA_LAUNCH(_Float16, DD);         \
    else if (dtype == NATTEN_AMD_BF16) NA_DELTA_LAUNCH(__bf16, DD);     \
    else return fail("compute_delta: unsupported dtype code %d", dtype); \
  } while (0)
  switch (head_dim) {
    case 32: NA_DELTA_DTYPE(32); break;
    case 64: NA_DELTA_DTYPE(64); break;
    case 128: NA_DELTA_DTYPE(128); break;
    default: return fail("compute_delta: head_dim must be 32, 64 or 128, got %d", head_dim);
  }
#undef NA_DELTA_DTYPE
#undef NA_DELTA_LAUNCH
  return check_launch("compute_delta");
}

int natten_amd_backward_prepare(const void* q, const void* out, const void* d_out, const float* lse, void* q_scaled,
                                float* neg_delta, float* neg_lse2, int dtype, int batch, int tokens, int heads, int head_dim,
                                float scale, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_kv, int num_seqs,
                                int rows_kv, int32_t* packed_tiles, void* stream) {
  g_error[0] = 0;
  const char* what = "backward_prepare";
  if (!q || !out || !d_out || !lse || !q_scaled || !neg_delta || !neg_lse2) return fail("%s: null pointer argument", what);
  if (batch < 1 || tokens < 1 || heads < 1) return fail("%s: batch, tokens and heads must be positive", what);
  if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(d_out) |
       reinterpret_cast<uintptr_t>(q_scaled)) & 15)
    return fail("%s: q, out, d_out and q_scaled must be 16-byte aligned", what);
  PackedCounts packed;
  memset(&packed, 0, sizeof(packed));
  if (packed_tiles) {
    if (!cu_seqlens_q || !cu_seqlens_kv || num_seqs < 1 || num_seqs > (1 << 28) || rows_kv < 1 || batch != 1)
      return fail("%s: a packed batch needs both cumulative length arrays, its sequence and key row counts and batch 1", what);
    if (reinterpret_cast<uintptr_t>(packed_tiles) & 7) return fail("%s: packed_tiles must be 8-byte aligned", what);
    packed.cu_q = cu_seqlens_q;
    packed.cu_kv = cu_seqlens_kv;
    packed.q = reinterpret_cast<int2*>(packed_tiles);
    packed.kv = packed.q + (num_seqs + 2);
    packed.num_seqs = num_seqs;
    packed.rows_q = tokens;
    packed.rows_kv = rows_kv;
  }
  int hb_lg = 0;
  while (hb_lg < 3 && heads % (2 << hb_lg) == 0) ++hb_lg;
  const int token_blocks = (tokens + (256 >> hb_lg) - 1) / (256 >> hb_lg), head_blocks = heads >> hb_lg;
  const long long blocks = (long long)token_blocks * head_blocks * batch + (packed_tiles ? 2 : 0);
  if (blocks > 0x7fffffffLL) return fail("%s: problem needs more than 2^31 workgroups", what);
  const float c_log2 = scale * 1.4426950408889634f;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define NA_PREPARE_LAUNCH(TYPE, DD)                                                                                        \
  hipLaunchKernelGGL((bwd_prepare_kernel<TYPE, DD>), dim3((unsigned)blocks), dim3(256), 0, s, static_cast<const TYPE*>(q),                     \
                     static_cast<const TYPE*>(out), static_cast<const TYPE*>(d_out), lse, static_cast<TYPE*>(q_scaled),       \
                     neg_delta, neg_lse2, tokens, heads, hb_lg, na_make_div(head_blocks), na_make_div(token_blocks), c_log2, packed)
#define NA_PREPARE_DTYPE(DD)                                             \
  do {                                                                   \
    if (dtype == NATTEN_AMD_F16) NA_PREPARE_LAUNCH(_Float16, DD);        \
    else if (dtype == NATTEN_AMD_BF16) NA_PREPARE_LAUNCH(__bf16, DD);    \
    else return fail("%s: unsupported dtype code %d", what, dtype);      \
  } while (0)
  switch (head_dim) {
    case 32: NA_PREPARE_DTYPE(32); break;
    case 64: NA_PREPARE_DTYPE(64); break;
    case 128: NA_PREPARE_DTYPE(128); break;
    default: return fail("%s: head_dim must be 32, 64 or 128, got %d", what, head_dim);
  }
#undef NA_PREPARE_DTYPE
#undef NA_PREPARE_LAUNCH
  return check_launch(what);
}

// widen: 0 = copy the payload, NATTEN_AMD_F8E4M3 / NATTEN_AMD_F8E5M2 = 8-bit float source, bf16 destination
static int tokperm_common(const char* what, bool unpermute, int widen, const void* src, void* dst, int elem_bytes, int na_dim,
                          int batch, int heads, int head_dim, const int32_t* token_layout, const int32_t* tile_shape,
                          const int32_t* dilation, int flip, void* stream) {
  g_error[0] = 0;
  if (!src || !dst) return fail("%s: null pointer argument", what);
  if (na_dim < 1 || na_dim > 3) return fail("%s: na_dim must be 1, 2 or 3, got %d", what, na_dim);
  if (elem_bytes != 1 && elem_bytes != 2 && elem_bytes != 4 && elem_bytes != 8)
    return fail("%s: elem_bytes must be 1, 2, 4 or 8, got %d", what, elem_bytes);
  if (batch < 1 || heads < 1 || head_dim < 1) return fail("%s: batch, heads and head_dim must be positive", what);
  if (!token_layout || !tile_shape || !dilation) return fail("%s: null shape argument", what);
  TokPermParams p;
  memset(&p, 0, sizeof(p));
  p.src = static_cast<const char*>(src);
  p.dst = static_cast<char*>(dst);
  p.na_dim = na_dim;
  p.batch = batch;
  p.num_groups = 1;
  p.perm_len = 1;
  p.orig_len = 1;
  p.row_bytes = int64_t(heads) * head_dim * elem_bytes;
  int R[3] = {1, 1, 1};
  for (int a = 0; a < na_dim; ++a) {
    if (token_layout[a] < 1 || tile_shape[a] < 1 || dilation[a] < 1)
      return fail("%s: token_layout, tile_shape and dilation must be positive (dimension %d)", what, a);
    p.layout[a] = token_layout[a];
    p.tile[a] = tile_shape[a];
    p.dil[a] = dilation[a];
    R[a] = na_ceil_div(na_ceil_div(token_layout[a], tile_shape[a]), dilation[a]);
    p.num_groups *= dilation[a];
    p.perm_len *= int64_t(R[a]) * tile_shape[a];
    p.orig_len *= token_layout[a];
  }
  for (int i = 0; i < na_dim; ++i) {
    const int a = flip ? i : na_dim - 1 - i;  // slot i (fastest first) -> original dimension
    p.t_dim[i] = a;
    p.t_size[i] = p.tile[a];
    p.r_size[i] = R[a];
    p.g_size[i] = p.dil[a];
  }
  const uintptr_t align = reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst) | uintptr_t(p.row_bytes);
  if (widen) {
    if (p.row_bytes % 8 != 0 || reinterpret_cast<uintptr_t>(src) % 8 != 0 || reinterpret_cast<uintptr_t>(dst) % 16 != 0)
      return fail("%s: heads * head_dim must be a multiple of 8, src 8-byte and dst 16-byte aligned", what);
  }
  const int vec = widen ? 8 : (align % 16 == 0) ? 16 : (align % 4 == 0) ? 4 : (align % 2 == 0) ? 2 : 1;
  const int64_t total = int64_t(batch) * p.num_groups * p.perm_len * (p.row_bytes / vec);
  int64_t blocks = (total + 255) / 256;
  const int64_t cap = 256 * 64;  // grid-stride beyond this many workgroups
  if (blocks > cap) blocks = cap;
  if (blocks < 1) blocks = 1;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define NA_TOKPERM_LAUNCH(VEC)                                                                    \
  do {                                                                                            \
    if (unpermute)                                                                                \
      hipLaunchKernelGGL((tokperm_kernel<VEC, true>), dim3(unsigned(blocks)), dim3(256), 0, s, p);  \
    else                                                                                          \
      hipLaunchKernelGGL((tokperm_kernel<VEC, false>), dim3(unsigned(blocks)), dim3(256), 0, s, p); \
  } while (0)
  if (widen == NATTEN_AMD_F8E5M2) {
    hipLaunchKernelGGL((tokperm_widen_kernel<true>), dim3(unsigned(blocks)), dim3(256), 0, s, p);
    return check_launch(what);
  } else if (widen) {
    hipLaunchKernelGGL((tokperm_widen_kernel<false>), dim3(unsigned(blocks)), dim3(256), 0, s, p);
    return check_launch(what);
  }
  if (vec == 16 && p.row_bytes >= 256) {
    // a wave per token row
    const int64_t rows = int64_t(batch) * p.num_groups * p.perm_len;
    int64_t wgs = (rows + 3) / 4;
    if (wgs > 256 * 32) wgs = 256 * 32;
    if (unpermute)
      hipLaunchKernelGGL(tokperm_rows_kernel<true>, dim3(unsigned(wgs)), dim3(256), 0, s, p);
    else
      hipLaunchKernelGGL(tokperm_rows_kernel<false>, dim3(unsigned(wgs)), dim3(256), 0, s, p);
    return check_launch(what);
  }
  switch (vec) {
    case 16: NA_TOKPERM_LAUNCH(16); break;
    case 4: NA_TOKPERM_LAUNCH(4); break;
    case 2: NA_TOKPERM_LAUNCH(2); break;
    default: NA_TOKPERM_LAUNCH(1); break;
  }
#undef NA_TOKPERM_LAUNCH
  return check_launch(what);
}

int natten_amd_token_permute(const void* src, void* dst, int elem_bytes, int na_dim, int batch, int heads,
                             int head_dim, const int32_t* token_layout, const int32_t* tile_shape,
                             const int32_t* dilation, int flip_tiled_dims, void* stream) {
  return tokperm_common("token_permute", false, 0, src, dst, elem_bytes, na_dim, batch, heads, head_dim, token_layout,
                        tile_shape, dilation, flip_tiled_dims, stream);
}

int natten_amd_token_unpermute(const void* src, void* dst, int elem_bytes, int na_dim, int batch, int heads,
                               int head_dim, const int32_t* token_layout, const int32_t* tile_shape,
                               const int32_t* dilation, int flip_tiled_dims, void* stream) {
  return tokperm_common("token_unpermute", true, 0, src, dst, elem_bytes, na_dim, batch, heads, head_dim, token_layout,
                        tile_shape, dilation, flip_tiled_dims, stream);
}

int natten_amd_token_permute_widen(const void* src, void* dst, int src_dtype, int na_dim, int batch, int heads,
                                   int head_dim, const int32_t* token_layout, const int32_t* tile_shape,
                                   const int32_t* dilation, int flip_tiled_dims, void* stream) {
  if (src_dtype != NATTEN_AMD_F8E4M3 && src_dtype != NATTEN_AMD_F8E5M2) {
    g_error[0] = 0;
    return fail("token_permute_widen: src_dtype must be an 8-bit float code, got %d", src_dtype);
  }
  return tokperm_common("token_permute_widen", false, src_dtype, src, dst, 1, na_dim, batch, heads, head_dim,
                        token_layout, tile_shape, dilation, flip_tiled_dims, stream);
}

int natten_amd_merge_attentions(const void* o0, const float* lse0, const void* o1, const float* lse1, void* out,
                                float* lse_out, int dtype, int64_t rows, int head_dim, void* stream) {
  g_error[0] = 0;
  if (!o0 || !lse0 || !o1 || !lse1 || !out || !lse_out) return fail("merge_attentions: null pointer argument");
  if (rows < 1 || head_dim < 1) return fail("merge_attentions: rows and head_dim must be positive");
  if (lse_out == lse0 || lse_out == lse1) return fail("merge_attentions: lse_out must not alias an input");
  hipStream_t s = static_cast<hipStream_t>(stream);
  // eight elements per thread where head dim and alignment allow 16-byte accesses
  const uintptr_t align = reinterpret_cast<uintptr_t>(o0) | reinterpret_cast<uintptr_t>(o1) | reinterpret_cast<uintptr_t>(out);
  const bool wide = head_dim % 8 == 0 && align % (dtype == NATTEN_AMD_F32 ? 32 : 16) == 0;
  const int64_t total = rows * (wide ? head_dim / 8 : head_dim);
  int64_t blocks = (total + 255) / 256;
  if (blocks > 256 * 64) blocks = 256 * 64;
#define NA_MERGE_LAUNCH(T, VEC)                                                                                     \
  hipLaunchKernelGGL((merge_kernel<T, VEC>), dim3(unsigned(blocks)), dim3(256), 0, s, static_cast<const T*>(o0), lse0, \
                     static_cast<const T*>(o1), lse1, static_cast<T*>(out), lse_out, rows, head_dim)
  switch (dtype) {
    case NATTEN_AMD_F16:
      if (wide) NA_MERGE_LAUNCH(_Float16, 8); else NA_MERGE_LAUNCH(_Float16, 1);
      break;
    case NATTEN_AMD_BF16:
      if (wide) NA_MERGE_LAUNCH(__bf16, 8); else NA_MERGE_LAUNCH(__bf16, 1);
      break;
    case NATTEN_AMD_F32:
      if (wide) NA_MERGE_LAUNCH(float, 8); else NA_MERGE_LAUNCH(float, 1);
      break;
    default:
      return fail("merge_attentions: unsupported dtype code %d", dtype);
  }
#undef NA_MERGE_LAUNCH
  return check_launch("merge_attentions");
}

int natten_amd_merge_attention_parts(const void* parts, const float* lse_parts, int num_parts, void* out, float* lse_out,
                                     int dtype, int64_t rows, int head_dim, void* stream) {
  g_error[0] = 0;
  if (!parts || !lse_parts || !out || !lse_out) return fail("merge_attention_parts: null pointer argument");
  if (rows < 1 || head_dim < 1) return fail("merge_attention_parts: rows and head_dim must be positive");
  if (num_parts < 1 || num_parts > 64) return fail("merge_attention_parts: num_parts must be 1 .. 64, got %d", num_parts);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uintptr_t align = reinterpret_cast<uintptr_t>(parts) | reinterpret_cast<uintptr_t>(out);
  const bool wide = head_dim % 8 == 0 && align % (dtype == NATTEN_AMD_F32 ? 32 : 16) == 0;
  const int64_t total = rows * (wide ? head_dim / 8 : head_dim);
  int64_t blocks = (total + 255) / 256;
  if (blocks > 256 * 64) blocks = 256 * 64;
  const int64_t part_stride = rows * head_dim;
#define NA_MERGE_LAUNCH(T, VEC)                                                                                      \
  hipLaunchKernelGGL((merge_parts_kernel<T, VEC>), dim3(unsigned(blocks)), dim3(256), 0, s, static_cast<const T*>(parts), \
                     lse_parts, num_parts, part_stride, static_cast<T*>(out), lse_out, rows, head_dim)
  switch (dtype) {
    case NATTEN_AMD_F16:
      if (wide) NA_MERGE_LAUNCH(_Float16, 8); else NA_MERGE_LAUNCH(_Float16, 1);
      break;
    case NATTEN_AMD_BF16:
      if (wide) NA_MERGE_LAUNCH(__bf16, 8); else NA_MERGE_LAUNCH(__bf16, 1);
      break;
    case NATTEN_AMD_F32:
      if (wide) NA_MERGE_LAUNCH(float, 8); else NA_MERGE_LAUNCH(float, 1);
      break;
    default:
      return fail("merge_attention_parts: unsupported dtype code %d", dtype);
  }
#undef NA_MERGE_LAUNCH
  return check_launch("merge_attention_parts");
}

int natten_amd_mfma_probe(const void* operands, float* sink, uint64_t* clocks, int iters, int fma_per_mfma,
                          void* stream) {
  g_error[0] = 0;
  if (!operands || !sink || !clocks) return fail("mfma_probe: null pointer argument");
  if (iters < 1) return fail("mfma_probe: iters must be positive");
  hipStream_t s = static_cast<hipStream_t>(stream);
  unsigned long long* c = reinterpret_cast<unsigned long long*>(clocks);
  switch (fma_per_mfma) {
    case 0:
      hipLaunchKernelGGL(mfma_probe_kernel<0>, dim3(kProbeBlocks), dim3(kProbeThreads), 0, s, operands, sink, c, iters);
      break;
    case 4:
      hipLaunchKernelGGL(mfma_probe_kernel<4>, dim3(kProbeBlocks), dim3(kProbeThreads), 0, s, operands, sink, c, iters);
      break;
    default:
      return fail("mfma_probe: fma_per_mfma must be 0 or 4, got %d", fma_per_mfma);
  }
  return check_launch("mfma_probe");
}

}  // extern "C"

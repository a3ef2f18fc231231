// fa_internal.hpp - host-side launchers behind the C ABI (fa_api.cpp).
#pragma once

#include <algorithm>

#include <hip/hip_runtime.h>

#include "../../include/fa_mi355x.h"

namespace fa {

// Buffer-addressed tiles use 32-bit byte offsets inside a window of `rows`
// rows: the fast kernels need rows * stride * 2 < 2^31.
inline bool buf_rows_ok(int64_t stride_elems, int rows) {
  return stride_elems >= 0 && stride_elems * 2 * (int64_t)rows < (int64_t(1) << 31);
}

// Optional caller memory of a forward (fa_fwd_ws); ptr NULL: none.
struct FwdScratch {
  void* ptr;
  int64_t bytes;
};
// Workgroups that share a row block's keys (1: none), and the scratch their
// states take.
int fwd_split_count(const fa_fwd_params& p);
size_t fwd_workspace_bytes(const fa_fwd_params& p);
// Output of a split forward from its shares' states (fwd16_split_kernel).
hipError_t launch_fwd_merge(const fa_fwd_params& p, int nmb, int nsplit, const float* ws, hipStream_t stream);

// Each launcher validates nothing beyond what it needs to pick a kernel
// instantiation; fa_api.cpp has already checked the arguments.  They return
// hipSuccess, hipErrorInvalidValue for an unsupported configuration, or the
// launch error.
hipError_t launch_fwd(const fa_fwd_params& p, const FwdScratch& w, hipStream_t stream);
// phases: bit 0 delta, bit 1 dK/dV, bit 2 dQ.
hipError_t launch_bwd(const fa_bwd_params& p, int phases, hipStream_t stream);
hipError_t launch_decode(const fa_decode_params& p, hipStream_t stream);
// launch_decode with the library's static per-device scratch as workspace and
// tickets (sizes already checked against FA_NOALLOC_*).
hipError_t launch_decode_noalloc(const fa_decode_params& p, hipStream_t stream);
hipError_t launch_paged(const fa_paged_params& p, hipStream_t stream);
hipError_t launch_tiny(const fa_tiny_params& p, hipStream_t stream);
hipError_t launch_append(const fa_append_params& p, hipStream_t stream);

size_t decode_workspace_bytes(int batch, int heads_q, int seqlen_q, int head_dim, int num_splits);

// Score-gradient scratch of the 16-bit backward: per (sequence, query head)
// a region of tiles of 64 keys x 128 queries (16 KiB of 16-bit dS), tile
// (key block kb, query block qb) at kb * ds_qblocks(Sq) + qb; the regions of
// a varlen batch are packed in sequence order.  Inside a tile, queries come
// in 4 sub-tiles of 32 (4 KiB each, key-major rows of 32 queries): element
// (key n, query q) at (q / 32) * 2048 + n * 32 + q % 32.  A dK/dV step (32
// queries) then writes whole 64-byte rows, 2 KiB contiguous per wave, and a
// dQ step reads one tile's 16 contiguous KiB.  The scratch ends
// in 1 KiB of slack where lanes past the last key of a dK/dV wave write.
constexpr int kDsMaxVarlenBatch = 512;
constexpr int kDsTileKeys = 64, kDsTileQueries = 128, kDsTileElems = kDsTileKeys * kDsTileQueries;
constexpr int kDsSubQueries = 32, kDsSubElems = kDsTileKeys * kDsSubQueries;
__host__ __device__ inline int64_t ds_qblocks(int sq) { return ((int64_t)sq + kDsTileQueries - 1) / kDsTileQueries; }
__host__ __device__ inline int64_t ds_region_elems(int sq, int sk) {
  return ((int64_t)sk + kDsTileKeys - 1) / kDsTileKeys * ds_qblocks(sq) * kDsTileElems;
}
size_t bwd_ds_only_bytes(const fa_bwd_params& p);  // without the shares below
size_t bwd_ds_bytes(const fa_bwd_params& p);
// D = 256 with dS scratch: workgroups that share a key block's query steps
// (1: none); their fp32 sums follow the dS in the scratch.
int bwd_share_count(const fa_bwd_params& p);
int64_t bwd_share_offset(const fa_bwd_params& p);  // bytes from the scratch's start
// dK and dV from the shares' sums.
hipError_t launch_dkdv_merge(const fa_bwd_params& p, int nshare, hipStream_t stream);
// dS scratch for `kv_heads` KV heads (with their query heads) of p, or 0
// when the backward cannot run in KV-head chunks: the per-head modifiers
// (bias, ALiBi, dropout) are indexed by the head, so only problems without
// them are chunked.
size_t bwd_ds_chunk_bytes(const fa_bwd_params& p, int kv_heads);
// KV heads per chunk when a backward with `ws` bytes of dS scratch runs in
// chunks, or 0 when it does not (the whole dS fits, or the problem cannot
// be chunked, or chunking would not pay: it is used only for two chunks of
// at least 1 GiB of dS each).
int bwd_ds_chunk_heads(const fa_bwd_params& p, int64_t ws);
constexpr int64_t kDsMinChunkBytes = int64_t(1) << 30;

// Raise a kernel's dynamic LDS limit once per process (gfx950: 160 KiB/CU).
hipError_t allow_lds(const void* kernel, int bytes);

// Compute units of the current device (cached per device).
int device_cu_count();

// Most keys that `rows` consecutive query rows of a dense problem see.
inline int64_t visible_keys(const fa_fwd_params& p, int rows) {
  const int64_t right = p.causal ? 0 : p.window_right;
  int64_t n = p.seqlen_k;
  if (p.window_left >= 0) {
    n = std::min<int64_t>(n, (int64_t)p.seqlen_q + p.window_left);
    if (right >= 0) n = std::min<int64_t>(n, p.window_left + right + rows);
  }
  return n;
}

// Most query rows that see a key among `keys` consecutive ones.
inline int64_t visible_queries(const fa_fwd_params& p, int keys) {
  const int64_t right = p.causal ? 0 : p.window_right;
  int64_t n = p.seqlen_q;
  if (right >= 0) {
    n = std::min<int64_t>(n, p.seqlen_k + right);
    if (p.window_left >= 0) n = std::min<int64_t>(n, p.window_left + right + keys);
  }
  return n;
}

// Whether a dense problem's row blocks cost about the same: the keys that
// five rows, from the first to the last, see average at least two thirds of
// the most any of them sees (a causal mask: half).
inline bool equal_blocks(const fa_fwd_params& p) {
  const int64_t off = (int64_t)p.seqlen_k - p.seqlen_q;
  int64_t sum = 0, most = 0;
  for (int i = 0; i < 5; ++i) {
    const int64_t at = ((int64_t)p.seqlen_q - 1) * i / 4 + off;
    int64_t lo = 0, hi = p.seqlen_k;
    if (p.window_left >= 0) lo = std::max<int64_t>(lo, at - p.window_left);
    if (p.window_right >= 0) hi = std::min<int64_t>(hi, at + p.window_right + 1);
    if (p.causal) hi = std::min<int64_t>(hi, at + 1);
    const int64_t seen = std::max<int64_t>(0, hi - lo);
    sum += seen;
    most = std::max(most, seen);
  }
  return 3 * sum >= 2 * 5 * most;
}

// fp32 up to D = 128 (backward: 64): whether workgroups of 64 rows (or keys)
// whose other range is split between two halves (NH = 2) beat ones of 128
// rows, given the number of 128-row blocks.  A round of the former takes 0.56
// (backward) to 0.66 of a round of the latter, so equal blocks take them when
// the rounds come out shorter: mostly when a last round of whole blocks would
// leave half of the CUs idle (16 x 1000 x 64, 128 blocks: forward 59 against
// 95 us, step 255 against 435; 192 blocks 112 against 96, 512 blocks 224
// against 165).  At D = 32 more workgroups fit a CU: 384 blocks 83 against
// 96 us, 512 106 against 97.  Causal blocks even out better when they are
// small: D = 64, 384 blocks 106 against 118 us, 512 137 against 125 (rows of
// 1000; of 4096: 435 against 466); D = 128, 256 blocks 120 against 162 us,
// 384 190 against 165; D = 32, 768 blocks 94 against 96.
inline bool f32_halves(const fa_fwd_params& p, int64_t blocks, bool backward) {
  const int64_t cus = device_cu_count();
  const int d = p.head_dim;
  if (!equal_blocks(p)) {
    if (d == 32) return blocks <= 3 * cus;
    if (d == 64) return blocks * 2 <= (p.seqlen_q >= 2048 ? 4 : 3) * cus;
    return blocks <= cus;
  }
  if (d == 32) return blocks * 2 <= 3 * cus;
  const int half_cost = backward ? 27 : d == 64 ? 32 : 30;  // of a whole round's 48
  return (2 * blocks + cus - 1) / cus * half_cost < (blocks + cus - 1) / cus * 48;
}

}  // namespace fa

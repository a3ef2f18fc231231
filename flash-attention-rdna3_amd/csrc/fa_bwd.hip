// Dtype dispatch of the bwd kernels (instantiated in fa_bwd_{f16,bf16,f32}.hip).
#include "fa_internal.hpp"
#include "fa_bwd_roles.hpp"

namespace fa {

template <typename Tag>
hipError_t bwd_by_mods(const fa_bwd_params& p, int ph, hipStream_t s);

// Shares of the D = 256 dK/dV pass: a grid that would leave half the CUs
// idle is split until it fills them (at least eight query steps of 32 rows
// each in the block that sees the most), and a causal grid of one round at
// most in two, since it lasts as long as its heaviest block, twice the mean
// (1 x 16/8 x 2048 x 256 bf16: dK/dV 150 -> 108 us and 14 for the merge).  At 1 x 4 x 500 x 256, two shares of
// eight steps, it is 26.7 -> 21.2 + 4.3 us.
int bwd_share_count(const fa_bwd_params& p) {
  const fa_fwd_params& f = p.fwd;
  if (f.dtype == FA_DTYPE_F32 || f.head_dim != 256 || f.cu_seqlens_q) return 1;
  if (f.batch <= 0 || f.heads_q <= 0 || f.heads_kv <= 0 || f.seqlen_q <= 0 || f.seqlen_k <= 0) return 1;
  // (problems that may run in chunks of KV heads have none; the chunks' own
  // launches get scratch for their dS only)
  if (bwd_share_offset(p) >= kDsMinChunkBytes) return 1;
  const int64_t groups = ((int64_t)f.seqlen_k + 63) / 64 * f.batch * f.heads_kv;
  const int64_t steps = (visible_queries(f, 64) + 31) / 32;
  const int64_t cus = device_cu_count();
  if (groups > cus) return 1;
  if (groups * 2 > cus) return f.causal && (f.window_left < 0 || !equal_blocks(f)) && steps >= 32 ? 2 : 1;
  return (int)std::max<int64_t>(1, std::min({cus / groups, steps / 8, (int64_t)8}));
}

int64_t bwd_share_offset(const fa_bwd_params& p) {
  const fa_fwd_params& f = p.fwd;
  return (int64_t)f.batch * f.heads_q * ds_region_elems(f.seqlen_q, f.seqlen_k) * 2 + 1024;
}

template <typename Tag>
static hipError_t run_dkdv_merge(const fa_bwd_params& p, int nshare, hipStream_t s) {
  const fa_fwd_params& f = p.fwd;
  const unsigned items = (unsigned)((f.seqlen_k + 63) / 64 * f.batch * f.heads_kv);
  const float* part = reinterpret_cast<const float*>(static_cast<const char*>(p.ds_workspace) + bwd_share_offset(p));
  hipLaunchKernelGGL((dkdv_merge_kernel<Tag, 256>), dim3(items * 4), dim3(256), 0, s, p, nshare, part);
  return hipGetLastError();
}

hipError_t launch_dkdv_merge(const fa_bwd_params& p, int nshare, hipStream_t s) {
  return p.fwd.dtype == FA_DTYPE_F16 ? run_dkdv_merge<f16_t>(p, nshare, s) : run_dkdv_merge<bf16_t>(p, nshare, s);
}

size_t bwd_ds_only_bytes(const fa_bwd_params& p) {
  const fa_fwd_params& f = p.fwd;
  if (f.dtype == FA_DTYPE_F32 || f.head_dim > 256 || f.head_dim < 64) return 0;
  if (f.head_dim > 128 && f.cu_seqlens_q) return 0;
  if (f.batch <= 0 || f.heads_q <= 0 || f.seqlen_q <= 0 || f.seqlen_k <= 0) return 0;
  int64_t elems;
  if (f.cu_seqlens_q) {
    if (f.batch > kDsMaxVarlenBatch || f.total_q < 0) return 0;
    // sum_b kblocks(Sk_b) * qblocks(Sq_b)
    //   <= kblocks(max_seqlen_k) * (total_q / 128 + batch)
    const int64_t kb = ((int64_t)f.seqlen_k + kDsTileKeys - 1) / kDsTileKeys;
    elems = (int64_t)f.heads_q * kb * ((int64_t)f.total_q / kDsTileQueries + f.batch) * kDsTileElems;
  } else {
    elems = (int64_t)f.batch * f.heads_q * ds_region_elems(f.seqlen_q, f.seqlen_k);
  }
  return (size_t)elems * 2 + 1024;
}

size_t bwd_ds_bytes(const fa_bwd_params& p) {
  const fa_fwd_params& f = p.fwd;
  size_t bytes = bwd_ds_only_bytes(p);
  if (bytes == 0) return 0;
  if (const int n = bwd_share_count(p); n > 1)  // 64 keys of dK and dV in fp32 per share
    bytes += ((size_t)f.seqlen_k + 63) / 64 * f.batch * f.heads_kv * n * (2 * 64 * 256 * 4);
  return bytes;
}

size_t bwd_ds_chunk_bytes(const fa_bwd_params& p, int kv_heads) {
  const fa_fwd_params& f = p.fwd;
  if (f.bias || f.alibi_slopes || f.dropout_p > 0.f) return 0;
  if (f.heads_kv <= 0 || kv_heads <= 0 || kv_heads > f.heads_kv) return 0;
  const size_t full = bwd_ds_bytes(p);
  if (full == 0) return 0;
  // The bound is linear in the number of heads (plus the 1 KiB slack).
  return (full - 1024) / f.heads_kv * kv_heads + 1024;
}

// Two chunks of near-equal size, each with at least 1 GiB of dS: measured on
// MI355X, two such chunks run as fast as the whole scratch (B=1, H=32,
// S=16384 causal: 9.71 against 9.75 ms), while three or more, or smaller
// chunks, lose to recomputing dQ (the same step with three chunks 10.09 ms,
// recompute 10.08 ms; config 2 in two chunks of 134 MB 244 against 210 us).
int bwd_ds_chunk_heads(const fa_bwd_params& p, int64_t ws) {
  const fa_fwd_params& f = p.fwd;
  if (f.heads_kv < 2) return 0;
  const size_t full = bwd_ds_bytes(p);
  if (full == 0 || ws >= (int64_t)full) return 0;
  const int per = (f.heads_kv + 1) / 2;
  const size_t chunk = bwd_ds_chunk_bytes(p, per);
  if (chunk == 0 || (int64_t)chunk - 1024 < kDsMinChunkBytes || ws < (int64_t)chunk) return 0;
  return per;
}

hipError_t launch_bwd(const fa_bwd_params& p, int ph, hipStream_t s) {
  switch (p.fwd.dtype) {
    case FA_DTYPE_F16: return bwd_by_mods<f16_t>(p, ph, s);
    case FA_DTYPE_BF16: return bwd_by_mods<bf16_t>(p, ph, s);
    case FA_DTYPE_F32: return bwd_by_mods<f32_t>(p, ph, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace fa

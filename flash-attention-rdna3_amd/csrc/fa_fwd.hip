// Dtype dispatch of the fwd kernels (instantiated in fa_fwd_{f16,bf16,f32}.hip).
#include "fa_internal.hpp"
#include "fa_common.hpp"

namespace fa {

template <typename Tag>
hipError_t fwd_by_mods(const fa_fwd_params& p, const FwdScratch& w, hipStream_t s);

// Key splits of a forward whose row blocks leave most CUs idle (wide heads
// only: an autoencoder's single head of 4096 rows is 64 workgroups).  Each
// share keeps at least four 32-key tiles, so its state (512 KiB at most per
// 128 rows) costs less to store and merge than the keys it takes over.
int fwd_split_count(const fa_fwd_params& p) {
  if (p.dtype == FA_DTYPE_F32 || p.head_dim <= 128 || p.cu_seqlens_q) return 1;
  if (p.batch <= 0 || p.heads_q <= 0 || p.seqlen_q <= 0 || p.seqlen_k <= 0) return 1;
  const int64_t groups = ((int64_t)p.seqlen_q + 127) / 128 * p.batch * p.heads_q * (p.head_dim > 256 ? 2 : 1);
  const int64_t cus = device_cu_count();
  if (groups * 2 > cus) return 1;
  const int64_t tiles = ((int64_t)p.seqlen_k + 31) / 32;
  const int64_t n = std::min(cus / groups, tiles / 4);
  return (int)std::max<int64_t>(1, std::min<int64_t>(n, 16));
}

size_t fwd_workspace_bytes(const fa_fwd_params& p) {
  const int n = fwd_split_count(p);
  if (n < 2) return 0;
  // Per share: 128 rows of O in fp32, and their m and l for each column half.
  const size_t blocks = ((size_t)p.seqlen_q + 127) / 128 * p.batch * p.heads_q;
  return blocks * n * ((size_t)128 * p.head_dim + 256 * (p.head_dim > 256 ? 2 : 1)) * 4;
}

hipError_t launch_fwd(const fa_fwd_params& p, const FwdScratch& w, hipStream_t s) {
  switch (p.dtype) {
    case FA_DTYPE_F16: return fwd_by_mods<f16_t>(p, w, s);
    case FA_DTYPE_BF16: return fwd_by_mods<bf16_t>(p, w, s);
    case FA_DTYPE_F32: return fwd_by_mods<f32_t>(p, w, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace fa

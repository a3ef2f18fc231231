// Dtype dispatch of the fwd kernels (instantiated in fa_fwd_{f16,bf16,f32}.hip).
#include "fa_internal.hpp"
#include "fa_fwd16.hpp"

namespace fa {

template <typename Tag>
hipError_t fwd_by_mods(const fa_fwd_params& p, const FwdScratch& w, hipStream_t s);

// Key splits of a forward whose row blocks leave CUs idle (wide heads only):
// too few blocks (an autoencoder's single head of 4096 rows is 64 workgroups),
// or a causal grid of one round at most, which lasts as long as its heaviest
// block, twice the mean (1 x 16 x 2048 x 256 bf16: 115 us, in two shares 77
// and 15 for their merge).  The shares of the block that sees the most keys
// keep at least four 32-key tiles each, so that its state (130 KiB for 128
// rows of 256 columns) costs less to store and merge than the keys it takes
// over: a window of 64 on 1 x 1 x 4096 x 256 fp16 takes 16.4 us the call
// unsplit and 25.7 in eight shares.  (A causal window leaves the blocks about
// equal: 16/8 x 2048 x 256 bf16, window 300, 33.5 against 57.3 us in two.)
int fwd_split_count(const fa_fwd_params& p) {
  if (p.dtype == FA_DTYPE_F32 || p.head_dim <= 128 || p.cu_seqlens_q) return 1;
  if (p.batch <= 0 || p.heads_q <= 0 || p.seqlen_q <= 0 || p.seqlen_k <= 0) return 1;
  const int64_t groups = ((int64_t)p.seqlen_q + 127) / 128 * p.batch * p.heads_q * (p.head_dim > 256 ? 2 : 1);
  const int64_t cus = device_cu_count();
  const int64_t tiles = (visible_keys(p, 128) + 31) / 32;
  if (groups * 2 > cus) return p.causal && (p.window_left < 0 || !equal_blocks(p)) && groups <= cus && tiles >= 32 ? 2 : 1;
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

// Merge of fwd16_split_kernel's shares, 64 output columns of one row block
// per workgroup: O = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s in the
// accumulator layout the shares were parked in (1 KiB per load), then whole
// 128-byte row pieces through LDS.  (Instantiated in fa_fwd.hip: with the
// minimum-register scheduler of the other 16-bit files its loads go out one
// after another, 13.5 against 8.9 us at 1 x 1 x 4096 x 512 in four shares.)
template <typename Tag, int D>
__global__ __launch_bounds__(256) void fwd16_merge_kernel(fa_fwd_params p, int num_m_blocks, int nsplit,
                                                          const float* ws) {
  using C = Fwd16Cfg<D, 1>;
  using S = uint16_t;
  constexpr int MD = 64;  // columns per workgroup
  constexpr int PER = C::DO / MD;
  __shared__ __align__(16) uint16_t stage[C::NQ * 32 * (MD + 8)];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, l32 = lane & 31;
  const int cc = blockIdx.x % PER;
  const int item = blockIdx.x / PER;
  const int dc = item % C::NDC;
  const int bh_count = p.batch * p.heads_q;
  const int mb_rev = item / C::NDC / bh_count;
  const int bh = item / C::NDC - mb_rev * bh_count;
  const int b = bh / p.heads_q, hq = bh - b * p.heads_q;
  const int m0w = (num_m_blocks - 1 - mb_rev) * C::BM + 32 * wave;
  const int mrows = min(32, p.seqlen_q - m0w);
  const float* src = ws + (int64_t)item * nsplit * C::PART;
  float M = kNegInf;
  for (int s = 0; s < nsplit; ++s) M = fmaxf(M, src[(int64_t)s * C::PART + C::PART_O + 32 * wave + l32]);
  const float Mu = (M == kNegInf) ? 0.f : M;
  float L = 0.f;
  f32x16 acc[MD / 32];
#pragma unroll
  for (int i = 0; i < MD / 32; ++i) acc[i] = zero16();
  for (int s = 0; s < nsplit; ++s) {
    const float* ps = src + (int64_t)s * C::PART;
    const float w = __builtin_amdgcn_exp2f(ps[C::PART_O + 32 * wave + l32] - Mu);
    L += ps[C::PART_O + C::BM + 32 * wave + l32] * w;
#pragma unroll
    for (int i = 0; i < MD / 32; ++i) {
      const f32x16 o = unpark_acc(ps + (wave * C::NDB + cc * (MD / 32) + i) * 1024, lane);
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][e] += o[e] * w;
    }
  }
  const float l_safe = (L == 0.f) ? 1.f : L;
  S* orow0 = reinterpret_cast<S*>(p.out) + b * p.out_stride[0] + hq * p.out_stride[1] +
             (int64_t)m0w * p.out_stride[2] + dc * C::DO + cc * MD;
  store_rows_staged<Tag, MD>(acc, 1.f / l_safe, stage + wave * 32 * (MD + 8), orow0, p.out_stride[2], mrows, lane);
  if (l32 < mrows && h == 0 && dc == 0 && cc == 0)
    p.lse[b * p.lse_stride[0] + hq * p.lse_stride[1] + (int64_t)(m0w + l32) * p.lse_stride[2]] =
        (M == kNegInf || L == 0.f) ? kNegInf : (M + __log2f(l_safe)) * kLn2;
}

template <typename Tag, int D>
static hipError_t run_merge(const fa_fwd_params& p, int nmb, int nsplit, const float* ws, hipStream_t s) {
  using C = Fwd16Cfg<D, 1>;
  const unsigned items = (unsigned)(nmb * p.batch * p.heads_q * C::NDC);
  hipLaunchKernelGGL((fwd16_merge_kernel<Tag, D>), dim3(items * (C::DO / 64)), dim3(256), 0, s, p, nmb, nsplit, ws);
  return hipGetLastError();
}

hipError_t launch_fwd_merge(const fa_fwd_params& p, int nmb, int nsplit, const float* ws, hipStream_t s) {
  const bool f16 = p.dtype == FA_DTYPE_F16;
  if (p.head_dim == 256)
    return f16 ? run_merge<f16_t, 256>(p, nmb, nsplit, ws, s) : run_merge<bf16_t, 256>(p, nmb, nsplit, ws, s);
  return f16 ? run_merge<f16_t, 512>(p, nmb, nsplit, ws, s) : run_merge<bf16_t, 512>(p, nmb, nsplit, ws, s);
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

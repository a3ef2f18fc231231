#pragma once
// Kernel templates of fa_fwd; instantiated per dtype by fa_fwd_<dtype>.hip.
// fa_fwd.hip - FlashAttention-2 forward (dense and packed varlen) for gfx950.
//
// Follows the algorithm of the reference's `_attention_forward` /
// `_attention_forward_varlen` (fa_rdna3/kernels/forward.py:28-164,
// varlen.py:41-149, inner loop _common.py:233-345): exp2 online softmax over
// key tiles, output normalised by the row sum, LSE = m*ln2 + ln(l).
//
// MI355X layout.  A workgroup is 4 waves; each wave owns 32 query rows, so a
// workgroup covers BM = 128 rows of one (batch, head).  Scores are computed
// TRANSPOSED, S^T = K Q^T (keys x queries), with v_mfma_f32_32x32x16: the
// query then lives on the lane (column) axis, so the row max / row sum of the
// softmax are a per-lane reduction over registers plus a single swap with the
// lane 32 apart, and the rescale of O^T = V^T P^T is a per-lane scalar.  Q^T is
// the B operand and stays in registers for the whole kernel; K (row-major) and
// V^T (transposed on the way into LDS) are double-buffered in LDS and shared
// by the 4 waves; P^T goes from the accumulator straight back into the B
// operand of the P.V MFMA without touching LDS.
//
// Work order: the m-block index is the slowest-varying grid coordinate and is
// walked from the last block down, so under causal masking the longest
// workgroups are dispatched first.
#include <type_traits>

#include "fa_internal.hpp"
#include "fa_tiles.hpp"
#include "fa_fwd16.hpp"

namespace fa {


template <typename Tag, int D, int NH>
struct FwdCfg {
  using EL = Elem<Tag>;
  using S = typename EL::S;
  // NH = 2, fp32 up to D = 128: 64 query rows (two waves) and their key tiles
  // split by parity between two halves of two waves, merged through LDS.  A wave is
  // MFMA-bound (64 cycles for 32x32x2), so what counts is that there are
  // enough of them: 1 x 16 x 1000 rows in blocks of 128 left half the CUs
  // idle.  At D = 64 the forward takes 61 us there against 100 us, dK/dV 119
  // against 203, dQ 86 against 135 (the operands of four MFMAs in one LDS
  // read, kslot, included); 4.1 / 8.2 / 6.1 GFLOP, card 153 TFLOP/s in fp32.
  // f32_halves says which grids take it.
  static constexpr int NWR = 4 / NH;          // row waves per half
  static constexpr int NW = NWR * NH;
  static constexpr int NT = 64 * NW;
  static constexpr int NTH = 64 * NWR;        // threads per half
  static constexpr int BM = 32 * NWR;
  static constexpr int BN = (D <= 128 && !(NH == 2 && D == 128)) ? 64 : 32;
  // Output columns per workgroup: D > 128 splits O^T over the grid (each
  // split recomputes the scores) to bound the accumulator registers.
  static constexpr int DO = (D <= 128) ? D : ((sizeof(S) == 4 && D == 512) ? 64 : 128);
  static constexpr bool QREG = (sizeof(S) == 2) ? (D <= 256) : (D <= 128);
  static constexpr int KLD = D + EL::CE;   // K tile row stride (elements)
  static constexpr int VLD = BN + EL::CE;  // V^T tile row stride
  static constexpr int KTILE = BN * KLD;
  static constexpr int VTILE = DO * VLD;
  static constexpr int STAGE = KTILE + VTILE;
  static constexpr int LOOP_BYTES = 2 * STAGE * (int)sizeof(S) * NH;
  static constexpr int MERGE_BYTES = NH == 1 ? 0 : NWR * (DO / 32) * 4096 + 2 * NWR * 64 * 4;
  static constexpr int LDS_BYTES = LOOP_BYTES > MERGE_BYTES ? LOOP_BYTES : MERGE_BYTES;
  static constexpr int NSTEP = D / EL::KSTEP;   // MFMA k-steps over D
  static constexpr int NKB = BN / 32;           // 32-key accumulator blocks
  static constexpr int NPV = BN / (2 * EL::E);  // P.V MFMAs per d-block
  static constexpr int NDB = DO / 32;           // 32-wide output blocks
};

template <typename Tag, int D, int MODE, int NH>
__global__ __launch_bounds__(256) void fwd_kernel(fa_fwd_params p, int num_m_blocks) {
  using C = FwdCfg<Tag, D, NH>;
  using EL = Elem<Tag>;
  using S = typename EL::S;
  using Op = typename EL::Op;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  S* smem = reinterpret_cast<S*>(smem_raw);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform (SGPR)
  const int khalf = NH == 1 ? 0 : wave_all / C::NWR, wave = wave_all % C::NWR;
  const int htid = NH == 1 ? tid : tid % C::NTH;
  const int h = lane >> 5, l32 = lane & 31;

  const int ndc = D / C::DO;
  const int bh_count = p.batch * p.heads_q;
  const int id = blockIdx.x;
  const int mb_rev = id / (bh_count * ndc);
  const int rest = id - mb_rev * bh_count * ndc;
  const int bh = rest / ndc, dc = rest - (rest / ndc) * ndc;
  const int b = bh / p.heads_q, hq = bh - b * p.heads_q;
  const int hk = hq / (p.heads_q / p.heads_kv);
  const int mblk = num_m_blocks - 1 - mb_rev;

  int q_start = 0, sq = p.seqlen_q, k_start = 0, sk = p.seqlen_k;
  if (p.cu_seqlens_q) {
    bounded_seq(p.cu_seqlens_q, b, p.total_q, q_start, sq);
    bounded_seq(p.cu_seqlens_k, b, p.total_k, k_start, sk);
  }
  const int m0 = mblk * C::BM;
  if (m0 >= sq) return;  // uniform: past the end of a short varlen sequence

  const S* qb = reinterpret_cast<const S*>(p.q) + b * p.q_stride[0] + hq * p.q_stride[1] +
                (int64_t)q_start * p.q_stride[2];
  const S* kb = reinterpret_cast<const S*>(p.k) + b * p.k_stride[0] + hk * p.k_stride[1] +
                (int64_t)k_start * p.k_stride[2];
  const S* vb = reinterpret_cast<const S*>(p.v) + b * p.v_stride[0] + hk * p.v_stride[1] +
                (int64_t)k_start * p.v_stride[2] + dc * C::DO;
  S* ob = reinterpret_cast<S*>(p.out) + b * p.out_stride[0] + hq * p.out_stride[1] +
          (int64_t)q_start * p.out_stride[2];
  float* lb = p.lse + b * p.lse_stride[0] + hq * p.lse_stride[1] + (int64_t)q_start * p.lse_stride[2];
  const int64_t qs = p.q_stride[2], ks = p.k_stride[2], vs = p.v_stride[2];

  const Mods md = make_mods(p, b, hq, sq, sk);

  // Key range of the workgroup (reference forward.py:92-127, tightened to the
  // rows that exist).
  const int mlast = min(m0 + C::BM, sq) - 1;
  int lo = 0, hi = sk;
  if (p.causal) hi = min(hi, mlast + md.off + 1);
  if (p.window_right >= 0) hi = min(hi, mlast + md.off + p.window_right + 1);
  if (p.window_left >= 0) lo = max(0, m0 + md.off - p.window_left);
  lo = lo / C::BN * C::BN;
  const int ntiles = hi > lo ? (hi - lo + C::BN - 1) / C::BN : 0;

  // This wave's query rows.
  const int m0w = m0 + 32 * wave;
  const int mrows = min(32, sq - m0w);  // <= 0: the wave only helps load
  const int m = m0w + l32;
  const bool mvalid = m < sq;

  Op qop[C::QREG ? C::NSTEP : 1];
  const S* qrow = qb + (int64_t)(mvalid ? m : 0) * qs + khalf_slot<Tag>(h);
  if constexpr (C::QREG) {
#pragma unroll
    for (int s = 0; s < C::NSTEP; ++s)
      qop[s] = mvalid ? load_op<Tag>(qrow + kslot<Tag>(s)) : zero_op<Tag>();
    wait_vm_all();
  }

  float m_i = kNegInf, l_i = 0.f;
  f32x16 acc[C::NDB];
#pragma unroll
  for (int i = 0; i < C::NDB; ++i) acc[i] = zero16();

  RowTile<Tag, C::BN, D, C::NTH> kt;
  TransTile<Tag, C::BN, C::DO, C::NTH> vt;

  auto load_tiles = [&](int n0) {
    kt.load([&](int r) -> const S* { int n = n0 + r; return n < sk ? kb + (int64_t)n * ks : nullptr; }, kb, htid);
    vt.load([&](int r) -> const S* { int n = n0 + r; return n < sk ? vb + (int64_t)n * vs : nullptr; }, vb, htid);
  };
  auto store_tiles = [&](int stage) {
    S* base = smem + (2 * khalf + stage) * C::STAGE;
    kt.store(base, C::KLD, htid);
    vt.store(base + C::KTILE, C::VLD, htid);
  };

  // Half 0 takes the even key tiles, half 1 the odd ones; both run nh0 steps.
  const int nh0 = (ntiles + NH - 1) / NH;
  const int my_count = (ntiles - khalf + NH - 1) / NH;
  if (my_count > 0) {
    load_tiles(lo + khalf * C::BN);
    store_tiles(0);
  }
  __syncthreads();

  for (int t = 0; t < nh0; ++t) {
    const int n0 = lo + (khalf + NH * t) * C::BN;
    const int stage = t & 1;
    if (t + 1 < my_count) load_tiles(n0 + NH * C::BN);

    const int vis = mrows > 0 && t < my_count ? rect_visibility(md, m0w, mrows, n0, C::BN) : 0;
    if (vis) {
      const S* Ks = smem + (2 * khalf + stage) * C::STAGE;
      const S* Vs = Ks + C::KTILE;
      f32x16 sacc[C::NKB];
#pragma unroll
      for (int kb2 = 0; kb2 < C::NKB; ++kb2) {
        sacc[kb2] = zero16();
        const S* krow = Ks + (kb2 * 32 + l32) * C::KLD + khalf_slot<Tag>(h);
#pragma unroll
        for (int s = 0; s < C::NSTEP; ++s) {
          Op a = load_op<Tag>(krow + kslot<Tag>(s));
          Op bq;
          if constexpr (C::QREG) bq = qop[s];
          else bq = mvalid ? load_op<Tag>(qrow + kslot<Tag>(s)) : zero_op<Tag>();
          sacc[kb2] = EL::mma(a, bq, sacc[kb2]);
        }
      }
      // Scores in the log2 domain, masked, and the tile max per query.
      float tmax = kNegInf;
#pragma unroll
      for (int kb2 = 0; kb2 < C::NKB; ++kb2) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int n = n0 + kb2 * 32 + acc_row(i, h);
          float tc;
          float x = score<(MODE >= 1)>(md, sacc[kb2][i], m, n, tc);
          if (vis == 1 && !keep_pos(md, m, n)) x = kNegInf;
          sacc[kb2][i] = x;
          tmax = fmaxf(tmax, x);
        }
      }
      tmax = half_max(tmax);
      const float m_new = fmaxf(m_i, tmax);
      const float m_use = (m_new == kNegInf) ? 0.f : m_new;  // safe softmax
      const float alpha = exp2f(m_i - m_use);
      float rsum = 0.f;
#pragma unroll
      for (int kb2 = 0; kb2 < C::NKB; ++kb2) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float pv = exp2f(sacc[kb2][i] - m_use);
          sacc[kb2][i] = pv;
          rsum += pv;
        }
      }
      rsum = half_sum(rsum);
      l_i = l_i * alpha + rsum;
      m_i = m_new;
#pragma unroll
      for (int db = 0; db < C::NDB; ++db) acc[db] *= alpha;
      if constexpr (MODE == 2) {
        if (md.drop_p > 0.f) {
#pragma unroll
          for (int kb2 = 0; kb2 < C::NKB; ++kb2)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const int n = n0 + kb2 * 32 + acc_row(i, h);
              sacc[kb2][i] = dropout_keep(md, m, n) ? sacc[kb2][i] * md.drop_scale : 0.f;
            }
        }
      }
      // O^T += V^T P^T.  bf16 keeps only 8 mantissa bits, so P is fed as
      // hi + lo bf16 parts (two MFMAs on the same V^T operand); the product
      // then carries P to ~2^-17 and the output error is dominated by the
      // final rounding of O.
      constexpr bool PSPLIT = std::is_same<Tag, bf16_t>::value;
      Op pb[C::NPV], pl[PSPLIT ? C::NPV : 1];
      constexpr int J = 16 / EL::E;  // MFMAs per 32-key accumulator block
#pragma unroll
      for (int j = 0; j < C::NPV; ++j) pb[j] = pack_op<Tag>(sacc[j / J], j % J);
      if constexpr (PSPLIT) {
#pragma unroll
        for (int kb2 = 0; kb2 < C::NKB; ++kb2)
#pragma unroll
          for (int i = 0; i < 16; ++i) sacc[kb2][i] -= EL::to_f(EL::from_f(sacc[kb2][i]));
#pragma unroll
        for (int j = 0; j < C::NPV; ++j) pl[j] = pack_op<Tag>(sacc[j / J], j % J);
      }
#pragma unroll
      for (int db = 0; db < C::NDB; ++db) {
        const S* vrow = Vs + (db * 32 + l32) * C::VLD;
#pragma unroll
        for (int j = 0; j < C::NPV; ++j) {
          const Op a = lds_op_rowmap<Tag>(vrow, j, h);
          acc[db] = EL::mma(a, pb[j], acc[db]);
          if constexpr (PSPLIT) acc[db] = EL::mma(a, pl[j], acc[db]);
        }
      }
    }

    if (t + 1 < my_count) store_tiles(stage ^ 1);
    __syncthreads();
  }

  // Half 1 parks (O^T, m, l) in LDS, half 0 folds them in (as fwd16_item).
  if constexpr (NH == 2) {
    float* ow = reinterpret_cast<float*>(smem_raw);
    float* mw = ow + C::NWR * C::NDB * 1024;
    float* lw = mw + C::NWR * 64;
    if (khalf == 1) {
#pragma unroll
      for (int db = 0; db < C::NDB; ++db) park_acc(ow + (wave * C::NDB + db) * 1024, lane, acc[db]);
      mw[wave * 64 + lane] = m_i;
      lw[wave * 64 + lane] = l_i;
    }
    __syncthreads();
    if (khalf == 1) return;
    const float m2 = mw[wave * 64 + lane], l2 = lw[wave * 64 + lane];
    const float mn = fmaxf(m_i, m2);
    const float mu = (mn == kNegInf) ? 0.f : mn;
    const float sa = exp2f(m_i - mu), sb = exp2f(m2 - mu);
#pragma unroll
    for (int db = 0; db < C::NDB; ++db) {
      const f32x16 o2 = unpark_acc(ow + (wave * C::NDB + db) * 1024, lane);
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[db][i] = acc[db][i] * sa + o2[i] * sb;
    }
    l_i = l_i * sa + l2 * sb;
    m_i = mn;
  }

  if (!mvalid) return;
  const float l_safe = (l_i == 0.f) ? 1.f : l_i;
  const float inv = 1.f / l_safe;
  S* orow = ob + (int64_t)m * p.out_stride[2] + dc * C::DO;
#pragma unroll
  for (int db = 0; db < C::NDB; ++db) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = db * 32 + 8 * g + 4 * h;
      if constexpr (sizeof(S) == 2) {
        s16x4 w;
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = (short)EL::from_f(acc[db][4 * g + r] * inv);
        *reinterpret_cast<s16x4*>(orow + d) = w;
      } else {
        f32x4 w;
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = acc[db][4 * g + r] * inv;
        *reinterpret_cast<f32x4*>(orow + d) = w;
      }
    }
  }
  if (h == 0 && dc == 0)
    lb[(int64_t)m * p.lse_stride[2]] = (m_i == kNegInf) ? kNegInf : (m_i + __log2f(l_safe)) * kLn2;
}

template <typename Tag, int D, int MODE, int NH, bool PAIR = false, bool FOLLOW = false>
static hipError_t launch_fwd16(const fa_fwd_params& p, long grid, int nmb, hipStream_t stream, bool exact) {
  using C = Fwd16Cfg<D, NH>;
  auto kern = fwd16_kernel<Tag, D, MODE, NH, PAIR, FOLLOW>;
  hipError_t e = allow_lds((const void*)kern, C::LDS_BYTES);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(C::NT), C::LDS_BYTES, stream, p, nmb, exact ? 1 : 0);
  return hipGetLastError();
}

template <typename Tag, int D, int MODE>
static hipError_t launch_fwd16_split(const fa_fwd_params& p, int nmb, int nsplit, float* ws, hipStream_t stream) {
  using C = Fwd16Cfg<D, 1>;
  auto kern = fwd16_split_kernel<Tag, D, MODE>;
  hipError_t e = allow_lds((const void*)kern, C::LDS_BYTES);
  if (e != hipSuccess) return e;
  const unsigned items = (unsigned)(nmb * p.batch * p.heads_q * C::NDC);
  hipLaunchKernelGGL(kern, dim3(items * nsplit), dim3(C::NT), C::LDS_BYTES, stream, p, nmb, nsplit, ws);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_fwd_merge(p, nmb, nsplit, ws, stream);
}

template <typename Tag, int D, int MODE, int NH>
static hipError_t launch_fwd_generic(const fa_fwd_params& p, hipStream_t stream) {
  using C = FwdCfg<Tag, D, NH>;
  auto kern = fwd_kernel<Tag, D, MODE, NH>;
  hipError_t e = allow_lds((const void*)kern, C::LDS_BYTES);
  if (e != hipSuccess) return e;
  const int nmb = (p.seqlen_q + C::BM - 1) / C::BM;
  const long grid = (long)nmb * p.batch * p.heads_q * (D / C::DO);
  if (grid <= 0) return hipSuccess;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(C::NT), C::LDS_BYTES, stream, p, nmb);
  return hipGetLastError();
}

template <typename Tag, int D, int MODE>
static hipError_t run_fwd(const fa_fwd_params& p, const FwdScratch& scratch, hipStream_t stream) {
  if constexpr (!std::is_same<Tag, f32_t>::value && D > 128) {
    // Wide heads: up to 512 registers a wave (O^T of 32 rows takes 128 of
    // them, Q 64 to 128), one key half.  Measured against fwd_kernel (O^T
    // split two to four ways over the grid, scores recomputed for each):
    // D = 256 bf16 causal, 1 x 16 x 2048 (34 GFLOP): 207 -> 115 us;
    // D = 512 fp16, 1 x 1 x 4096 (34 GFLOP), with key splits: 787 -> 92 us
    // (shares 79, merge 13; 52 GFLOP with the scores of both column halves).
    using C = Fwd16Cfg<D, 1>;
    if (buf_rows_ok(p.k_stride[2], C::BN) && buf_rows_ok(p.v_stride[2], C::BN)) {
      const int nmb = (p.seqlen_q + C::BM - 1) / C::BM;
      const long grid = (long)nmb * p.batch * p.heads_q * C::NDC;
      const int nsplit = fwd_split_count(p);
      if (nsplit > 1 && scratch.ptr && scratch.bytes >= (int64_t)fwd_workspace_bytes(p))
        return launch_fwd16_split<Tag, D, MODE>(p, nmb, nsplit, static_cast<float*>(scratch.ptr), stream);
      return launch_fwd16<Tag, D, MODE, 1>(p, grid, nmb, stream, true);
    }
  }
  if constexpr (!std::is_same<Tag, f32_t>::value && D <= 128) {
    using C = Fwd16Cfg<D>;
    if (buf_rows_ok(p.k_stride[2], C::BN) && buf_rows_ok(p.v_stride[2], C::BN)) {
    const int nmb = (p.seqlen_q + C::BM - 1) / C::BM;
    const long grid = (long)nmb * p.batch * p.heads_q;
    if (grid <= 0) return hipSuccess;
    // One key half, independent 4-wave workgroups, for packed varlen batches,
    // for blocks of equal cost once there are more of them than CUs, and for
    // other grids (causal, a window on one side) of more than four rounds of
    // one 8-wave workgroup per CU (a window at D = 64: two).  Equal blocks gain nothing from the key
    // split, and 640 of them in pairs took two rounds of 256 CUs:
    // 2 x 10 x 4096 x 64 fp16 190 -> 140 us, 2 x 10 x 4096 x 154 with a key
    // mask 41 -> 20 us.  At D = 32 two 8-wave workgroups fit a CU, so equal
    // blocks keep the key split up to two per CU (300 blocks, 4096 keys:
    // 59 against 71 us).  Causal 1 x 32/8 x 8000 x 128 bf16: 729 -> 711 us the
    // call; two rounds (config 2) keep the key split, 61.0 against 59.2 us.
    // A left window of 300 on 4096 x 4096, key split and one half: 10 heads of
    // 64 bf16 80 and 94 us, 20 heads 123 and 122, 20 heads of 128 172 and 181.
    // (Varlen always: a sequence's output then does not depend on the batch
    // it is packed with.  The two forms sum the key tiles in different
    // orders, so they agree to rounding, not bit for bit.)
    const long cus = device_cu_count();
    const bool one_sided = (p.window_left >= 0) != (p.window_right >= 0);
    const bool uneven = p.causal || (one_sided && !equal_blocks(p));
    const long split_rounds = p.causal ? 4 : uneven ? (D == 64 ? 2 : 4) : D == 32 ? 2 : 1;
    if (p.cu_seqlens_q || grid > split_rounds * cus) {
      // fp16 dense: as close as the key split's output up to the eight rounds
      // where the key split is the alternative (fwd16_item); FOLLOW for few
      // visible keys, or where a bias may hide all but a few (otherwise it
      // costs up to 3 %).  Exact max against lazy: 5 % (96 x 4096 x 4096 x 64
      // 522 against 497 us).
      const bool exact = !p.cu_seqlens_q && grid <= 8 * cus;
      if constexpr (std::is_same<Tag, f16_t>::value)
        if (exact && (p.bias || visible_keys(p, C::BM) <= 512))
          return launch_fwd16<Tag, D, MODE, 1, false, true>(p, grid, nmb, stream, exact);
      return launch_fwd16<Tag, D, MODE, 1>(p, grid, nmb, stream, exact);
    }
    // Heavy and light row blocks of a head paired in one workgroup, when the
    // pairs fill whole rounds of the CUs (config 2: 256 pairs): forward
    // 52.5 -> 51.4 us, same results bit for bit.
    const long pairs = (long)((nmb + 1) / 2) * p.batch * p.heads_q;
    if (p.causal && pairs >= cus && (cus - pairs % cus) % cus * 8 <= pairs)
      return launch_fwd16<Tag, D, MODE, 2, true>(p, pairs, nmb, stream, false);
    return launch_fwd16<Tag, D, MODE, 2>(p, grid, nmb, stream, !p.causal && grid > cus);
    }
  }
  // The generic kernel has no softcap-only variant (MODE 3 is MODE 1 there).
  constexpr int GMODE = MODE == 3 ? 1 : MODE;
  if constexpr (std::is_same<Tag, f32_t>::value && D <= 128) {
    const int64_t blocks = ((int64_t)p.seqlen_q + 127) / 128 * p.batch * p.heads_q;
    if (f32_halves(p, blocks, false)) return launch_fwd_generic<Tag, D, GMODE, 2>(p, stream);
  }
  return launch_fwd_generic<Tag, D, GMODE, 1>(p, stream);
}

template <typename Tag, int MODE>
static hipError_t fwd_by_dim(const fa_fwd_params& p, const FwdScratch& w, hipStream_t s) {
  switch (p.head_dim) {
    case 32: return run_fwd<Tag, 32, MODE>(p, w, s);
    case 64: return run_fwd<Tag, 64, MODE>(p, w, s);
    case 128: return run_fwd<Tag, 128, MODE>(p, w, s);
    case 256: return run_fwd<Tag, 256, MODE>(p, w, s);
    case 512: return run_fwd<Tag, 512, MODE>(p, w, s);
  }
  return hipErrorInvalidValue;
}

template <typename Tag>
hipError_t fwd_by_mods(const fa_fwd_params& p, const FwdScratch& w, hipStream_t s) {
  // 0: plain, 1: softcap / bias / ALiBi, 2: also dropout (Philox per score),
  // 3: softcap without bias or ALiBi (16-bit kernels; one score variant).
  if (p.dropout_p > 0.f) return fwd_by_dim<Tag, 2>(p, w, s);
  if constexpr (!std::is_same<Tag, f32_t>::value)
    if (p.softcap > 0.f && !p.bias && !p.alibi_slopes) return fwd_by_dim<Tag, 3>(p, w, s);
  if (p.softcap > 0.f || p.bias || p.alibi_slopes) return fwd_by_dim<Tag, 1>(p, w, s);
  return fwd_by_dim<Tag, 0>(p, w, s);
}

}  // namespace fa

// fa_bwd_roles.hpp - dK/dV for 16-bit inputs with the two products of a key
// block on two waves.
//
// Same math as dkdv16_kernel (fa_bwd16.hpp; reference
// kernels/backward.py:49-200, _common.py:347-434).  A pair of waves owns a
// key group and walks the same query steps:
//  * the V wave keeps the group's K operands in registers, computes
//    S = Q K^T and P, and accumulates dV += P^T dO;
//  * the K wave keeps the V operands, computes dP = dO V^T, takes P from the
//    V wave through LDS (fp32), forms dS = P (dP - delta) and accumulates
//    dK += dS^T Q; it also stores dS for the dQ pass.
// Each wave holds one accumulator set instead of two and one resident
// operand set in registers, so every MFMA reads at most one operand from LDS
// where dkdv16_kernel's score products read two.  That makes D = 256 fit two
// waves per SIMD (a wave holding dK and dV of 32 keys would need 256 registers
// for them alone).  LDS reads and the two barriers per step bound it.  The
// registers are full, so whatever lives across the step loop is kept small
// (row_op / tr_op / DmaLeanTile addresses, LDS reads two MFMAs ahead, dS
// stores by buffer window): a reload from scratch inside the loop waits for
// the next stage's loads too.  The plain form has none there; softcap, the
// variants for bias and ALiBi and dropout keep 18, 79 and 49 registers in
// scratch, some of them read back in the loop.
// Measured at 1 x 16/8 x 2048 x 256 bf16 causal (69 GFLOP): 102 us with the
// dS stores in two shares and 14 for their merge, against 920 us for
// bwd_dkdv_kernel; dQ from that dS 47 us against 453 us for bwd_dq_kernel.
// Without a mask (103 GFLOP), bwd_dkdv_kernel and this: plain 1012 and 157,
// softcap 1142 and 222, ALiBi 1141 and 285, a bf16 bias 1704 and 415, dropout
// 1534 and 448.
#pragma once

#include <type_traits>

#include "fa_bwd16.hpp"

namespace fa {

// A workgroup owns BN keys (NK pairs of waves, 32 keys each) and splits their
// query steps in two halves of four waves, as dkdv16_kernel does.  The two
// waves of a SIMD (w and w + 4) take opposite roles.
template <int D>
struct DkdvRolesCfg {
  static_assert(D == 256, "dkdv16_kernel holds both sums of the narrower heads in one wave");
  static constexpr int NK = 2;  // wave pairs per half
  static constexpr int NW = 4 * NK;
  static constexpr int NT = 64 * NW;
  static constexpr int NTH = NT / 2;
  static constexpr int BN = 32 * NK;
  static constexpr int BMQ = 32;
  static constexpr int QT = BMQ * D;  // elements per Q / dO tile
  static constexpr int STAGE_BYTES = 2 * QT * 2 + 2 * BMQ * 4;
  static constexpr int HALF_BYTES = 2 * STAGE_BYTES;
  static constexpr int XCH_FLOATS = 1024;  // one pair's P of a step
  static constexpr int LOOP_BYTES = 2 * HALF_BYTES + 2 * NK * XCH_FLOATS * 4;
  static constexpr int NSTEP = D / 16;
  static constexpr int NPV = BMQ / 16;
  static constexpr int NDB = D / 32;
  static constexpr int PARK_WAVE_BYTES = NDB * 4096;
  static constexpr int MERGE_BYTES = 2 * NK * PARK_WAVE_BYTES;
  static constexpr int LDS_BYTES = LOOP_BYTES > MERGE_BYTES ? LOOP_BYTES : MERGE_BYTES;
  static_assert(LDS_BYTES <= 160 * 1024, "one workgroup per CU");
  static_assert(32 * (D + 8) * 2 <= PARK_WAVE_BYTES, "rows leave through the wave's merge block");
};

// nshare > 1: the query steps of a key block (of each of its query heads) are
// shared out over nshare workgroups, blockIdx = (block, KV head) * nshare +
// share, which leave their sums in `part` for dkdv_merge_kernel.
template <typename Tag, int D, int MODE>
__global__ __launch_bounds__(512, 1) void dkdv_roles_kernel(fa_bwd_params p, int num_n_blocks, int nshare,
                                                            float* part) {
  using C = DkdvRolesCfg<D>;
  using EL = Elem<Tag>;
  using S = uint16_t;
  extern __shared__ __align__(256) unsigned char smem_raw[];
  const fa_fwd_params& f = p.fwd;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qhalf = wave8 / (2 * C::NK);
  const int wave = wave8 % (2 * C::NK);
  const int pair = wave >> 1;
  const bool kwave = ((wave & 1) ^ qhalf) != 0;  // role
  const int slot = 2 * pair + (kwave ? 1 : 0);   // merge block, the same in both halves
  const int htid = tid % C::NTH;
  const int h = lane >> 5, l32 = lane & 31;
  const int bhk_count = f.batch * f.heads_kv;
  // Low key blocks first: under causal masking they see the most query rows.
  const int item = blockIdx.x / nshare;
  const int share = blockIdx.x - item * nshare;
  const int nblk = item / bhk_count;
  const int bhk = item - nblk * bhk_count;
  const int b = bhk / f.heads_kv, hk = bhk - b * f.heads_kv;
  const int group = f.heads_q / f.heads_kv;

  int q_start = 0, sq = f.seqlen_q, k_start = 0, sk = f.seqlen_k;
  if (f.cu_seqlens_q) {
    bounded_seq(f.cu_seqlens_q, b, f.total_q, q_start, sq);
    bounded_seq(f.cu_seqlens_k, b, f.total_k, k_start, sk);
  }
  const int n0 = nblk * C::BN;
  if (n0 >= sk || num_n_blocks <= 0) return;

  const int n0w = n0 + 32 * pair;
  const int ncols = min(32, sk - n0w);

  // The resident operands (MFMA B layout): K rows of the V wave, V rows of
  // the K wave; rows past the last key are zero.
  s16x8 op[C::NSTEP];
  {
    const int64_t st = kwave ? f.v_stride[2] : f.k_stride[2];
    const S* base = kwave ? reinterpret_cast<const S*>(f.v) + b * f.v_stride[0] + hk * f.v_stride[1]
                          : reinterpret_cast<const S*>(f.k) + b * f.k_stride[0] + hk * f.k_stride[1];
    const S* row = base + (int64_t)(k_start + min(n0w + l32, sk - 1)) * st + 8 * h;
#pragma unroll
    for (int s = 0; s < C::NSTEP; ++s) op[s] = load_op<Tag>(row + 16 * s);
    wait_vm_all();
    if (n0w + l32 >= sk) {
#pragma unroll
      for (int s = 0; s < C::NSTEP; ++s) op[s] = zero_op<Tag>();
    }
  }

  f32x16 acc[C::NDB];  // dV (V wave) or dK (K wave)
#pragma unroll
  for (int i = 0; i < C::NDB; ++i) acc[i] = zero16();

  DmaLeanTile<C::BMQ, D, C::NTH> qd, gd;
  qd.init(f.q_stride[2], htid);
  gd.init(p.dout_stride[2], htid);
  unsigned char* const hsmem = smem_raw + qhalf * C::HALF_BYTES;
  const uint32_t lds0 = lds_addr(hsmem);
  const uint32_t row_off = row_lane_off<D>(lane), tr_off = tr_lane_off<D>(lane);
  static_assert(C::STAGE_BYTES % 256 == 0, "row_op / tr_op addressing");
  float* const xch = reinterpret_cast<float*>(smem_raw + 2 * C::HALF_BYTES) + (qhalf * C::NK + pair) * C::XCH_FLOATS;
  const int nlast = min(n0 + C::BN, sk) - 1;

  // (dS scratch is for dense problems only at this head dim)
  const int64_t ds_base = (int64_t)b * f.heads_q * ds_region_elems(sq, sk);
  for (int g = 0; g < group; ++g) {
    const int hq = hk * group + g;
    const Mods md = make_mods(f, b, hq, sq, sk);
    const float c = md.scale_log2;
    const S* qbase = reinterpret_cast<const S*>(f.q) + b * f.q_stride[0] + hq * f.q_stride[1] +
                     (int64_t)q_start * f.q_stride[2];
    const S* gbase = reinterpret_cast<const S*>(p.dout) + b * p.dout_stride[0] + hq * p.dout_stride[1] +
                     (int64_t)q_start * p.dout_stride[2];
    const float* lbase = f.lse + b * f.lse_stride[0] + hq * f.lse_stride[1] + (int64_t)q_start * f.lse_stride[2];
    const float* dbase = p.delta + b * p.delta_stride[0] + hq * p.delta_stride[1] +
                         (int64_t)q_start * p.delta_stride[2];
    const int64_t qs = f.q_stride[2], gs = p.dout_stride[2];

    int mlo = 0, mhi = sq;
    if (f.causal) mlo = max(mlo, n0 - md.off);
    if (f.window_right >= 0) mlo = max(mlo, n0 - md.off - f.window_right);
    if (f.window_left >= 0) mhi = min(mhi, nlast - md.off + f.window_left + 1);
    mlo = max(mlo, 0) / C::BMQ * C::BMQ;
    int nsteps = mhi > mlo ? (mhi - mlo + C::BMQ - 1) / C::BMQ : 0;
    const int step0 = nsteps * share / nshare;
    nsteps = nsteps * (share + 1) / nshare - step0;
    mlo += step0 * C::BMQ;
    // Steps [0, nh0) go to half 0, [nh0, nsteps) to half 1; both run nh0
    // iterations so their barriers line up.
    const int nh0 = (nsteps + 1) / 2;
    const int my_first = qhalf == 0 ? 0 : nh0;
    const int my_count = qhalf == 0 ? nh0 : nsteps - nh0;

    float lreg = 0.f, dreg = 0.f;  // this thread's lse2 / delta for the next stage
    auto load_stage = [&](int m0, int st) {
      const int rows = min(C::BMQ, sq - m0);
      const uint32_t base = lds0 + (uint32_t)(st * C::STAGE_BYTES);
      qd.load(rows_rsrc_words<D>(qbase + (int64_t)m0 * qs, qs, rows), base, wave);
      gd.load(rows_rsrc_words<D>(gbase + (int64_t)m0 * gs, gs, rows), base + C::QT * 2u, wave);
      if (htid < C::BMQ) {
        const int m = min(m0 + htid, sq - 1);
        lreg = lbase[(int64_t)m * f.lse_stride[2]];
        dreg = dbase[(int64_t)m * p.delta_stride[2]];
      }
    };
    // Row constants: lse2 (MODE 3: cap2 - lse2) for the V wave, -delta (the
    // dP accumulator's seed; delta itself under dropout) for the K wave.
    auto store_stage = [&](int st, int m0) {
      if (htid < C::BMQ) {
        float* lf = reinterpret_cast<float*>(hsmem + st * C::STAGE_BYTES + 2 * C::QT * 2);
        const float l2v = (m0 + htid < sq) ? lse2_of(lreg) : __builtin_inff();
        lf[htid] = (MODE == 3) ? md.cap2 - l2v : l2v;
        lf[C::BMQ + htid] = (MODE != 2) ? -dreg : dreg;
      }
    };

    // dS of this wave's first key in the scratch (see dkdv16_kernel).
    bool ds_on = false;
    const S* dsn = nullptr;
    if (p.ds_workspace != nullptr) {
      const int64_t region = ds_region_at(p, ds_base, hq, sq, sk);
      ds_on = region >= 0;
      dsn = reinterpret_cast<const S*>(p.ds_workspace) + (ds_on ? region : 0) +
            (int64_t)(n0w / kDsTileKeys) * ds_qblocks(sq) * kDsTileElems + (n0w % kDsTileKeys) * kDsSubQueries;
    }
    const VisBounds kvb = key_block_bounds(md, n0w, ncols);
    if (my_count > 0) {
      const int m_first = mlo + my_first * C::BMQ;
      load_stage(m_first, 0);
      store_stage(0, m_first);
    }
    wait_vm_all();
    __syncthreads();
    for (int t = 0; t < nh0; ++t) {
      const int m0 = mlo + (my_first + t) * C::BMQ;
      const int st = t & 1;
      if (t + 1 < my_count) load_stage(m0 + C::BMQ, st ^ 1);
      const int vis = t < my_count ? bounds_vis(kvb, m0 + md.off, min(m0 + C::BMQ, sq) - 1 + md.off) : 0;
      const unsigned char* base = hsmem + st * C::STAGE_BYTES;
      const uint32_t qtile = lds0 + (uint32_t)(st * C::STAGE_BYTES);
      const float* L2 = reinterpret_cast<const float*>(base + 2 * C::QT * 2);
      const float* DL = L2 + C::BMQ;

      f32x16 x;  // S then P (V wave), dP then dS (K wave)
      s16x8 xb[C::NPV];
      if (vis) {
        // Both roles: x += tile . resident operand.
        if (kwave && MODE != 2) {
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4) {
            const f32x4 d = *reinterpret_cast<const f32x4*>(DL + 8 * q4 + 4 * h);
#pragma unroll
            for (int r = 0; r < 4; ++r) x[4 * q4 + r] = d[r];
          }
        } else {
          x = zero16();
        }
        const uint32_t ra = tile_lane(qtile + (kwave ? C::QT * 2u : 0u), row_off);
#pragma unroll
        for (int i = 0; i < C::NSTEP; ++i) {
          // k-steps 8 apart share an address (row_op): taken in turn.
          const int s = (i >> 1) + 8 * (i & 1);
          x = EL::mma(row_op<D>(ra, s), op[s], x);
        }
        sched_reads<C::NSTEP, 2, 1, 1>();
        if (!kwave) {
          // P, and what the K wave needs of it: P times the softcap's
          // derivative, negative where dropout dropped the pair.  (All of the
          // derivative: a dS stored as a quarter, as the narrower kernels do,
          // falls below fp16's smallest normal number four times sooner.  At
          // 512 x 512, softcap 50, upstream gradients of 1e-3, dK is off by
          // 4.4e-4 of its norm that way's 1.4e-3.)
          auto scores = [&](auto cap_t, auto bias_t, auto alibi_t, auto mask_t) {
            constexpr bool CAP = decltype(cap_t)::value;
            constexpr bool MASK = decltype(mask_t)::value;
            Span rs{0, 0};
            if constexpr (MASK) {
              int rlo, rhi;
              row_bounds(md, n0w + l32, rlo, rhi);
              rs = make_span(rlo, rhi, m0 + 4 * h);
            }
            f32x16 w;
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
              const f32x4 l2 = *reinterpret_cast<const f32x4*>(L2 + 8 * q4 + 4 * h);
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const int i = 4 * q4 + r;
                float pv, tc = 0.f, wv;
                if constexpr (MODE == 0) {
                  pv = __builtin_amdgcn_exp2f(__builtin_fmaf(x[i], c, -l2[r]));
                } else if constexpr (MODE == 3) {
                  const float rr = softcap_r(md, x[i]);
                  pv = __builtin_amdgcn_exp2f(__builtin_fmaf(md.cap2_m2, rr, l2[r]));
                  tc = __builtin_fmaf(-rr, rr, rr);
                } else {
                  const int m = m0 + acc_row(i, h), n = n0w + l32;
                  float sc;
                  if constexpr (MODE == 2) sc = score<true>(md, x[i], m, n, tc);
                  else sc = score_m<CAP, decltype(bias_t)::value, decltype(alibi_t)::value>(md, x[i], m, n, tc);
                  pv = __builtin_amdgcn_exp2f(sc - l2[r]);
                }
                if constexpr (MASK) pv = in_span(rs, acc_row(i, 0)) ? pv : 0.f;
                wv = pv;
                if constexpr (MODE == 3) wv *= 4.f * tc;
                else if constexpr (CAP) wv *= (1.f - tc * tc);
                if constexpr (MODE == 2) {
                  if (md.drop_p > 0.f) {
                    const bool keep = dropout_keep(md, m0 + acc_row(i, h), n0w + l32);
                    pv = keep ? pv * md.drop_scale : 0.f;
                    wv = keep ? wv : -wv;
                  }
                }
                x[i] = pv;
                w[i] = wv;
              }
            }
            park_acc(xch, lane, w);
          };
          using T_ = std::true_type;
          using F_ = std::false_type;
          using B0 = std::integral_constant<int, 0>;
          if constexpr (MODE == 0 || MODE == 3) {
            if (vis == 1) scores(F_{}, B0{}, F_{}, T_{});
            else scores(F_{}, B0{}, F_{}, F_{});
          } else if constexpr (MODE == 2) {
            // One variant that tests for each modifier (CAP: tc is 0 without
            // a softcap) and masks: sixteen of them left 1195 reads of spilled
            // registers and a call in the step loop (1 x 16/8 x 2048 x 256
            // bf16, dropout: dK/dV 2673 -> 448 us).
            scores(T_{}, B0{}, F_{}, T_{});
          } else {
            if (vis == 1) dispatch_mods(md, [&](auto a, auto b_, auto c_) { scores(a, b_, c_, T_{}); });
            else dispatch_mods(md, [&](auto a, auto b_, auto c_) { scores(a, b_, c_, F_{}); });
          }
#pragma unroll
          for (int j = 0; j < C::NPV; ++j) xb[j] = pack_op<Tag>(x, j);
        }
      }
      __syncthreads();  // P of every pair is in LDS
      if (vis) {
        if (kwave) {
          const f32x16 w = unpark_acc(xch, lane);
          if constexpr (MODE == 2) {
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
              const f32x4 d = *reinterpret_cast<const f32x4*>(DL + 8 * q4 + 4 * h);
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const int i = 4 * q4 + r;
                const bool keep = !(__float_as_uint(w[i]) >> 31);
                const float dp = keep ? x[i] * md.drop_scale : 0.f;
                x[i] = fabsf(w[i]) * (dp - d[r]);
              }
            }
          } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) x[i] *= w[i];
          }
#pragma unroll
          for (int j = 0; j < C::NPV; ++j) xb[j] = pack_op<Tag>(x, j);
        }
        const uint32_t ta = tile_lane(qtile + (kwave ? 0u : C::QT * 2u), tr_off);
#pragma unroll
        for (int j = 0; j < C::NPV; ++j)
#pragma unroll
          for (int db = 0; db < C::NDB; ++db) acc[db] = EL::mma(tr_op<D>(ta, j, db), xb[j], acc[db]);
        sched_reads<C::NPV * C::NDB, 2, 2, 1>();
      }
      if (t + 1 < my_count) store_stage(st ^ 1, m0 + C::BMQ);
      const bool ds_store = ds_on && vis && kwave;
      if (ds_store) {
        // As in dkdv16_kernel: one permlane32 swap per dword pair gives each
        // lane 16 consecutive queries of its key, two 16-byte stores.
        static_assert(C::NPV == 2 && C::BMQ == kDsSubQueries, "a query step is one dS sub-tile");
        u32x4 w0 = __builtin_bit_cast(u32x4, xb[0]), w1 = __builtin_bit_cast(u32x4, xb[1]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const auto r = __builtin_amdgcn_permlane32_swap(w0[i], w1[i], false, false);
          w0[i] = r[0];
          w1[i] = r[1];
        }
        // A buffer window over this wave's rows of the sub-tile: lanes past
        // the last key fall outside it and store nothing, yet every wave
        // issues the same stores (the wait below counts them).
        const int rows = min(32, ncols);
        const S* at = dsn + (int64_t)(m0 / kDsTileQueries) * kDsTileElems +
                      (m0 % kDsTileQueries) / kDsSubQueries * kDsSubElems;
        const __amdgpu_buffer_rsrc_t rs = rows_rsrc<kDsSubQueries>(at, kDsSubQueries, rows);
        const uint32_t o = (uint32_t)(l32 * kDsSubQueries * 2 + 32 * h);
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{w0[0], w0[1], w1[0], w1[1]}, rs, o, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{w0[2], w0[3], w1[2], w1[3]}, rs, o + 16, 0, 0);
      }
      // The next stage must have landed; this step's dS stores, issued after
      // its loads, may still be in flight.
      if (ds_store) wait_vm<2>();
      else wait_vm_all();
      __syncthreads();
    }
  }

  // First query half + second query half, in that order.
  {
    __syncthreads();
    float* ow = reinterpret_cast<float*>(smem_raw) + slot * C::NDB * 1024;
    if (qhalf == 1) {
#pragma unroll
      for (int db = 0; db < C::NDB; ++db) park_acc(ow + db * 1024, lane, acc[db]);
    }
    __syncthreads();
    if (qhalf == 1) return;
#pragma unroll
    for (int db = 0; db < C::NDB; ++db) acc[db] += unpark_acc(ow + db * 1024, lane);
  }
  if (nshare > 1) {
    float* pw = part + ((int64_t)blockIdx.x * 2 * C::NK + slot) * (C::NDB * 1024);
#pragma unroll
    for (int db = 0; db < C::NDB; ++db) park_acc(pw + db * 1024, lane, acc[db]);
    return;
  }
  // Whole-row stores through this wave's merge block (read back already).
  const int64_t ost = kwave ? p.dk_stride[2] : p.dv_stride[2];
  S* orow0 = kwave ? reinterpret_cast<S*>(p.dk) + b * p.dk_stride[0] + hk * p.dk_stride[1]
                   : reinterpret_cast<S*>(p.dv) + b * p.dv_stride[0] + hk * p.dv_stride[1];
  const float sc = kwave ? f.softmax_scale : 1.f;
  uint16_t* const stage = reinterpret_cast<uint16_t*>(smem_raw + slot * C::PARK_WAVE_BYTES);
  store_rows_staged<Tag, D>(acc, sc, stage, orow0 + (int64_t)(k_start + n0w) * ost, ost, ncols, lane);
}

// dK / dV of the shares above, added in share order: 64 columns of one item
// per workgroup, one wave per (pair, role).
template <typename Tag, int D>
__global__ __launch_bounds__(256) void dkdv_merge_kernel(fa_bwd_params p, int nshare, const float* part) {
  using C = DkdvRolesCfg<D>;
  using S = uint16_t;
  constexpr int MD = 64, PER = D / MD;
  static_assert(2 * C::NK == 4, "one wave per merge block");
  __shared__ __align__(16) uint16_t stage[4 * 32 * (MD + 8)];
  const fa_fwd_params& f = p.fwd;
  const int lane = threadIdx.x & 63;
  const int slot = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool kwave = (slot & 1) != 0;
  const int cc = blockIdx.x % PER, item = blockIdx.x / PER;
  const int bhk_count = f.batch * f.heads_kv;
  const int nblk = item / bhk_count, bhk = item - nblk * bhk_count;
  const int b = bhk / f.heads_kv, hk = bhk - b * f.heads_kv;
  const int n0w = nblk * C::BN + 32 * (slot >> 1);
  f32x16 acc[MD / 32];
#pragma unroll
  for (int i = 0; i < MD / 32; ++i) acc[i] = zero16();
  for (int s = 0; s < nshare; ++s) {
    const float* pw = part + (((int64_t)item * nshare + s) * 4 + slot) * (C::NDB * 1024) + cc * (MD / 32) * 1024;
#pragma unroll
    for (int i = 0; i < MD / 32; ++i) acc[i] += unpark_acc(pw + i * 1024, lane);
  }
  const int64_t ost = kwave ? p.dk_stride[2] : p.dv_stride[2];
  S* orow0 = kwave ? reinterpret_cast<S*>(p.dk) + b * p.dk_stride[0] + hk * p.dk_stride[1]
                   : reinterpret_cast<S*>(p.dv) + b * p.dv_stride[0] + hk * p.dv_stride[1];
  const float sc = kwave ? f.softmax_scale : 1.f;
  store_rows_staged<Tag, MD>(acc, sc, stage + slot * 32 * (MD + 8), orow0 + (int64_t)n0w * ost + cc * MD, ost,
                             min(32, f.seqlen_k - n0w), lane);
}

}  // namespace fa

// Fused row blocks of a narrow layer stack for gfx950 (kf_layer_block).
//
// Everything of a transformer layer except attention works on rows: out_proj, the two
// residual adds with the row mask, both LayerNorms, the feed-forward and the next layer's
// QKV projection. For a narrow model (d <= 256) one block of BM rows fits on a CU, so one
// kernel takes those rows from the attention output to the next attention's operands:
//
//   s = (res + ctx.Wo^T + bo) * keep;  h = LN(s)                            (TAIL)
//   s = (s + gelu(h.W1^T + b1).W2^T + b2) * keep;  h = LN(s)                (TAIL)
//   q, k, v^T = h.Wqkv^T + bqkv in the attention layout, or y = h [* keep]  (QKV / final)
//
// (kernelforge/optimized.py:483-585; without TAIL: s = x * keep, h = LN(s), then QKV). The
// row values s stay in fp32 registers and the 16-bit operands (planes of ctx, h, the
// hidden chunk) in LDS; only ctx and res are read and only s and the outputs written.
//
// What bounds it: for few rows the latency of the chain of products, each block streaming every
// weight. For many rows (10000 x 128 rows of d = F = 128, f16x3; profiles/pmc_layer_kernel.txt) the
// tail runs VALU instructions (LayerNorm, GELU, plane splits) in 52 % of the SIMDs' cycles and MFMAs
// in 25 %, at 2.6 TB/s; the entry block 32 % and 24 %, at 3.6 TB/s, its wavefronts waiting to issue
// for most of the rest. HBM traffic is what the operands are, each once: per element of [M, d] 16
// bytes for an entry block, 24 for a tail with the next projections, 12 for the last tail, where
// separate launches of that one's operations move 52. Measured on MI355X against the separate
// kernels that it replaced: that model, one layer, 4.95 -> 2.00 ms; four layers of d = F = 128 over
// one 128-token sequence 206 -> 69.5 us; d 64, F 256, 64 x 1024 rows 185 -> 101 us. Against today's
// separate kernels (small GEMM tiles) see FusedTransformer.ROW_KERNEL_BYTES.
//
// Split: a block has d / 16 / FN wavefronts, each owning 16 FN columns of every product and all
// BM rows. The product is formed as W . A^T, so a lane holds four
// consecutive columns of one row (as in the GEMM kernels); the v part swaps the operands, so
// a lane holds four consecutive tokens of one column and stores V^T in 8-byte pieces. Weights
// are read from global memory (L2) straight into MFMA operand registers: each block reads
// every weight once and wavefronts share none, so LDS staging would only add a copy. They are
// laid out in fragment order (kf_fragments), so that a wavefront's load is 1 KB of whole lines:
// from the row-major weight, sixteen 64-byte pieces of sixteen lines, the loads ran at about
// 16 B/clk per CU (tail + QKV, d 256, F 1024, M 256: 87 us, 31 us in fragment order). The fragments
// form one stream over all products (a
// ring of GK k-steps): a k-step's registers are reloaded, for the next group of k-steps or
// the next product, as soon as its MFMAs have been issued, so the loads of a product are in
// flight during the previous product's epilogue and LayerNorm.
//
// Row statistics: each wavefront reduces its 16-column tiles to (mean, M2) with shuffles and
// the d / 16 tiles are merged through LDS (the parallel variance of Chan, Golub and LeVeque),
// in column order: a row's results do not depend on BM or FN.
#include <type_traits>

#include "kf_common.h"

// Multiply-adds are written out: left to the compiler they are fused differently in different
// instantiations, and the results of a row would depend on the rows of its block.
#pragma clang fp contract(off)

namespace kf {

struct LayerArgs {
  // TAIL
  const _Float16* ctx_hi; const _Float16* ctx_lo;
  const float* res; int64_t ld_res;
  const uint8_t* keep;
  const _Float16* wo_hi; const _Float16* wo_lo; const float* bo;
  const float* g2; const float* b2n; float eps2;
  const _Float16* w1_hi; const _Float16* w1_lo; const float* b1;
  const _Float16* w2_hi; const _Float16* w2_lo; const float* b2;
  // the LayerNorm that ends the block
  const float* gn; const float* bn; float epsn;
  float* s_out;
  // QKV
  const _Float16* wq_hi; const _Float16* wq_lo; const float* bq;
  float* q_out; _Float16* k_hi; _Float16* k_lo; _Float16* vt_hi; _Float16* vt_lo;
  int64_t sp; int S;
  // final
  void* y; int y_dtype;
  int M, F;
  int m_out, m_f1, m_f2, m_attn;      // MFMA modes: KF_MMA_F16 / F16X2 / F16X3
};

template <int D_, int BM_, int FN_> struct LayerCfg {
  static constexpr int D = D_, BM = BM_, FN = FN_;
  static constexpr int NW = D / 16 / FN, NT = 64 * NW;
  static constexpr int FM = BM / 16;
  static constexpr int KS = D / 32;                         // k-steps of a D-wide product
  static constexpr int GK = KS <= 4 ? KS : KS % 4 == 0 ? 4 : 3;
  static constexpr int NG = KS / GK;
  static constexpr int LDA = D + 8;                         // LDS row stride (elements)
  static_assert(D % 32 == 0 && D % (16 * FN) == 0 && BM % 16 == 0, "layer tile");
  static_assert(KS % GK == 0, "k-steps come in whole groups");
  // registers: two blocks a CU where a block has 8 wavefronts or more (the row loads of one
  // hide behind the products of the other)
  static constexpr int WPE = FN > 1 ? 2 : NW >= 16 ? 4 : NW >= 8 ? 4 : NW >= 6 ? 3 : 2;
};

enum { LAYER_TAIL = 1, LAYER_QKV = 2 };

__device__ __forceinline__ int mode_planes_a(int mode) { return mode == KF_MMA_F16X3 ? 2 : 1; }

// UNI: every stage is f16x3 (the default plan), known at compile time; else the modes are
// read from the arguments (wave-uniform branches around whole groups of k-steps).
template <class C, int ROLE, bool UNI>
__global__ __launch_bounds__(C::NT) __attribute__((amdgpu_waves_per_eu(C::WPE)))
void layer_kernel(LayerArgs g) {
  constexpr bool TAIL = ROLE & LAYER_TAIL, QKV = ROLE & LAYER_QKV;
  constexpr int D = C::D, BM = C::BM, FN = C::FN, FM = C::FM, LDA = C::LDA;
  __shared__ __attribute__((aligned(16))) _Float16 xa[2][BM * LDA];
  __shared__ __attribute__((aligned(16))) _Float16 hid[TAIL ? 2 : 1][TAIL ? BM * LDA : 8];
  constexpr int CT = D / 16;                     // 16-column tiles of a row
  __shared__ float2 red[CT][BM];       // (mean, M2) of each 16-column tile, per row
  // biases and norm parameters: bo, norm2 w / b, b2 | norm w / b | bqkv
  constexpr int kOwn = TAIL ? 4 : 0, kPar = kOwn + 2 + (QKV ? 3 : 0);
  __shared__ __attribute__((aligned(16))) float par[kPar * D];
  constexpr int NPT = (kPar * D / 4 + C::NT - 1) / C::NT;   // 16-byte pieces per thread

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, grp = lane >> 4;
  const int m0 = blockIdx.x * BM;
  const int col0 = wave * 16 * FN;               // this wavefront's first column
  const int nc = TAIL ? (g.F + D - 1) / D : 0;   // hidden chunks of D columns

  // ---- weight stream: products p = 0 (out_proj), 1 + 2c (ffn_in chunk c), 2 + 2c (ffn_out
  // chunk c), then the q, k, v parts
  constexpr int kFirst = TAIL ? 0 : 1;
  const int p_qkv = TAIL ? 1 + 2 * nc : 1;
  const int p_end = p_qkv + (QKV ? 3 : 0);
  half8 w[C::GK][FN][2];
  const _Float16* nw_hi = nullptr;               // source of the group being fetched
  const _Float16* nw_lo = nullptr;
  int nw_at[FN], nw_k0 = 0, nw_kt = 0;           // its column tiles, first k-step, k-steps
  auto aim = [&](int p, int grpk) KF_INLINE {
    if (p >= p_end) { p = p_end - 1; }           // past the end: refetch (never used)
    int tile = 0, tiles = D / 16;
    nw_kt = C::KS;
    nw_k0 = grpk * C::GK;
    if (TAIL && p == 0) {
      nw_hi = g.wo_hi; nw_lo = g.wo_lo;
    } else if (TAIL && p < p_qkv) {
      const int c = (p - 1) >> 1;
      if ((p & 1) == 1) { nw_hi = g.w1_hi; nw_lo = g.w1_lo; tile = c * (D / 16); tiles = g.F / 16; }
      else { nw_hi = g.w2_hi; nw_lo = g.w2_lo; nw_kt = g.F / 32; nw_k0 += c * C::KS; }
    } else {
      nw_hi = g.wq_hi; nw_lo = g.wq_lo; tile = (p - p_qkv) * (D / 16); tiles = 3 * (D / 16);
    }
#pragma unroll
    for (int i = 0; i < FN; ++i) nw_at[i] = min(tile + col0 / 16 + i, tiles - 1) * nw_kt;
  };
  auto fetch = [&](int ks, auto LO) KF_INLINE {
    const int kk = min(nw_k0 + ks, nw_kt - 1);
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const int64_t at = (int64_t)(nw_at[i] + kk) * 512;     // wave-uniform
      w[ks][i][0] = *(const half8*)(nw_hi + at + lane * 8);
      if constexpr (decltype(LO)::value) w[ks][i][1] = *(const half8*)(nw_lo + at + lane * 8);
    }
  };
  using Yes = std::true_type;
  using No = std::false_type;

  struct Acc { f32x4 v[FN][FM]; };
  auto zero = [&](Acc& c) KF_INLINE {
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) c.v[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  // acc += product p of the rows in `a`; fetches the group after each group as it goes
  auto group = [&](Acc& c, const _Float16 (*a)[BM * LDA], int gk, auto Z, auto PAc, auto PWc,
                   auto SWc, auto LO) KF_INLINE {
    constexpr int PA = decltype(PAc)::value, PW = decltype(PWc)::value;
#pragma unroll
    for (int ks = 0; ks < C::GK; ++ks) {
      half8 af[FM][PA];
#pragma unroll
      for (int j = 0; j < FM; ++j)
#pragma unroll
        for (int pl = 0; pl < PA; ++pl)
          af[j][pl] = *(const half8*)&a[pl][(16 * j + r) * LDA + (gk * C::GK + ks) * 32 + grp * 8];
      auto mm = [&](const half8& wv, const half8& av, f32x4& d) KF_INLINE {
        if constexpr (decltype(SWc)::value) d = mma16(av, wv, d);
        else d = mma16(wv, av, d);
      };
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        // a product that starts from zero passes it to its first MFMAs
        if constexpr (decltype(Z)::value) {
          if (gk == 0 && ks == 0)
#pragma unroll
            for (int j = 0; j < FM; ++j) c.v[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        if constexpr (PA == 2)
#pragma unroll
          for (int j = 0; j < FM; ++j) mm(w[ks][i][0], af[j][1], c.v[i][j]);
        if constexpr (PW == 2)
#pragma unroll
          for (int j = 0; j < FM; ++j) mm(w[ks][i][1], af[j][0], c.v[i][j]);
#pragma unroll
        for (int j = 0; j < FM; ++j) mm(w[ks][i][0], af[j][0], c.v[i][j]);
      }
      fetch(ks, LO);
    }
  };
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  auto product = [&](Acc& c, const _Float16 (*a)[BM * LDA], int p, int mode, auto Z, auto SWc)
      KF_INLINE {
#pragma unroll
    for (int gk = 0; gk < C::NG; ++gk) {
      const bool more = gk + 1 < C::NG;
      aim(more ? p : p + 1, more ? gk + 1 : 0);
      if constexpr (UNI) {
        group(c, a, gk, Z, I2{}, I2{}, SWc, Yes{});
      } else {
        const bool lo = nw_lo != nullptr;
        if (mode == KF_MMA_F16X3) {
          if (lo) group(c, a, gk, Z, I2{}, I2{}, SWc, Yes{});
          else group(c, a, gk, Z, I2{}, I2{}, SWc, No{});
        } else if (mode == KF_MMA_F16X2) {
          if (lo) group(c, a, gk, Z, I1{}, I2{}, SWc, Yes{});
          else group(c, a, gk, Z, I1{}, I2{}, SWc, No{});
        } else {
          if (lo) group(c, a, gk, Z, I1{}, I1{}, SWc, Yes{});
          else group(c, a, gk, Z, I1{}, I1{}, SWc, No{});
        }
      }
    }
  };

  // ---- prologue: everything the block reads first goes out at once, what is needed first
  // in front (loads return in order): ctx rows and parameters for LDS, mask bytes, the first
  // weights, the residual rows
  constexpr int CPR = D / 8;                     // 16-byte chunks per row of ctx
  constexpr int NCH = TAIL ? BM * CPR : 0, NCT = (NCH + C::NT - 1) / C::NT;
  U4 cx[2][NCT > 0 ? NCT : 1];
  if constexpr (TAIL) {
    const bool two = UNI || g.m_out == KF_MMA_F16X3;
    const _Float16* lo = two ? g.ctx_lo : g.ctx_hi;
#pragma unroll
    for (int q = 0; q < NCT; ++q) {
      const int ch = min(q * C::NT + tid, NCH - 1);
      const int64_t at = (int64_t)min(m0 + ch / CPR, g.M - 1) * D + (ch % CPR) * 8;
      cx[0][q] = *(const U4*)(g.ctx_hi + at);
      cx[1][q] = *(const U4*)(lo + at);
    }
  }
  f32x4 pv[NPT];
#pragma unroll
  for (int q = 0; q < NPT; ++q) {
    const int f = min(q * C::NT + tid, kPar * D / 4 - 1), pi = f / (D / 4);
    const float* src = pi == kOwn ? g.gn : pi == kOwn + 1 ? g.bn : g.bq + (pi - kOwn - 2) * D;
    if constexpr (TAIL) src = pi == 0 ? g.bo : pi == 1 ? g.g2 : pi == 2 ? g.b2n : pi == 3 ? g.b2 : src;
    pv[q] = *(const f32x4*)(src + (f % (D / 4)) * 4);
  }
  // no mask: any readable byte will do
  const uint8_t* kp = g.keep ? g.keep : (const uint8_t*)g.res;
  uint8_t kb[FM];
#pragma unroll
  for (int j = 0; j < FM; ++j) kb[j] = kp[min(m0 + 16 * j + r, g.M - 1)];
  aim(kFirst, 0);
#pragma unroll
  for (int ks = 0; ks < C::GK; ++ks) {
    if (UNI || nw_lo != nullptr) fetch(ks, Yes{});
    else fetch(ks, No{});
  }
  Acc s;
#pragma unroll
  for (int j = 0; j < FM; ++j) {
    const int64_t m = min(m0 + 16 * j + r, g.M - 1);
#pragma unroll
    for (int i = 0; i < FN; ++i)
      s.v[i][j] = *(const f32x4*)(g.res + m * g.ld_res + col0 + 16 * i + 4 * grp);
  }
  if constexpr (TAIL) {
#pragma unroll
    for (int q = 0; q < NCT; ++q) {
      const int ch = q * C::NT + tid;
      if (NCH % C::NT == 0 || ch < NCH) {
        const int at = (ch / CPR) * LDA + (ch % CPR) * 8;
        *(U4*)&xa[0][at] = cx[0][q];
        *(U4*)&xa[1][at] = cx[1][q];
      }
    }
  }
#pragma unroll
  for (int q = 0; q < NPT; ++q)
    if (q * C::NT + tid < kPar * D / 4) *(f32x4*)&par[(q * C::NT + tid) * 4] = pv[q];
  lds_barrier();
  float kv[FM];
#pragma unroll
  for (int j = 0; j < FM; ++j) kv[j] = g.keep == nullptr || kb[j] ? 1.0f : 0.0f;
  auto param = [&](int which, int i) KF_INLINE {   // four columns of a parameter row
    return *(const f32x4*)&par[which * D + col0 + 16 * i + 4 * grp];
  };

  // sum over the four column groups of a row, in every lane of the row
  auto row_sum = [&](float t) KF_INLINE {
    auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(t), __float_as_uint(t), false, false);
    t = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(t), __float_as_uint(t), false, false);
    return __uint_as_float(q[0]) + __uint_as_float(q[1]);
  };
  // Two quads of adjacent tiles p and q, traded between neighbouring lane groups: each lane
  // ends with eight consecutive values of one tile, those from offset pair8 on. Stores then
  // leave in 16-byte pieces, a wavefront's row (or V^T column) in 64 bytes of 16-bit values
  // instead of 32 (10000 x 128 rows of d 128: entry, attention and tail 2150 -> 1999 us).
  auto trade = [&](const f32x4& p, const f32x4& q, float* v) KF_INLINE {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(p[e]), __float_as_uint(q[e]), false, false);
      v[e] = __uint_as_float(t[0]);
      v[4 + e] = __uint_as_float(t[1]);
    }
  };
  const int pair8 = 16 * (grp & 1) + 4 * (grp & 2);
  // eight fp32 values, or their fp16 plane(s), at an element offset
  auto put8 = [&](float* p, int64_t at, const float* v) KF_INLINE {
    *(f32x4*)(p + at) = f32x4{v[0], v[1], v[2], v[3]};
    *(f32x4*)(p + at + 4) = f32x4{v[4], v[5], v[6], v[7]};
  };
  auto put8h = [&](_Float16* hi_p, _Float16* lo_p, int64_t at, const float* v) KF_INLINE {
    half8 hi, lo;
    split_n<_Float16, 8>(v, hi, lo);
    *(half8*)(hi_p + at) = hi;
    if (lo_p) *(half8*)(lo_p + at) = lo;
  };
  // (mean, M2) of this wavefront's 16-column tiles of s, per row
  auto stats_out = [&]() KF_INLINE {
    float2 t[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) {
        const f32x4 v = s.v[i][j];
        const float mu = row_sum((v[0] + v[1]) + (v[2] + v[3])) * (1.0f / 16.0f);
        float q = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) q = __builtin_fmaf(v[e] - mu, v[e] - mu, q);
        t[i][j] = make_float2(mu, row_sum(q));
      }
    if (grp == 0) {
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) red[wave * FN + i][16 * j + r] = t[i][j];
    }
  };
  // (mean, 1 / std) of this lane's rows. The lanes of a row all need them: each column group
  // works out its share of the FM rows and the groups exchange the results.
  auto stats_in = [&](float eps, float (&mean)[FM], float (&rstd)[FM]) KF_INLINE {
    constexpr int OWN = FM > 4 ? FM / 4 : 1, GRPS = FM / OWN;   // rows per group, groups used
    static_assert(GRPS == 1 || GRPS == 2 || GRPS == 4, "rows over the four column groups");
    float om[OWN], os[OWN];
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const int j = (grp % GRPS) * OWN + o;
      float2 t[CT];
      float sum = 0.0f;
#pragma unroll
      for (int n = 0; n < CT; ++n) { t[n] = red[n][16 * j + r]; sum += t[n].x; }
      om[o] = sum * (1.0f / CT);
      float m2 = 0.0f;
#pragma unroll
      for (int n = 0; n < CT; ++n) {
        const float dm = t[n].x - om[o];
        m2 += __builtin_fmaf(16.0f * dm, dm, t[n].y);
      }
      os[o] = 1.0f / sqrtf(__builtin_fmaf(m2, 1.0f / D, eps));
    }
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      if constexpr (GRPS == 1) { mean[j] = om[j]; rstd[j] = os[j]; }
      else {
        mean[j] = __shfl(om[j % OWN], 16 * (j / OWN) + r);
        rstd[j] = __shfl(os[j % OWN], 16 * (j / OWN) + r);
      }
    }
  };
  // planes of four values into an LDS operand tile
  auto put4 = [&](_Float16 (*a)[BM * LDA], int row, int col, const float* v, bool two) KF_INLINE {
    half4 hi, lo;
    split_n<_Float16, 4>(v, hi, lo);
    *(half4*)&a[0][row * LDA + col] = hi;
    if (two) *(half4*)&a[1][row * LDA + col] = lo;
  };
  // normalised rows: h planes into xa
  auto norm_to_lds = [&](int which, float eps, bool two) KF_INLINE {
    float mean[FM], rstd[FM];
    stats_in(eps, mean, rstd);
#pragma unroll
    for (int j = 0; j < FM; ++j) {
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        const f32x4 gv = param(which, i), bv = param(which + 1, i);
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[e] = __builtin_fmaf((s.v[i][j][e] - mean[j]) * rstd[j], gv[e], bv[e]);
        put4(xa, 16 * j + r, col0 + 16 * i + 4 * grp, v, two);
      }
    }
  };
  // s = (s + (product + bias)) * keep
  auto add_rows = [&](const Acc& c, int which) KF_INLINE {
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const f32x4 bv = param(which, i);
#pragma unroll
      for (int j = 0; j < FM; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          s.v[i][j][e] = (s.v[i][j][e] + (c.v[i][j][e] + bv[e])) * kv[j];
    }
  };

  if constexpr (TAIL) {
    Acc acc, out;
    product(out, xa, 0, g.m_out, Yes{}, No{});
    add_rows(out, 0);
    stats_out();
    lds_barrier();                               // also: every read of ctx is done
    norm_to_lds(1, g.eps2, UNI || mode_planes_a(g.m_f1) == 2);
    lds_barrier();
    zero(out);
    const bool two_h = UNI || mode_planes_a(g.m_f2) == 2;
    for (int c = 0; c < nc; ++c) {
      f32x4 b1[FN];                              // ahead of the product's weight loads
#pragma unroll
      for (int i = 0; i < FN; ++i)
        b1[i] = *(const f32x4*)(g.b1 + min(c * D + col0 + 16 * i + 4 * grp, g.F - 4));
      product(acc, xa, 1 + 2 * c, g.m_f1, Yes{}, No{});
      if (c > 0) lds_barrier();                  // the previous chunk's reads of hid are done
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        const bool in = c * D + col0 + 16 * i < g.F;       // F % 32 == 0: a tile is in or out
#pragma unroll
        for (int j = 0; j < FM; ++j) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = in ? gelu_erf(acc.v[i][j][e] + b1[i][e]) : 0.0f;
          put4(hid, 16 * j + r, col0 + 16 * i + 4 * grp, v, two_h);
        }
      }
      lds_barrier();
      product(out, hid, 2 + 2 * c, g.m_f2, No{}, No{});
    }
    add_rows(out, 3);
  } else {
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) s.v[i][j][e] *= kv[j];
  }

  if (g.s_out) {
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = m0 + 16 * j + r;
      if constexpr (FN == 2) {
        float v[8];
        trade(s.v[0][j], s.v[1][j], v);
        if (m < g.M) put8(g.s_out, (int64_t)m * D + col0 + pair8, v);
      } else if (m < g.M) {
#pragma unroll
        for (int i = 0; i < FN; ++i)
          *(f32x4*)(g.s_out + (int64_t)m * D + col0 + 16 * i + 4 * grp) = s.v[i][j];
      }
    }
  }
  stats_out();
  lds_barrier();
  if constexpr (!QKV) {
    float mean[FM], rstd[FM];
    stats_in(g.epsn, mean, rstd);
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = m0 + 16 * j + r;
      f32x4 o[FN];
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        const f32x4 gv = param(kOwn, i), bv = param(kOwn + 1, i);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[i][e] = __builtin_fmaf((s.v[i][j][e] - mean[j]) * rstd[j], gv[e], bv[e]) * kv[j];
      }
      if constexpr (FN == 2) {
        float v[8];
        trade(o[0], o[1], v);
        if (m < g.M) {
          const int64_t at = (int64_t)m * D + col0 + pair8;
          if (g.y_dtype == KF_F32) put8((float*)g.y, at, v);
          else {
            store4_any(g.y, nullptr, g.y_dtype, at, v);
            store4_any(g.y, nullptr, g.y_dtype, at + 4, v + 4);
          }
        }
      } else if (m < g.M) {
#pragma unroll
        for (int i = 0; i < FN; ++i) {
          const float v[4] = {o[i][0], o[i][1], o[i][2], o[i][3]};
          store4_any(g.y, nullptr, g.y_dtype, (int64_t)m * D + col0 + 16 * i + 4 * grp, v);
        }
      }
    }
  } else {
    norm_to_lds(kOwn, g.epsn, UNI || mode_planes_a(g.m_attn) == 2);
    lds_barrier();
    const bool k_two = g.k_lo != nullptr;
    Acc acc;
    // q, k and v read the same rows: where their fragments are more than the registers
    // hold, the compiler is kept from carrying them over (it spilled up to 256 bytes a lane)
    auto reread = [&]() KF_INLINE {
      if constexpr (FM * C::KS > 8) asm volatile("" ::: "memory");
    };
    // q: fp32, token-major
    product(acc, xa, p_qkv, g.m_attn, Yes{}, No{});
    auto add_bias = [&](int which) KF_INLINE {
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        const f32x4 bv = param(which, i);
#pragma unroll
        for (int j = 0; j < FM; ++j) acc.v[i][j] += bv;
      }
    };
    add_bias(kOwn + 2);
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = m0 + 16 * j + r;
      if constexpr (FN == 2) {
        float v[8];
        trade(acc.v[0][j], acc.v[1][j], v);
        if (m < g.M) put8(g.q_out, (int64_t)m * D + col0 + pair8, v);
      } else if (m < g.M) {
#pragma unroll
        for (int i = 0; i < FN; ++i)
          *(f32x4*)(g.q_out + (int64_t)m * D + col0 + 16 * i + 4 * grp) = acc.v[i][j];
      }
    }
    // k: planes, token-major
    reread();
    product(acc, xa, p_qkv + 1, g.m_attn, Yes{}, No{});
    add_bias(kOwn + 3);
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = m0 + 16 * j + r;
      if constexpr (FN == 2) {
        float v[8];
        trade(acc.v[0][j], acc.v[1][j], v);
        if (m < g.M) put8h(g.k_hi, g.k_lo, (int64_t)m * D + col0 + pair8, v);
      } else {
#pragma unroll
        for (int i = 0; i < FN; ++i) {
          const int64_t at = (int64_t)m * D + col0 + 16 * i + 4 * grp;
          const float v[4] = {acc.v[i][j][0], acc.v[i][j][1], acc.v[i][j][2], acc.v[i][j][3]};
          half4 hi, lo;
          split_n<_Float16, 4>(v, hi, lo);
          if (m < g.M) {
            *(half4*)(g.k_hi + at) = hi;
            if (k_two) *(half4*)(g.k_lo + at) = lo;
          }
        }
      }
    }
    // v^T [B, d, sp]: the operands swapped, so a lane holds tokens 4 grp .. 4 grp + 3 of
    // column r; the lane that has a sequence's last token also zeroes the pad [S, roundup(S, 8))
    reread();
    product(acc, xa, p_qkv + 2, g.m_attn, Yes{}, Yes{});
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const int n = col0 + 16 * i + r;
      const float bv = par[(kOwn + 4) * D + n];
      _Float16* vh = g.vt_hi + (int64_t)n * g.sp;
      _Float16* vl = k_two ? g.vt_lo + (int64_t)n * g.sp : nullptr;
      if constexpr (FM % 2 == 0) {
        if (g.S % 8 == 0) {                      // eight tokens are of one sequence; no padding
#pragma unroll
          for (int j = 0; j < FM; j += 2) {
            float v[8];
            trade(acc.v[i][j], acc.v[i][j + 1], v);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += bv;
            const int m = m0 + 16 * j + pair8;
            if (m < g.M) {
              const int b = m / g.S, t = m - b * g.S;
              put8h(vh, vl, (int64_t)b * D * g.sp + t, v);
            }
          }
          continue;
        }
      }
#pragma unroll
      for (int j = 0; j < FM; ++j) {
        const int m = m0 + 16 * j + 4 * grp;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc.v[i][j][e] + bv;
        half4 hi, lo;
        split_n<_Float16, 4>(v, hi, lo);
        int b = m / g.S, t = m - b * g.S;
        const int64_t row = (int64_t)D * g.sp;
        if (g.S % 4 == 0) {                      // the four tokens are of one sequence
          if (m < g.M) {
            const int64_t at = b * row + t;
            *(half4*)(vh + at) = hi;
            if (k_two) *(half4*)(vl + at) = lo;
            if (t + 4 == g.S && (g.S & 4)) {     // one quad of padding to a multiple of 8
              *(half4*)(vh + at + 4) = half4{0, 0, 0, 0};
              if (k_two) *(half4*)(vl + at + 4) = half4{0, 0, 0, 0};
            }
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (m + e < g.M) {
              const int64_t at = b * row + t;
              vh[at] = hi[e];
              if (k_two) vl[at] = lo[e];
            }
            if (++t == g.S) {
              if (m + e < g.M)
                for (int64_t x = g.S; x < ((g.S + 7) & ~7); ++x) {
                  vh[b * row + x] = (_Float16)0.0f;
                  if (k_two) vl[b * row + x] = (_Float16)0.0f;
                }
              t = 0;
              ++b;
            }
          }
        }
      }
    }
  }
}

// row-major [N, K] 16-bit values -> fragment order (kf950.h): one 16-byte piece per thread
__global__ __launch_bounds__(256) void fragments_kernel(const U4* src, U4* dst, int K, int64_t n) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= n) return;
  const int lane = q & 63, kt = (int)((q >> 6) % (K / 32));
  const int64_t nt = (q >> 6) / (K / 32);
  dst[q] = src[((nt * 16 + (lane & 15)) * K + kt * 32 + (lane >> 4) * 8) / 8];
}

template <class C, bool UNI>
static void launch_layer(const LayerArgs& a, int role, hipStream_t st) {
  const dim3 blocks((unsigned)((a.M + C::BM - 1) / C::BM)), threads(C::NT);
  switch (role) {
    case LAYER_TAIL: hipLaunchKernelGGL((layer_kernel<C, LAYER_TAIL, UNI>), blocks, threads, 0, st, a); break;
    case LAYER_QKV: hipLaunchKernelGGL((layer_kernel<C, LAYER_QKV, UNI>), blocks, threads, 0, st, a); break;
    default: hipLaunchKernelGGL((layer_kernel<C, LAYER_TAIL | LAYER_QKV, UNI>), blocks, threads, 0, st, a); break;
  }
}

template <class C>
static void launch_role(const LayerArgs& a, int role, bool uni, hipStream_t st) {
  if (uni) launch_layer<C, true>(a, role, st);
  else launch_layer<C, false>(a, role, st);
}

// Rows per block. Few rows a block while the grid does not fill the chip (the chain of
// products of one block is the launch time), more where it does (a block reads every weight
// once). Measured on MI355X, tail + QKV, f16x3, F = d, 16 / 32 / 64 rows: d 128 M 8192 15.4 / 13.3
// / 20.2 us, M 65536 103 / 74 / 62; d 256 M 8192 45 / 31 / 43, M 65536 389 / 259 / 218; d 64
// (F 256) M 8192 10.6 / 11.3, M 65536 52 / 40; d 32 M 8192 5.5 / 6.1, M 65536 14.5 / 13.4. The
// 64-row block gives a wavefront two column tiles (half the LDS reads per product; 4 wavefronts
// a block at d 128) and needs the registers of the single-mode kernel: with stage modes read
// at run time it spills, and widths up to 64 gain nothing from it, so those keep 32.
template <int D>
static void launch_d(const LayerArgs& a, int role, int rows, bool uni, hipStream_t st) {
  const int64_t cus = cu_count();
  if (rows == 0) rows = a.M <= (D <= 64 ? 32 : 16) * cus ? 16 : a.M < 128 * cus ? 32 : 64;
  if constexpr (D > 64) {
    if (rows == 64 && uni) return launch_layer<LayerCfg<D, 64, 2>, true>(a, role, st);
  }
  if (rows >= 32) launch_role<LayerCfg<D, 32, 1>>(a, role, uni, st);
  else launch_role<LayerCfg<D, 16, 1>>(a, role, uni, st);
}

static inline bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }
static bool mode_ok(int m) { return m == KF_MMA_F16 || m == KF_MMA_F16X2 || m == KF_MMA_F16X3; }
// a stage's operands: 16-byte aligned weight planes (lo where the mode has one) and bias
static bool stage_ok(int m, const void* hi, const void* lo, const void* bias) {
  return mode_ok(m) && hi && bias && al16(hi) && al16(bias) && (m == KF_MMA_F16 || (lo && al16(lo)));
}

}  // namespace kf

using namespace kf;

extern "C" int kf_fragments(const void* src, void* dst, int64_t N, int64_t K, void* stream) {
  if (!src || !dst || N < 0 || K <= 0) { kf_set_error("kf_fragments: bad arguments"); return KF_EINVAL; }
  if (N % 16 || K % 32 || !al16(src) || !al16(dst) || N > (1 << 24) || K > (1 << 24)) {
    kf_set_error("kf_fragments: needs N %% 16 == 0, K %% 32 == 0 and 16-byte aligned planes "
                 "(N=%lld K=%lld)", (long long)N, (long long)K);
    return KF_EUNSUPPORTED;
  }
  const int64_t n = N * K / 8, blocks = (n + 255) / 256;
  if (blocks > 0x7fffffffLL) { kf_set_error("kf_fragments: too large"); return KF_EUNSUPPORTED; }
  if (n == 0) return KF_OK;
  hipLaunchKernelGGL(fragments_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     (const U4*)src, (U4*)dst, (int)K, n);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { kf_set_error("kf_fragments: launch failed: %s", hipGetErrorString(e)); return KF_ELAUNCH; }
  return KF_OK;
}

extern "C" int kf_layer_block(const kf_layer_args* p, void* stream) {
  if (!p || p->M < 0 || p->d <= 0 || !p->res || !p->norm_w || !p->norm_b ||
      !(p->flags & (KF_LAYER_TAIL | KF_LAYER_QKV)) || (p->flags & ~(KF_LAYER_TAIL | KF_LAYER_QKV))) {
    kf_set_error("kf_layer_block: bad arguments");
    return KF_EINVAL;
  }
  const bool tail = p->flags & KF_LAYER_TAIL, qkv = p->flags & KF_LAYER_QKV;
  const int64_t d = p->d;
  if (d != 32 && d != 64 && d != 96 && d != 128 && d != 192 && d != 256) {
    kf_set_error("kf_layer_block: unsupported width %lld (32, 64, 96, 128, 192, 256)", (long long)d);
    return KF_EUNSUPPORTED;
  }
  if (p->M > (1LL << 30) || p->ld_res < d || p->ld_res % 4 || !al16(p->res) || !al16(p->norm_w) ||
      !al16(p->norm_b) || (p->s_out && !al16(p->s_out)) || (p->rows && p->rows != 16 && p->rows != 32 && p->rows != 64)) {
    kf_set_error("kf_layer_block: unsupported shape/alignment (M=%lld ld_res=%lld rows=%d)",
                 (long long)p->M, (long long)p->ld_res, p->rows);
    return KF_EUNSUPPORTED;
  }
  LayerArgs a{};
  a.res = p->res; a.ld_res = p->ld_res; a.keep = p->keep;
  a.gn = p->norm_w; a.bn = p->norm_b; a.epsn = p->norm_eps;
  a.s_out = p->s_out; a.M = (int)p->M;
  bool uni = true;
  if (tail) {
    if (!p->ctx_hi || !p->norm2_w || !p->norm2_b || p->F <= 0 ||
        (p->out_mode == KF_MMA_F16X3 && !p->ctx_lo)) {
      kf_set_error("kf_layer_block: bad arguments (tail)");
      return KF_EINVAL;
    }
    if (p->F % 32 || p->F > (1 << 20) || !al16(p->ctx_hi) || (p->ctx_lo && !al16(p->ctx_lo)) || !al16(p->norm2_w) ||
        !al16(p->norm2_b) || !stage_ok(p->out_mode, p->wo_hi, p->wo_lo, p->bo) ||
        !stage_ok(p->f1_mode, p->w1_hi, p->w1_lo, p->b1) ||
        !stage_ok(p->f2_mode, p->w2_hi, p->w2_lo, p->b2)) {
      kf_set_error("kf_layer_block: unsupported tail operands (F=%lld modes %d/%d/%d)",
                   (long long)p->F, p->out_mode, p->f1_mode, p->f2_mode);
      return KF_EUNSUPPORTED;
    }
    a.ctx_hi = (const _Float16*)p->ctx_hi; a.ctx_lo = (const _Float16*)p->ctx_lo;
    a.wo_hi = (const _Float16*)p->wo_hi; a.bo = p->bo; a.m_out = p->out_mode;
    a.w1_hi = (const _Float16*)p->w1_hi; a.b1 = p->b1; a.m_f1 = p->f1_mode;
    a.w2_hi = (const _Float16*)p->w2_hi; a.b2 = p->b2; a.m_f2 = p->f2_mode;
    a.wo_lo = p->out_mode == KF_MMA_F16 ? nullptr : (const _Float16*)p->wo_lo;
    a.w1_lo = p->f1_mode == KF_MMA_F16 ? nullptr : (const _Float16*)p->w1_lo;
    a.w2_lo = p->f2_mode == KF_MMA_F16 ? nullptr : (const _Float16*)p->w2_lo;
    a.g2 = p->norm2_w; a.b2n = p->norm2_b; a.eps2 = p->norm2_eps;
    a.F = (int)p->F;
    uni = p->out_mode == KF_MMA_F16X3 && p->f1_mode == KF_MMA_F16X3 && p->f2_mode == KF_MMA_F16X3;
  }
  if (qkv) {
    if (!p->q_out || !p->k_hi || !p->vt_hi || p->S <= 0 || p->H <= 0 || p->hd <= 0 ||
        p->H * p->hd != d || p->M % p->S || p->sp < p->S || p->sp % 8 || (!p->k_lo != !p->vt_lo) ||
        (p->attn_mode == KF_MMA_F16X2 && !p->k_lo) || (p->attn_mode == KF_MMA_F16 && p->k_lo)) {
      kf_set_error("kf_layer_block: bad arguments (qkv)");
      return KF_EINVAL;
    }
    if (!stage_ok(p->attn_mode, p->wqkv_hi, p->wqkv_lo, p->bqkv) || !al16(p->q_out) ||
        !al16(p->k_hi) || !al16(p->vt_hi) || (p->k_lo && (!al16(p->k_lo) || !al16(p->vt_lo)))) {
      kf_set_error("kf_layer_block: unsupported qkv operands (mode %d)", p->attn_mode);
      return KF_EUNSUPPORTED;
    }
    a.wq_hi = (const _Float16*)p->wqkv_hi; a.bq = p->bqkv; a.m_attn = p->attn_mode;
    a.wq_lo = p->attn_mode == KF_MMA_F16 ? nullptr : (const _Float16*)p->wqkv_lo;
    a.q_out = p->q_out; a.k_hi = (_Float16*)p->k_hi; a.k_lo = (_Float16*)p->k_lo;
    a.vt_hi = (_Float16*)p->vt_hi; a.vt_lo = (_Float16*)p->vt_lo;
    a.sp = p->sp; a.S = (int)p->S;
    uni = uni && p->attn_mode == KF_MMA_F16X3;
  } else {
    if (!p->y || p->y_dtype < KF_F32 || p->y_dtype > KF_BF16 || !al16(p->y)) {
      kf_set_error("kf_layer_block: bad output");
      return KF_EINVAL;
    }
    a.y = p->y; a.y_dtype = p->y_dtype;
  }
  if (p->M == 0) return KF_OK;
  const int role = (tail ? LAYER_TAIL : 0) | (qkv ? LAYER_QKV : 0);
  hipStream_t st = (hipStream_t)stream;
  switch (d) {
    case 32: launch_d<32>(a, role, p->rows, uni, st); break;
    case 64: launch_d<64>(a, role, p->rows, uni, st); break;
    case 96: launch_d<96>(a, role, p->rows, uni, st); break;
    case 128: launch_d<128>(a, role, p->rows, uni, st); break;
    case 192: launch_d<192>(a, role, p->rows, uni, st); break;
    default: launch_d<256>(a, role, p->rows, uni, st); break;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { kf_set_error("kf_layer_block: launch failed: %s", hipGetErrorString(e)); return KF_ELAUNCH; }
  return KF_OK;
}

// carekv_eval prefill correction (CAREKVLayer._apply_sparse_prefill_correction_eval,
// layer.py:363-456) on v_mfma_f32_16x16x32_f16.  Per (row t, query head):
// the base weights a_j = half(softmax(q.K_hat_j / sqrt(D))), j <= t, the V and
// K scores from a_j, ||r_v,j||, q.r_k,j and ||V_hat_j - o|| (r_k = half(K - K_hat),
// r_v = half(V - V_hat), layer.py:770-775), the top-k tokens of the kind's
// score, and o + sum a r_v + k_corr sum a clamp(q.r_k) (V_hat - o) over them.
//
// One work-group of 16 waves takes NC consecutive rows of one head, the MFMA's
// columns.  The row products q.K_hat, q.r_k and V_hat.o and the weighted sums
// are contractions, so each 16-token tile of K, K_hat, V, V_hat is read once
// per pass for all of the rows instead of once per row, and the rows' scores
// stay in LDS (NC rows of T floats):
//   1. x = q.K_hat / sqrt(D), the rows' softmax maxima and sums;
//   2. the scores, into LDS (with normalize first a pass for their means);
//   3. the k-th largest score of each row, a row per wave with the row's
//      scores in registers: a search over the (non-negative) float bits that
//      ends as soon as exactly k scores lie above the bound; ties at the k-th
//      value go to the lower tokens.  The selection is one bit per token;
//   4. the weighted sums over all tokens with the weights of unselected ones
//      zero: at the usual few percent read, 8 MFMA per 32 tokens of 16 rows
//      cost less than gathering each row's own tokens.
// Two work-groups cannot share a CU (the scores of 16 rows of 2048 tokens are
// 131 KB of its 160 KB LDS), hence 16 waves.  Measured on a 2048-token prompt
// of 32 query / 4 kv heads, D = 64, ratio 0.05: 539 us, against 5324 us for one
// work-group per (row, head) with scalar products, which read each row's tokens
// from L2 twice (D = 128, 8 kv heads, 1024 tokens: 305 us, 1720 before).  Of the
// 539 us (builds that end after a step) launching and filling the CUs takes at
// most 20, step 1 56, step 2 147, step 3 158, step 4 127 and the output 31; steps
// 1, 2 and 4 are bound by the loads' and lane exchanges' latency (four waves per
// SIMD), step 3 by its compares.  At D = 128 the 128 VGPRs of a 16-wave
// work-group do not hold step 4's tiles: 12 of the 646 instructions of its loop
// are scratch accesses.  A prompt of 64 tokens takes one wave's latency through
// the four steps, 19 us at D = 128 (21 with normalize), 28 for the scalar form.
//
// Every sum over a row's tokens is taken in an order that depends on the token
// indices alone (tiles dealt to the 16 waves), and infinities and NaN in tokens
// that a row does not read are kept out of its sums, so a row's result does not
// change with NC, the batch or the prompt's length after the row.
#include <cmath>

#include "decode_page.h"
#include "host_util.h"

namespace carekv {

constexpr int kEvalMaxT = 8192;
constexpr int kEvalWaves = 16;

struct EvalArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const uint16_t* kh;
  const uint16_t* vh;
  const uint16_t* o;
  uint16_t* out;
  int32_t* diag;
  int B, Hq, Hkv, T, diag_cap, min_res, kind, v_norm, normalize;
  double ratio;
  float k_corr, inv_sqrt_d, sqrt_d, rcp_sqrt_d;
};

// Rows a work-group takes at a prompt length: as many of the MFMA's 16 columns
// as the CU's LDS holds score rows for (16 rows of 2304 tokens: 158 KB with the
// kernel's own arrays).  A half or a quarter of the columns costs its share of
// the matrix and VALU work: 8 heads of 4000 tokens 1.13 ms, 4 heads of 8000
// 3.19 ms at D = 64.
__host__ __device__ constexpr int eval_rows(int T) { return T <= 2304 ? 16 : T <= 4608 ? 8 : 4; }
// 512-token chunks a wave of a row's 16 / NC waves holds in registers.
__host__ __device__ constexpr int eval_chunks(int NC) { return NC == 4 ? 4 : 5; }
__host__ __device__ constexpr int eval_stride(int T) { return (T + 15) / 16 * 16 + 4; }
// the scores; then the V tiles of step 4; then the waves' partial sums
constexpr size_t eval_lds(int D, int NC, int T) {
  const size_t sc = (size_t)NC * eval_stride(T) * 4, st = (size_t)kEvalWaves * 32 * (2 * D + 32),
               rd = (size_t)kEvalWaves * D * 17 * 4;
  return sc > st ? (sc > rd ? sc : rd) : (st > rd ? st : rd);
}

// x / d with r = 1 / d: one Newton step on the quotient, within an ulp of the
// division.
__device__ __forceinline__ float div_r(float x, float d, float r) {
  const float q = x * r;
  return fmaf(fmaf(-d, q, x), r, q);
}
// x - y in fp16, rounded once, as one packed FMA per pair: the -1 passes
// through an empty asm, since the subtraction itself (which the compiler makes
// of a visible -1) takes three operations per pair.
__device__ __forceinline__ half8_t minus(const half8_t& x, const half8_t& y) {
  uint32_t m = 0xbc00bc00u;
  asm("" : "+s"(m));
  half2_t neg;
  __builtin_memcpy(&neg, &m, 4);
  half8_t r;
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const half2_t d = __builtin_elementwise_fma(half2_t{y[i], y[i + 1]}, neg, half2_t{x[i], x[i + 1]});
    r[i] = d[0];
    r[i + 1] = d[1];
  }
  return r;
}
// Its infinite and NaN elements as zero.
__device__ __forceinline__ half8_t finite_part(const half8_t& x) {
  half8_t r;
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = __builtin_fabsf16(x[i]) < (_Float16)INFINITY ? x[i] : (_Float16)0.f;
  return r;
}
// s / sqrt(D): exact for D = 64; an infinite score stays infinite.
template <int D>
__device__ __forceinline__ float score_of(float s, const EvalArgs& a) {
  if constexpr (D == 64) return s * 0.125f;
  return fabsf(s) < INFINITY ? div_r(s, a.sqrt_d, a.rcp_sqrt_d) : s;
}
// exp(x) for x <= 0 within 2 ulp: x log2(e) as an unevaluated sum of two floats
// (Dekker's product with the FMA's exact remainder, log2(e) itself in two
// floats), the low one applied to the base-2 exponential to first order.
// Below -104, and for NaN, the value at -104 (0 as a weight in fp16; a NaN
// score reaches the row through its sum).
__device__ __forceinline__ float exp_neg(float x) {
  x = fmaxf(x, -104.f);
  const float ph = x * 1.44269502f;
  const float pl = fmaf(x, 1.92596303e-8f, fmaf(x, 1.44269502f, -ph));
  const float e = __builtin_amdgcn_exp2f(ph);
  return fmaf(e, pl * 0.693147182f, e);
}
// The sum and the union of bits over the wave.
__device__ __forceinline__ int wave_isum(int v) {
  v += row_ror_i<8>(v);
  v += row_ror_i<4>(v);
  v += row_ror_i<2>(v);
  v += row_ror_i<1>(v);
  const auto p = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
  v = (int)(p[0] + p[1]);
  const auto r = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
  return __builtin_amdgcn_readfirstlane((int)(r[0] + r[1]));
}
__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
  v |= (uint32_t)row_ror_i<8>((int)v);
  v |= (uint32_t)row_ror_i<4>((int)v);
  v |= (uint32_t)row_ror_i<2>((int)v);
  v |= (uint32_t)row_ror_i<1>((int)v);
  const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = p[0] | p[1];
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)(r[0] | r[1]));
}

template <int D, int NC>
__global__ __launch_bounds__(64 * kEvalWaves) void prefill_eval_kernel(EvalArgs a) {
  constexpr int KS = D / 32;           // 32-dim steps of a product
  constexpr int DT = D / 16;           // 16-dim output tiles
  constexpr int NW = kEvalWaves;
  constexpr int WPC = NW / NC;         // waves per row in step 3
  constexpr int CPP = eval_chunks(NC); // 512-token chunks per wave there
  constexpr int MW = 8 * CPP * WPC;    // 64-token words of a row's selection
  constexpr int VRS = 2 * D + 32;      // staged V row stride, bytes
  // An expanded distance's terms are at most this multiple of its square (an error
  // of 2^-24 of the terms is 2^-23 of the distance; the scores' dot products
  // lose more).  Rows whose selection differs from 64-bit scores, of 500 000 rows:
  // 4, against 6 for the differences alone and 8 with a multiple of 32.
  constexpr float kCancel = 4.f;
  typedef short short4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) short4_t lds_short4;
  typedef __attribute__((address_space(3))) char lds_char;
  extern __shared__ __align__(16) char dyn[];
  __shared__ uint64_t s_sel[NC][MW];
  __shared__ float s_wmax[NW][16], s_wsum[NW][16], s_sum[2][NW][16], s_w[NW][16];
  __shared__ __align__(16) float s_mx[16], s_den[16], s_oo[16], s_mean[2][16];
  __shared__ int s_cnt[2][NW];
  float* const sc = reinterpret_cast<float*>(dyn);

  // the latest (longest) rows first; consecutive heads, which share a kv head,
  // on one XCD (work-groups go to the 8 XCDs in turn)
  const int nhb = a.Hq * a.B;
  int hb = (int)blockIdx.x % nhb;
  if (nhb % 8 == 0) hb = hb % 8 * (nhb / 8) + hb / 8;
  const int nblk = (a.T + NC - 1) / NC;
  const int t0 = (nblk - 1 - (int)blockIdx.x / nhb) * NC;
  const int h = hb % a.Hq, b = hb / a.Hq, hk = h / (a.Hq / a.Hkv);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  const int T = a.T, nmax = min(t0 + NC, T), ntile = (nmax + 15) / 16;
  const int stride = eval_stride(T);
  const uint32_t span = (uint32_t)T * D * 2;
  const long qbase = ((long)b * a.Hq + h) * T * D, kvbase = ((long)b * a.Hkv + hk) * T * D;
  const __amdgpu_buffer_rsrc_t rq = make_rsrc(a.q + qbase, span), ro = make_rsrc(a.o + qbase, span);
  const __amdgpu_buffer_rsrc_t rk = make_rsrc(a.k + kvbase, span), rkh = make_rsrc(a.kh + kvbase, span);
  const __amdgpu_buffer_rsrc_t rv = make_rsrc(a.v + kvbase, span), rvh = make_rsrc(a.vh + kvbase, span);

  // 16 rows of a matrix as an MFMA operand: lane (row c16, dims 32 ks + 8 g ..);
  // rows past the prompt read as zero.  Four consecutive lanes load 64
  // consecutive bytes of a row and the lanes then trade places: loaded in the
  // operand's own order, every lane of a load is in another row's line and the
  // cache serves a line a cycle (the kernel took 775 us)
  const int from = (c16 * 4 + g) * 4;
  auto load_rows = [&](__amdgpu_buffer_rsrc_t r, int row0, half8_t (&x)[KS]) {
    const uint32_t off = ((uint32_t)(row0 + (lane >> 2)) * D + 8 * (lane & 3)) * 2;
    uint32_t v[KS][4];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const auto u = __builtin_amdgcn_raw_buffer_load_b128(r, off + 64 * ks, 0, 0);
      __builtin_memcpy(v[ks], &u, 16);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[ks][i] = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)v[ks][i]);
      __builtin_memcpy(&x[ks], v[ks], 16);
    }
  };

  // run body(tile, rows) over this wave's tiles of r, each loaded while the one before is used
  auto tiles = [&](__amdgpu_buffer_rsrc_t r, auto&& body) {
    half8_t x[KS], y[KS];
    int tile = w;
    if (tile < ntile) load_rows(r, 16 * tile, x);
    for (; tile < ntile; tile += 2 * NW) {
      load_rows(r, 16 * (tile + NW), y);
      body(tile, x);
      if (tile + NW >= ntile) break;
      load_rows(r, 16 * (tile + 2 * NW), x);
      body(tile + NW, y);
    }
  };
  // the fp16 base weight of a score q.K_hat (softmax in fp32, cast to fp16)
  auto weight = [&](float s, float mx, float den) {
    return (float)(_Float16)div_r(exp_neg(score_of<D>(s, a) - mx), den, __builtin_amdgcn_rcpf(den));
  };
  // ---- 1. the rows' softmax maxima and sums (with NC < 16, the rows past NC
  // are computed and dropped): each lane keeps its tokens' running maximum and
  // sum for row c16
  const int last = min(t0 + c16, T - 1);  // row c16's last token
  {
    half8_t qf[KS];
    load_rows(rq, t0, qf);
    float m = -INFINITY, l = 0.f;
    auto body = [&](int tile, const half8_t (&kh)[KS]) {
      float4_t s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = mfma16x32(kh[ks], qf[ks], s);
      const int tok = 16 * tile + 4 * g;
      float mn = m;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[i] = score_of<D>(s[i], a);
        if (tok + i <= last) mn = fmaxf(mn, s[i]);
      }
      if (__any(mn != m)) l *= m == mn ? 1.f : exp_neg(m - mn);
      m = mn;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (tok + i <= last) l += s[i] != s[i] ? s[i] : exp_neg(s[i] - m);
    };
    tiles(rkh, body);
    // the lanes of a row, then the waves
    const float mw = col_max(m);
    l *= m == mw ? 1.f : exp_neg(m - mw);
    l = col_sum(l);
    if (lane < 16) {
      s_wmax[w][lane] = mw;
      s_wsum[w][lane] = l;
    }
    if (w == 0) {
      half8_t of[KS];
      load_rows(ro, t0, of);
      float oo = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int i = 0; i < 8; ++i) oo = fmaf((float)of[ks][i], (float)of[ks][i], oo);
      oo = col_sum(oo);
      if (lane < 16) s_oo[lane] = oo;
    }
  }
  __syncthreads();
  if (tid < 16) {
    float m = -INFINITY, den = 0.f;
    for (int u = 0; u < NW; ++u) m = fmaxf(m, s_wmax[u][tid]);
    for (int u = 0; u < NW; ++u) den += s_wsum[u][tid] * exp_neg(s_wmax[u][tid] - m);
    s_mx[tid] = m;
    s_den[tid] = den;
  }
  __syncthreads();

  // ---- 2. the scores: lane (token c16, rows 4 g + i)
  // MODE 0 both, 1 k, 2 v, 3 both over their means, 4 the sums for the means
  auto scores = [&](auto mode) {
    constexpr int MODE = decltype(mode)::value;
    half8_t qf[KS], of[KS];
    if constexpr (D == 64) {
      load_rows(rq, t0, qf);
      load_rows(ro, t0, of);
    }
    float4_t vsum{0.f, 0.f, 0.f, 0.f}, ksum{0.f, 0.f, 0.f, 0.f};
    struct Rows {
      half8_t kh[KS], kk[KS], vh[KS], vv[KS];
    };
    auto load = [&](int tile, Rows& x) {
      load_rows(rkh, 16 * tile, x.kh);
      if constexpr (MODE != 2) load_rows(rk, 16 * tile, x.kk);
      load_rows(rvh, 16 * tile, x.vh);
      if constexpr (MODE != 1) load_rows(rv, 16 * tile, x.vv);
    };
    auto body = [&](int tile, const Rows& x) {
      if constexpr (D == 128) {  // (128 registers do not hold the rows' operands too)
        load_rows(rq, t0, qf);
        load_rows(ro, t0, of);
      }
      const float4_t oo = *reinterpret_cast<const float4_t*>(s_oo + 4 * g);
      float4_t s{0.f, 0.f, 0.f, 0.f}, qd = s, vo = s, v2 = s, r2 = s;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        s = mfma16x32(qf[ks], x.kh[ks], s);
        if constexpr (MODE != 2) qd = mfma16x32(qf[ks], minus(x.kk[ks], x.kh[ks]), qd);
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        vo = mfma16x32(of[ks], x.vh[ks], vo);
        v2 = mfma16x32(x.vh[ks], x.vh[ks], v2);
        if constexpr (MODE != 1) {
          const half8_t r = minus(x.vv[ks], x.vh[ks]);
          r2 = mfma16x32(r, r, r2);
        }
      }
      // the squared norms of token c16: the diagonals of V_hat V_hat^T and r_v r_v^T
      const float vv2 = diag16(v2, c16, g);
      float rvn = 0.f;
      if constexpr (MODE != 1) rvn = __builtin_amdgcn_sqrtf(diag16(r2, c16, g));
      const int tok = 16 * tile + c16;
      float vd2[4];
      uint32_t rows = 0;  // rows of the block with a token near their o
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        vd2[i] = fmaf(-2.f, vo[i], vv2 + oo[i]);
        const uint64_t b = __ballot(4 * g + i < NC && !(vd2[i] * kCancel >= vv2 + oo[i]));
#pragma unroll
        for (int u = 0; u < 4; ++u) rows |= (b >> (16 * u) & 0xffff) != 0 ? 1u << (4 * u + i) : 0u;
      }
      // V_hat_j close to o (a row whose weight sits on few tokens), or not
      // finite: the expansion cancels, so those pairs take the difference itself.
      // The operands hold both sides: lane (c16, g) has token c16's dims
      // 32 ks + 8 g .., and row r's come from lane (r, g).
#pragma unroll 1
      while (rows != 0) {
        const int r = __builtin_ctz(rows);
        rows &= rows - 1;
        float d2 = 0.f, one = 1.f;
        asm("" : "+s"(one));  // (a visible 1 becomes a subtraction and two conversions)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          uint32_t ow[4];
          __builtin_memcpy(ow, &of[ks], 16);
#pragma unroll
          for (int e = 0; e < 4; ++e) ow[e] = (uint32_t)__builtin_amdgcn_ds_bpermute((r + 16 * g) * 4, (int)ow[e]);
          half8_t o8;
          __builtin_memcpy(&o8, ow, 16);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float df = fmaf((float)x.vh[ks][e], one, -(float)o8[e]);
            d2 = fmaf(df, df, d2);
          }
        }
        d2 = col_sum(d2);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (r == 4 * g + i && !(vd2[i] * kCancel >= vv2 + oo[i])) vd2[i] = d2;
      }
      const float4_t mx = *reinterpret_cast<const float4_t*>(s_mx + 4 * g), den = *reinterpret_cast<const float4_t*>(s_den + 4 * g);
      float4_t vm, km;
      if constexpr (MODE == 3) {
        vm = *reinterpret_cast<const float4_t*>(s_mean[0] + 4 * g);
        km = *reinterpret_cast<const float4_t*>(s_mean[1] + 4 * g);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int cl = 4 * g + i;
        const float aw = weight(s[i], mx[i], den[i]);
        const float vdiff = __builtin_amdgcn_sqrtf(vd2[i]);
        float vs = 0.f, ks = 0.f;
        if constexpr (MODE != 1) vs = a.v_norm ? aw * rvn : aw * rvn * vdiff;
        if constexpr (MODE != 2) ks = aw * fabsf(qd[i] * a.inv_sqrt_d) * vdiff;
        if constexpr (MODE == 4) {
          if (tok <= t0 + cl) {
            vsum[i] += vs;
            ksum[i] += ks;
          }
        } else if (cl < NC) {
          float x;
          if constexpr (MODE == 0) x = vs + ks;
          if constexpr (MODE == 1) x = ks;
          if constexpr (MODE == 2) x = vs;
          if constexpr (MODE == 3) {
            // (over an infinite mean the rounded-off quotient itself: 0 for a
            // finite score, which the Newton step would make NaN)
            const float rv = __builtin_amdgcn_rcpf(vm[i]), rk = __builtin_amdgcn_rcpf(km[i]);
            x = (vm[i] < INFINITY ? div_r(vs, vm[i], rv) : vs * rv) + (km[i] < INFINITY ? div_r(ks, km[i], rk) : ks * rk);
          }
          sc[cl * stride + tok] = x;
        }
      }
    };
    // (loading a tile ahead needs registers that the 128 of a 16-wave
    // work-group do not have: 850-870 us against 773 us for the whole kernel)
    for (int tile = w; tile < ntile; tile += NW) {
      asm volatile("" ::: "memory");
      Rows x;
      load(tile, x);
      body(tile, x);
    }
    if constexpr (MODE == 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        vsum[i] = row16_sum(vsum[i]);
        ksum[i] = row16_sum(ksum[i]);
        if (c16 == 0) {
          s_sum[0][w][4 * g + i] = vsum[i];
          s_sum[1][w][4 * g + i] = ksum[i];
        }
      }
      __syncthreads();
      if (tid < 32) {
        const int cl = tid & 15;
        float x = 0.f;
        for (int u = 0; u < NW; ++u) x += s_sum[tid >> 4][u][cl];
        s_mean[tid >> 4][cl] = fmaxf(x / (float)(t0 + cl + 1), 1e-8f);
      }
      __syncthreads();
    }
  };
  using std::integral_constant;
  if (a.kind == 1) {
    scores(integral_constant<int, 1>{});
  } else if (a.kind == 2) {
    scores(integral_constant<int, 2>{});
  } else if (a.normalize) {
    scores(integral_constant<int, 4>{});
    scores(integral_constant<int, 3>{});
  } else {
    scores(integral_constant<int, 0>{});
  }
  __syncthreads();

  // ---- 3. the selection of row t0 + col (wave w takes its part `part`)
  const int col = w / WPC, part = w % WPC;
  const int n = t0 + col < T ? t0 + col + 1 : 0;  // tokens of the row
  // int(n * ratio) (layer.py:397); a ratio of 1 or more keeps all n, so the
  // conversion only ever sees values below n
  auto budget = [&](int nn) {
    const int K = a.ratio >= 1.0 ? nn : (int)((double)nn * a.ratio);
    return min(max(a.min_res, K), nn);
  };
  {
    const int K = budget(n), tok0 = 512 * part * CPP;
    uint32_t key[8 * CPP];
#pragma unroll
    for (int c = 0; c < CPP; ++c) {
#pragma unroll
      for (int r = 0; r < 8; ++r) key[8 * c + r] = 0u;
      if (tok0 + 512 * c < n) {
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const int tok = tok0 + 512 * c + 64 * r + lane;
          if (tok < n) key[8 * c + r] = __float_as_uint(sc[col * stride + tok]);
        }
      }
    }
    // sum of x over the row's waves (one barrier; two buffers in turn)
    int turn = 0;
    auto row_total = [&](int x) -> int {
      if constexpr (WPC == 1) return x;
      if (lane == 0) s_cnt[turn][w] = x;
      __syncthreads();
      int t = 0;
#pragma unroll
      for (int u = 0; u < WPC; ++u) t += s_cnt[turn][col * WPC + u];
      turn ^= 1;
      return __builtin_amdgcn_readfirstlane(t);
    };
    auto count_ge = [&](uint32_t cand) {
      int cnt = 0;
#pragma unroll
      for (int c = 0; c < CPP; ++c)
        if (tok0 + 512 * c < n) {
#pragma unroll
          for (int r = 0; r < 8; ++r) cnt += key[8 * c + r] >= cand;
        }
      return wave_isum(cnt);
    };
    uint32_t tau = 0u;
    bool cut = K == 0;  // exactly K keys are >= tau (K = 0: none is taken)
    int bit = 31;
    if constexpr (WPC == 1) {  // from the largest key's top bit (the scores of a short prompt's first rows are 0)
      uint32_t any = 0u;
#pragma unroll
      for (int k = 0; k < 8 * CPP; ++k) any |= key[k];
      bit = 31 - __builtin_clz(wave_or(any) | 1u);
    }
    for (; bit >= 0; --bit) {
      if (WPC == 1 && cut) break;  // a row of several waves passes every barrier
      const uint32_t cand = tau | (1u << bit);
      const int cnt = row_total(count_ge(cand));
      if (!cut && cnt >= K) {
        tau = cand;
        cut = cnt == K;
      }
    }
    // not cut: the keys above tau, and the lowest tokens at tau
    int eq_left = 0;
    if (WPC > 1 || !cut) {
      const int gt = tau == 0xffffffffu ? 0 : count_ge(tau + 1);
      int eq = 0;
#pragma unroll
      for (int c = 0; c < CPP; ++c)
#pragma unroll
        for (int r = 0; r < 8; ++r) eq += tok0 + 512 * c + 64 * r + lane < n && key[8 * c + r] == tau;
      eq = wave_isum(eq);
      eq_left = K - row_total(gt);
      if constexpr (WPC > 1) {
        if (lane == 0) s_cnt[turn][w] = eq;
        __syncthreads();
        for (int u = 0; u < part; ++u) eq_left -= s_cnt[turn][col * WPC + u];
        eq_left = __builtin_amdgcn_readfirstlane(eq_left);
      }
    }
    uint64_t mine = 0;
#pragma unroll
    for (int c = 0; c < CPP; ++c) {
      if (tok0 + 512 * c < n) {
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const bool ok = tok0 + 512 * c + 64 * r + lane < n;
          const uint32_t x = key[8 * c + r];
          uint64_t m;
          if (cut) {
            m = __ballot(ok && K > 0 && x >= tau);
          } else {
            m = __ballot(ok && x > tau);
            const uint64_t e = __ballot(ok && x == tau);
            if (e != 0 && eq_left > 0) {
              const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(e >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)e, 0));
              m |= __ballot(ok && x == tau && before < eq_left);
              eq_left -= __popcll(e);
            }
          }
          if (lane == 8 * c + r) mine = m;
        }
      }
    }
    if (lane < 8 * CPP) s_sel[col][part * 8 * CPP + lane] = mine;
  }
  __syncthreads();
  if (a.diag && w < NC && t0 + w < T) {  // the selected tokens in order
    int32_t* dg = a.diag + (((long)b * a.Hq + h) * T + t0 + w) * a.diag_cap;
    int pos = 0;
    for (int u = 0; 64 * u <= t0 + w; ++u) {
      const uint64_t m = s_sel[w][u];
      const int p = pos + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
      if ((m >> lane & 1) && p < a.diag_cap) dg[p] = 64 * u + lane;
      pos += __popcll(m);
    }
    for (int p = pos + lane; p < a.diag_cap; p += 64) dg[p] = -1;
  }

  // ---- 4. the corrections: lane (row c16, dims 16 dt + 4 g ..)
  float4_t av[DT], ak[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) av[dt] = ak[dt] = float4_t{0.f, 0.f, 0.f, 0.f};
  float wsum = 0.f;
  const int cc = c16 & (NC - 1);
  // scaled by 2^12 (|weight| <= 2), so that both halves of a small K weight
  // are normal fp16 values
  constexpr float kUp = 4096.f, kDown = 1.f / 4096.f;
  // the weights of tokens 32 p + 16 tt + 4 g + i: a (fp16) and a clamp(q.r_k)
  auto weights = [&](int p, float (&wa)[2][4], float (&wk)[2][4]) {
    const float mx = s_mx[c16], den = s_den[c16];
    const uint32_t bits = c16 < NC ? (uint32_t)(s_sel[cc][p >> 1] >> (32 * (p & 1))) >> (4 * g) : 0u;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      half8_t kh[KS], kk[KS], qf[KS];
      load_rows(rkh, 32 * p + 16 * tt, kh);
      load_rows(rk, 32 * p + 16 * tt, kk);
      load_rows(rq, t0, qf);
      float4_t s{0.f, 0.f, 0.f, 0.f}, qd{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        s = mfma16x32(kh[ks], qf[ks], s);
        qd = mfma16x32(minus(kk[ks], kh[ks]), qf[ks], qd);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool on = bits >> (16 * tt + i) & 1;
        const float aw = weight(s[i], mx, den);
        const float qc = fminf(fmaxf(qd[i] * a.inv_sqrt_d, -2.f), 2.f);
        wa[tt][i] = on ? aw : 0.f;
        wk[tt][i] = on ? aw * qc : 0.f;
      }
    }
  };
  const bool some = budget(nmax) > 0;  // the budget grows with the row
  if (some) {
    char* const vt = dyn + w * 32 * VRS;
    constexpr int NCH = 32 * D / 8 / 64;  // 16-byte chunks a lane stages
    // O^T += V^T P^T over the staged 32 tokens: source lane c16 of group g
    // reads row 4 g + c16 / 4 (and + 16), dims 16 dt + 4 (c16 % 4) ..
    const lds_char* vrow = (const lds_char*)vt + (4 * g + (c16 >> 2)) * VRS + (c16 & 3) * 8;
    auto v_operand = [&](int dt) {
      const short4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(vrow + 32 * dt));
      const short4_t v2 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(vrow + 16 * VRS + 32 * dt));
      half8_t x;
      __builtin_memcpy(&x, &v1, 8);
      __builtin_memcpy(reinterpret_cast<char*>(&x) + 8, &v2, 8);
      return x;
    };
    auto sums = [&](auto clean) {
      constexpr bool CLEAN = decltype(clean)::value;
      for (int p = w; 32 * p < nmax; p += NW) {
        auto load_chunk = [&](__amdgpu_buffer_rsrc_t r, int k) {
          half8_t x;
          const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (uint32_t)32 * p * D * 2 + (lane + 64 * k) * 16, 0, 0);
          __builtin_memcpy(&x, &v, 16);
          return x;
        };
        auto load_chunks = [&](__amdgpu_buffer_rsrc_t r, half8_t (&x)[NCH]) {
#pragma unroll
          for (int k = 0; k < NCH; ++k) x[k] = load_chunk(r, k);
        };
        auto chunk = [&](int k) {
          const int c = lane + 64 * k;
          return reinterpret_cast<half8_t*>(vt + c / (D / 8) * VRS + c % (D / 8) * 16);
        };
        half8_t xh[NCH], xv[NCH];
        if constexpr (D == 64 && !CLEAN) load_chunks(rvh, xh);
        float wa[2][4], wk[2][4];
        weights(p, wa, wk);
        half8_t pa, ph, pl;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          pa[j] = (_Float16)wa[j >> 2][j & 3];
          const float u = wk[j >> 2][j & 3] * kUp;
          ph[j] = (_Float16)u;
          pl[j] = (_Float16)(u - (float)ph[j]);
          if constexpr (!CLEAN) wsum += wk[j >> 2][j & 3];
        }
        if constexpr (D == 128 && !CLEAN) load_chunks(rvh, xh);
        lds_sync_wave();  // the last tile's reads
        if constexpr (CLEAN) {
#pragma unroll 1
          for (int k = 0; k < NCH; ++k) *chunk(k) = finite_part(load_chunk(rvh, k));
        } else {
#pragma unroll
          for (int k = 0; k < NCH; ++k) *chunk(k) = xh[k];
          load_chunks(rv, xv);
        }
        lds_sync_wave();
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const half8_t x = v_operand(dt);
          ak[dt] = mfma16x32(x, ph, ak[dt]);
          ak[dt] = mfma16x32(x, pl, ak[dt]);
        }
        if constexpr (CLEAN) {
          lds_sync_wave();
#pragma unroll 1
          for (int k = 0; k < NCH; ++k) *chunk(k) = finite_part(minus(load_chunk(rv, k), load_chunk(rvh, k)));
        } else {
#pragma unroll
          for (int k = 0; k < NCH; ++k) xv[k] = minus(xv[k], *chunk(k));  // r_v; the lane's own chunks of V_hat
          lds_sync_wave();
#pragma unroll
          for (int k = 0; k < NCH; ++k) *chunk(k) = xv[k];
        }
        lds_sync_wave();
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) av[dt] = mfma16x32(v_operand(dt), pa, av[dt]);
      }
    };
    sums(std::false_type{});
    bool bad = false;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bad |= !(fabsf(av[dt][i]) < INFINITY);
        bad |= !(fabsf(ak[dt][i]) < INFINITY);
      }
    if (__builtin_expect(__any(bad), 0)) {
      // An infinity or NaN in a token that a row does not read must not reach
      // it through a zero weight: the sums are taken again without such
      // elements, and the rows that read them add them afterwards.  The other
      // rows keep the bits that they have without those elements.
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) av[dt] = ak[dt] = float4_t{0.f, 0.f, 0.f, 0.f};
      sums(std::true_type{});
      for (int p = w; 32 * p < nmax; p += NW) {
        float wa[2][4], wk[2][4];
        weights(p, wa, wk);
        const uint32_t bits = c16 < NC ? (uint32_t)(s_sel[cc][p >> 1] >> (32 * (p & 1))) : 0u;
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll 1
          for (int gg = 0; gg < 4; ++gg) {
            const float xa = __shfl(wa[j >> 2][j & 3], 16 * gg + c16, 64), xk = __shfl(wk[j >> 2][j & 3], 16 * gg + c16, 64);
            const int tk = 16 * (j >> 2) + 4 * gg + (j & 3);
            if (!(bits >> tk & 1)) continue;
            const long row = kvbase + (long)(32 * p + tk) * D + 4 * g;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const _Float16 vhat = bits2half(a.vh[row + 16 * dt + i]);
                const float r = (float)(_Float16)(bits2half(a.v[row + 16 * dt + i]) - vhat), vf = (float)vhat;
                if (!(fabsf(r) < INFINITY)) av[dt][i] = fmaf(xa, r, av[dt][i]);
                if (!(fabsf(vf) < INFINITY)) ak[dt][i] = fmaf(xk * kUp, vf, ak[dt][i]);
              }
          }
      }
    }
    wsum = col_sum(wsum);
    if (lane < 16) s_w[w][lane] = wsum;
  }
  // ---- the waves' sums in wave order, and the output
  constexpr int NO = D * NC / (64 * NW) > 0 ? D * NC / (64 * NW) : 1;  // outputs a thread forms
  const int nact = min(NW, (nmax + 31) / 32);  // waves that had tokens; the others' sums are 0
  float tv[NO], tk[NO];
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    if (!some) {
#pragma unroll
      for (int k = 0; k < NO; ++k) tv[k] = tk[k] = 0.f;
      continue;
    }
    __syncthreads();
    if (w < nact) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          sc[(w * D + 16 * dt + 4 * g + i) * 17 + c16] = half ? ak[dt][i] : av[dt][i];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NO; ++k) {
      const int id = tid + 64 * NW * k, cl = id / D, d = id % D;
      float x = 0.f;
      if (cl < NC)
#pragma unroll 4
        for (int u = 0; u < nact; ++u) x += sc[(u * D + d) * 17 + cl];
      if (half) tk[k] = x * kDown;
      else tv[k] = x;
    }
  }
#pragma unroll
  for (int k = 0; k < NO; ++k) {
    const int id = tid + 64 * NW * k, cl = id / D, d = id % D;
    if (cl >= NC || t0 + cl >= T) continue;
    const long at = qbase + (long)(t0 + cl) * D + d;
    const float o = h2f(a.o[at]);
    float dk = 0.f;
    if (a.kind != 2 && some) {
      float ws = 0.f;
      for (int u = 0; u < nact; ++u) ws += s_w[u][cl];
      dk = fmaf(-ws, o, tk[k]);
    }
    const float dv = a.kind == 1 ? 0.f : tv[k];
    a.out[at] = f2h((o + dv) + a.k_corr * dk);
  }
}

}  // namespace carekv

using namespace carekv;

extern "C" int carekv_prefill_eval(const carekv_prefill_eval_params* p, const uint16_t* q, const uint16_t* k,
                                   const uint16_t* v, const uint16_t* k_hat, const uint16_t* v_hat,
                                   const uint16_t* o_base, uint16_t* out, int32_t* diag, void* stream) {
  CAREKV_REQUIRE(p && q && k && v && k_hat && v_hat && o_base && out, "null argument");
  CAREKV_REQUIRE(p->head_dim == 64 || p->head_dim == 128, "head_dim must be 64 or 128");
  CAREKV_REQUIRE(p->batch > 0 && p->n_heads > 0 && p->n_kv_heads > 0 && p->n_heads % p->n_kv_heads == 0,
                 "batch and head counts must be positive, n_heads a multiple of n_kv_heads");
  CAREKV_REQUIRE(p->seq_len > 0 && p->seq_len <= kEvalMaxT, "seq_len must be in 1..8192");
  // Python's int(n * ratio) raises on an infinite or NaN product (layer.py:397)
  CAREKV_REQUIRE(std::isfinite(p->ratio), "ratio must be finite");
  CAREKV_REQUIRE(p->ratio >= 0.0 && p->min_residuals >= 0, "ratio and min_residuals must be non-negative");
  CAREKV_REQUIRE(p->kind >= 0 && p->kind <= 2, "kind must be 0 (both), 1 (k) or 2 (v)");
  CAREKV_REQUIRE(!diag || p->diag_cap > 0, "diag needs diag_cap > 0");
  EvalArgs a{};
  a.q = q; a.k = k; a.v = v; a.kh = k_hat; a.vh = v_hat; a.o = o_base; a.out = out; a.diag = diag;
  a.B = p->batch; a.Hq = p->n_heads; a.Hkv = p->n_kv_heads; a.T = p->seq_len; a.diag_cap = diag ? p->diag_cap : 0;
  a.min_res = p->min_residuals; a.kind = p->kind; a.v_norm = p->v_score_norm != 0; a.normalize = p->normalize != 0;
  a.ratio = p->ratio; a.k_corr = p->k_corr_scale;
  a.sqrt_d = (float)std::sqrt((double)p->head_dim);
  a.inv_sqrt_d = (float)(1.0 / std::sqrt((double)p->head_dim));
  a.rcp_sqrt_d = 1.f / a.sqrt_d;
  const int T = p->seq_len, nc = eval_rows(T);
  const long nblk = (long)((T + nc - 1) / nc) * p->n_heads * p->batch;
  CAREKV_REQUIRE(nblk < (1L << 31), "too many (row block, head, sequence) work-groups");
  auto launch = [&](auto d, auto n) {
    constexpr int D = decltype(d)::value, NC = decltype(n)::value;
    const size_t shmem = eval_lds(D, NC, T);
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(prefill_eval_kernel<D, NC>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
    if (e != hipSuccess) (void)hipGetLastError();  // the launch itself reports an LDS size it cannot take
    hipLaunchKernelGGL((prefill_eval_kernel<D, NC>), dim3((unsigned)nblk), dim3(64 * kEvalWaves), shmem,
                       (hipStream_t)stream, a);
  };
  using std::integral_constant;
  auto by_rows = [&](auto d) {
    if (nc == 16) launch(d, integral_constant<int, 16>{});
    else if (nc == 8) launch(d, integral_constant<int, 8>{});
    else launch(d, integral_constant<int, 4>{});
  };
  if (p->head_dim == 128) by_rows(integral_constant<int, 128>{});
  else by_rows(integral_constant<int, 64>{});
  CAREKV_CHECK_LAUNCH("prefill_eval");
  return CAREKV_OK;
}


// Page terms of the sketch-proxy K score (CAREKV_KSCORE_LIVE=0): between the
// streaming and select kernels, one work-group per (split of pages, kv head,
// sequence).  For every query head of the GQA group and every page with a
// stored K slot, over the page's valid tokens t (attention.py:718-725, the
// same terms as ResidualRouter.route, residual_router.py:160-170):
//   mass     = sum_t a_t
//   boundary = sum_t a_t * (1 / max(s_top - s_t, 1e-6))
//   vdiff    = sum_t a_t * ||V_hat_t - O_base||
// with a = softmax(s) over the whole context, s_top = max_t s_t and O_base
// the fp32 base output.  The logits are the streaming kernel's own (x =
// s log2(e) in xbuf), so s_top is the maximum of exactly the values the
// margins subtract; a_t = 2^(x_t - M) / L from the split statistics; V_hat
// is dequantised exactly as in the streaming pass.
//
// Lane l = 16 j + m: token m, dims [j D/4, (j+1) D/4) of the page as it
// dequantises V_hat; afterwards token m of query 4 k + j.  The distances are
// ||V_hat_t||^2 + ||O||^2 - 2 V_hat_t . O on 16x16x32 MFMAs: the dequantised
// registers are the B operand as they stand (the dims in the codes' pair
// order), the A operand's rows 4 j .. 4 j + 2 hold query 4 k + j of O in three
// fp16 parts at a power of two of its own (33 bits of its largest element, the
// whole fp32 value), and the norms are the diagonal of V_hat V_hat^T.  Where the
// sum loses more than a third of its terms (a token near O_base), or is not
// finite, the pair takes the differences themselves, so that the distances keep
// the differences' error against 64 bits (D = 128, rms: V around zero 4.7e-8,
// differences 4.8e-8; around one deviation 5.3e-8 both, 6.5e-8 where it may
// lose half; around 3.5 deviations 7.6e-8 both, 4.3e-7 where it may lose
// 31/32).  A page of 4 queries costs about 200 VALU operations and 8 MFMAs; the
// differences alone took 384 VALU and 128 LDS reads.  A page's loads are issued
// while the page before it is worked on, and the split statistics are read by
// lanes side by side (a thread per query walked them before, two memory round
// trips a split).  Measured at 8 sequences x 8 kv heads x 8185 tokens, INT4, D =
// 128, 4 queries: 31.2 us, 56.8 us before.
//
// PF (prefill rows, the per-(head, row) router of correction_impl=cached,
// layer.py:573-640): a is the reference's fp16 attention weight of the row
// (the streaming pass's stored weights, against the row's log-sum-exp),
// s_top the row's largest logit (the streaming pass's per-wave maxima),
// O_base the fp16 base output half(sum_t a_t V_hat_t) (layer.py:964-965),
// V_hat the prompt's dense fp16 rows; logits past the row are -inf and
// their weights 0.
#include "decode_page.h"
#include "host_util.h"

namespace carekv {

// NG: groups of four queries whose operands a wave holds.
template <int D, int BITS, int SM, int NG, bool PF = false>
__global__ __launch_bounds__(256) void decode_proxy_kernel(carekv_arena A, DecodeArgs a) {
  using G = PageGeom<D, BITS>;
  using PB = typename G::PB;
  constexpr int NCG = G::NCG, CH = G::CH, CHB = G::CHB, RB = G::RB, NWC = G::NWC;
  constexpr int KS = CH / 8;                  // MFMA steps (8 dims of each lane group)
  constexpr float kEps = 1e-6f;               // residual_router.py:34
  constexpr float kLn2 = 0.693147180559945f;  // margins back from base-2 logits
  constexpr float kCancel = 1.5f;             // the expansion's terms are at most this multiple of the distance
  __shared__ float s_o[16 * D];               // O_base [query][dim]
  __shared__ float s_M[16], s_L[16], s_Mp[16], s_oo[16], s_up[16], s_dn[16];

  // prefill rows: the latest (longest) rows first
  const int split = blockIdx.x, kvh = blockIdx.y, b = a.pf ? (int)(gridDim.z - 1 - blockIdx.z) : (int)blockIdx.z;
  const int GQ = a.GQ;
  const int bk = b * A.n_kv_heads + kvh;
  const EntryRow er = entry_row(A, a, b);
  const int seq = er.seq, np = er.np;
  int p_lo, p_hi;
  launch_pages(A, a, seq, np, p_lo, p_hi);
  const int p_begin = p_lo + split * a.SP, p_end = min(p_begin + a.SP, p_hi);
  if (p_begin >= p_end) return;  // uniform over the work-group
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, lj = lane >> 4;
  const long pg_base = ((long)kvh * A.n_seq + seq) * A.max_pages;

  // ---- softmax statistics of the group's queries, a query per wave
  for (int qq = w; qq < GQ; qq += 4) {
    float M = -INFINITY, L = 0.f, xm = -INFINITY;
    for (int s = lane; s < a.nsplit; s += 64) M = fmaxf(M, a.pml[(((long)bk * a.nsplit + s) * 16 + qq) * 2]);
    M = wave_max(M);
    if (M != -INFINITY)
      for (int s = lane; s < a.nsplit; s += 64) {
        const long base = ((long)bk * a.nsplit + s) * 16 + qq;
        const float ms = a.pml[base * 2];
        if (ms != -INFINITY) L += a.pml[base * 2 + 1] * __builtin_amdgcn_exp2f(ms - M);
      }
    L = wave_sum(L);
    if constexpr (PF) {
      for (int i = lane; i < a.nsplit * 4; i += 64) xm = fmaxf(xm, a.xmax[((long)bk * a.nsplit * 4 + i) * 16 + qq]);
      xm = wave_max(xm);
    }
    if (lane == 0) {
      s_M[qq] = PF ? xm : M;  // the margins' s_top
      s_L[qq] = L;
      s_Mp[qq] = M;           // the split partials' reference maximum
    }
  }
  __syncthreads();
  // ---- O_base (split order), its norm and its operand's scale
  for (int i = 2 * threadIdx.x; i < GQ * D; i += 512) {
    const int qq = i / D, d = i % D;
    const float M = s_Mp[qq], L = s_L[qq];
    float2 O = make_float2(0.f, 0.f);
    if (M != -INFINITY)
#pragma unroll 8
      for (int s = 0; s < a.nsplit; ++s) {
        const long base = ((long)bk * a.nsplit + s) * 16 + qq;
        const float ms = a.pml[base * 2];
        const float2 o = *reinterpret_cast<const float2*>(a.po + base * D + d);  // (an empty split's is not used)
        const float f = __builtin_amdgcn_exp2f(ms - M);
        O.x = ms != -INFINITY ? O.x + o.x * f : O.x;
        O.y = ms != -INFINITY ? O.y + o.y * f : O.y;
      }
    // prefill rows: the fp16 base output, the weights already normalised
    s_o[i] = PF ? (float)(_Float16)O.x : (L > 0.f ? O.x / L : 0.f);
    s_o[i + 1] = PF ? (float)(_Float16)O.y : (L > 0.f ? O.y / L : 0.f);
  }
  __syncthreads();
  for (int qq = w; qq < GQ; qq += 4) {
    float oo = 0.f, mx = 0.f;
#pragma unroll
    for (int d = 0; d < D; d += 64) {
      const float o = s_o[qq * D + d + lane];
      oo = fmaf(o, o, oo);
      mx = fmaxf(mx, fabsf(o));
    }
    oo = wave_sum(oo);
    mx = wave_max(mx);
    if (lane == 0) {
      s_oo[qq] = oo;
      // 2^k that brings the largest element into [2^8, 2^9); 1 for a zero or infinite row
      const int e = __builtin_amdgcn_frexp_expf(mx);
      const int k = mx > 0.f && mx < INFINITY ? min(9 - e, 126) : 0;
      s_up[qq] = __builtin_amdgcn_ldexpf(1.f, k);
      s_dn[qq] = __builtin_amdgcn_ldexpf(1.f, -k);
    }
  }
  __syncthreads();
  // A operands: row ln = 4 (query) + part (high, middle, low, zero), this lane's dims in the codes' pair order
  half8_t op[NG][KS];
#pragma unroll
  for (int k = 0; k < NG; ++k) {
    const int qq = 4 * k + (ln >> 2);
    const int part = ln & 3;
    const bool on = qq < GQ && part < 3;
    const float up = on ? s_up[qq] : 0.f;
    const float* o = s_o + (on ? qq : 0) * D + lj * CH;
#pragma unroll
    for (int i = 0; i < CH / 2; ++i) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const float x = on ? o[u ? PB::T.b[i] : PB::T.a[i]] * up : 0.f;
        const _Float16 hi = (_Float16)x, mid = (_Float16)(x - (float)hi);
        const _Float16 lo = (_Float16)((x - (float)hi) - (float)mid);
        op[k][i / 4][2 * (i % 4) + u] = part == 0 ? hi : part == 1 ? mid : lo;
      }
    }
  }

  RowRes rr;
  if constexpr (PF) {
    static_assert(BITS == 16, "prefill rows are fp16");
    rr.vc = make_rsrc(a.pf_v + (long)kvh * a.pf_T * D, (uint32_t)a.pf_T * D * 2);  // rows past the prompt read 0
    rr.kc = rr.ks = rr.vs = make_rsrc(nullptr, 0u);
  } else {
    rr = row_resources<D, BITS, SM>(A, pg_base);
  }
  const float* ob = s_o + lj * CH;
  // a page's loads: V_hat of token ln, chunk lj, the queries' logits, metadata
  struct PageIn {
    uint32_t vw[NWC];
    int vcode, nv, hm, ksl[NCG];
    float vm, xs[NG];
  };
  auto load = [&](int p, PageIn& x) {
    const long pg = pg_base + p;
    const uint32_t row = (uint32_t)(p * kPage + ln);
    buf_load<CHB>(x.vw, rr.vc, row * RB + lj * CHB);
    const int gi = (lj * CH) / 32;
    if constexpr (SM == 1) x.vcode = (int)(int8_t)__builtin_amdgcn_raw_buffer_load_b8(rr.vs, row * NCG + gi, 0, 0);
    else x.vcode = __builtin_amdgcn_raw_buffer_load_b16(rr.vs, (row * NCG + gi) * 2, 0, 0);
    x.vm = SM == 1 ? h2f(A.vmaster[pg]) : 0.f;
#pragma unroll
    for (int k = 0; k < NG; ++k) x.xs[k] = a.xbuf[(((long)bk * GQ + min(4 * k + lj, GQ - 1)) * a.Pmax + p) * 16 + ln];
    x.nv = A.valid[pg];
    x.hm = A.has_meta[pg];
#pragma unroll
    for (int cg = 0; cg < NCG; ++cg) x.ksl[cg] = A.k_slot[pg * NCG + cg];
  };
  PageIn nx;
  if (p_begin + w < p_end) load(p_begin + w, nx);
  for (int p = p_begin + w; p < p_end; p += 4) {
    const PageIn in_ = nx;
    if (p + 4 < p_end) load(p + 4, nx);
    const int nv = in_.nv;
    bool anyk = false;
#pragma unroll
    for (int cg = 0; cg < NCG; ++cg) anyk |= in_.ksl[cg] >= 0 && in_.ksl[cg] < A.n_slots;
    if (nv <= 0 || !in_.hm || !anyk) continue;  // no K candidate on the page
    half2_t vp[CH / 2];
    dequant_pairs<BITS, CH, BITS>(in_.vw, lane_scale<SM>(in_.vcode, in_.vm), vp);
    half8_t vb[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        vb[ks][2 * i] = vp[4 * ks + i][0];
        vb[ks][2 * i + 1] = vp[4 * ks + i][1];
      }
    float4_t v2{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) v2 = mfma16x32(vb[ks], vb[ks], v2);
    const float vv = diag16(v2, ln, lj);  // token ln's norm

#pragma unroll
    for (int k = 0; k < NG; ++k) {
      const int q0 = 4 * k;
      if (q0 >= GQ) break;
      const int qq = q0 + lj;
      float4_t vo{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) vo = mfma16x32(op[k][ks], vb[ks], vo);
      const bool in = qq < GQ && ln < nv;
      const float sum = vv + s_oo[in ? qq : 0];
      float d2 = fmaf(-2.f, (vo[0] + (vo[1] + vo[2])) * s_dn[in ? qq : 0], sum);
      const bool near = in && !(d2 * kCancel >= sum);  // (or not finite)
      if (__any(near)) {
        // ||V_hat_t - O_q||^2 for queries q0 .. q0+3; row j keeps query q0 + j
#pragma unroll 1
        for (int u = 0; u < 4; ++u) {
          if (q0 + u >= GQ) break;
          const float* o = ob + (q0 + u) * D;
          float acc = 0.f;
#pragma unroll
          for (int i = 0; i < CH / 2; ++i) {
            const float d0 = (float)vp[i][0] - o[PB::T.a[i]];
            const float d1 = (float)vp[i][1] - o[PB::T.b[i]];
            acc = fmaf(d0, d0, acc);
            acc = fmaf(d1, d1, acc);
          }
          const float tot = col_sum(acc);
          if (lj == u && near) d2 = tot;
        }
      }
      float at = 0.f, bt = 0.f, vt = 0.f;
      if (in) {
        const float M = s_M[qq], L = s_L[qq];
        const float x = in_.xs[k];
        if (x != -INFINITY && M != -INFINITY && L > 0.f) {
          if constexpr (PF) at = h2f(a.ebuf[(((long)bk * GQ + qq) * a.Pmax + p) * 16 + ln]);
          else at = __builtin_amdgcn_exp2f(x - M) / L;
          bt = at * (1.f / fmaxf((M - x) * kLn2, kEps));
          vt = at * sqrtf(d2);
        }
      }
      at = row16_sum(at);
      bt = row16_sum(bt);
      vt = row16_sum(vt);
      if (qq < GQ && ln == 0)
        *reinterpret_cast<float4*>(a.prox + (((long)bk * GQ + qq) * a.Pmax + p) * 4) = make_float4(at, bt, vt, 0.f);
    }
  }
}

int launch_decode_proxy(const carekv_arena& A, const DecodeArgs& a, hipStream_t s) {
  const dim3 grid(a.nsplit_run, A.n_kv_heads, a.B);
  if (a.pf) {
    if (A.head_dim == 64) hipLaunchKernelGGL((decode_proxy_kernel<64, 16, 0, 4, true>), grid, dim3(256), 0, s, A, a);
    else hipLaunchKernelGGL((decode_proxy_kernel<128, 16, 0, 4, true>), grid, dim3(256), 0, s, A, a);
    CAREKV_CHECK_LAUNCH("decode_proxy (prefill rows)");
    return CAREKV_OK;
  }
  return dispatch_dbs16(A.head_dim, A.base_bits, A.scale_mode, [&](auto d, auto bb, auto sm) {
    constexpr int D = decltype(d)::value, BITS = decltype(bb)::value, SM = decltype(sm)::value;
    // one group of four queries costs a quarter of the operand registers (D =
    // 128: 114-122 VGPRs, four waves per SIMD, against 185-194, two; the
    // differences alone took 82).  Both beat the differences: 8 sequences of 8185
    // tokens, 32 / 8 heads 143 -> 106 us a step, 40 / 8 183 -> 170, 16 / 2 178 ->
    // 120, 32 / 2 253 -> 160; 32 / 2 heads, D = 64, 176 -> 122
    if (a.GQ <= 4) hipLaunchKernelGGL((decode_proxy_kernel<D, BITS, SM, 1>), grid, dim3(256), 0, s, A, a);
    else hipLaunchKernelGGL((decode_proxy_kernel<D, BITS, SM, 4>), grid, dim3(256), 0, s, A, a);
    CAREKV_CHECK_LAUNCH("decode_proxy");
    return CAREKV_OK;
  });
}

}  // namespace carekv

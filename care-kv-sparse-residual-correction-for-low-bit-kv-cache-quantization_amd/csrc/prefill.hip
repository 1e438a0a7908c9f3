// Prefill attention over dequantised K/V (CAREKVLayer._causal_attention_pure,
// layer.py:935-972) on v_mfma_f32_16x16x32_f16, flash style: the (T, T)
// score and weight matrices are never materialised; the kernel returns O and,
// optionally, the per-row log-sum-exp from which any weight can be rebuilt.
//
// One work-group per (block of 128 queries, query head, sequence), 4 waves of
// 32 queries, on a one-dimensional grid whose order starts the longest (latest)
// query blocks first, a few heads of an XCD at a time: with every head's blocks
// in flight their K/V passed the XCD's 4 MB L2 and the tiles came from HBM.
// K and V tiles of 32 tokens are staged in LDS (double buffered, one barrier per
// tile; the next tile's global loads are in flight while the current one is
// used); at D = 128, 160 VGPRs and 35 KB of LDS, three work-groups share a CU.
// 48 queries a wave (218 VGPRs, two work-groups) measured the same (4 x 40
// heads, T = 8192: 2912 us against 2917; 8 x 32 / 8 heads, T = 3000: 692 against
// 686).
//   * S^T = K_hat Q^T: A = K tile rows (one 16-byte LDS read per lane and
//     32-dim step), B = Q^T held in registers; lane l receives the scores of
//     tokens 16tt + 4(l/16) + i for query l % 16 of a 16-query sub-block;
//   * the online softmax runs per query column in fp32 on base-2 logits
//     (scores scaled by log2(e)/sqrt(D) after the fp32 product, as the
//     reference divides the fp32 product by sqrt(D)).
//     Each lane compares its own 8 scores with the column's running maximum;
//     only where one is larger are they reduced over the lane groups, the sums
//     rescaled and the maximum moved.  Columns that keep theirs are multiplied
//     by exactly 1, so that a row's bits depend on its own scores alone.  The
//     reduction and the factor in every tile took 3506 us against 3402 at B = 4,
//     40 heads, T = 8192, D = 128, and 216 against 208 at B = 8, 32 / 4 heads,
//     T = 2047, D = 64 (before the grouped order below).  A maximum that lags
//     behind the scores by up to 2^8 was faster still (2670 against 2890 us with
//     that order), but it rounds the weights of a row's largest scores, which
//     are exactly 1 here: the error against a 64-bit evaluation rose from
//     2.58e-4 to 2.69e-4 (D = 64: 2.52e-4 to 2.63e-4);
//   * O^T += V_hat^T P^T: the weights are already in the B layout (the 8 k
//     values of a lane are tokens 4(l/16) + i of two 16-token tiles), and
//     the A operand V_hat^T comes from the token-major V tile through the
//     gfx950 transpose load ds_read_b64_tr_b16 for the same token order.
// The K tile rows are padded to 2D + 16 bytes and the V tile rows to 2D + 32
// bytes, so that each group of consecutive lanes of either LDS read pattern
// touches every bank once.
#include <algorithm>
#include <cmath>

#include "decode_page.h"
#include "host_util.h"

namespace carekv {

struct PrefillArgs {
  const uint16_t* q;  // [B][Hq][T][D]
  const uint16_t* k;  // [B][Hkv][T][D]
  const uint16_t* v;
  uint16_t* out;      // [B][Hq][T][D]
  float* lse;         // [B][Hq][T] natural log-sum-exp of the scaled scores, or null
  int B, Hq, Hkv, T, causal;
  int group;          // heads of an XCD whose query blocks run together; 0: every head at once
  float sm_log2;      // sm_scale * log2(e)
};

template <int D>
__global__ __launch_bounds__(256, 3) void prefill_attn_kernel(PrefillArgs a) {
  constexpr int KT = 32;              // tokens per K/V tile
  constexpr int TT = KT / 16, NU = KT / 32;
  constexpr int NQ = 2;               // 16-query sub-blocks of a wave
  constexpr int QW = 16 * NQ;         // queries per wave
  constexpr int QB = 4 * QW;          // and per work-group
  constexpr int KRS = 2 * D + 16;     // K tile row stride, bytes
  constexpr int VRS = 2 * D + 32;     // V tile row stride, bytes
  constexpr int KS = D / 32;          // 32-dim steps of the score product
  constexpr int DT = D / 16;          // 16-dim output tiles
  constexpr int KBUF = KT * KRS, VBUF = KT * VRS, BUF = KBUF + VBUF;
  constexpr int CHR = D / 8;          // 16-byte chunks per row
  constexpr int NCH = 2 * KT * CHR / 256;  // chunks a thread stages per tile
  constexpr float kLow = -1e30f;      // below any score; finite, so that a masked score's weight is 0 from the first tile
  __shared__ __align__(16) char lds[2 * BUF];
  typedef short short4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) short4_t lds_short4;

  // The longest (latest) query blocks start first.  Work-group ids go round the
  // 8 XCDs; with a.group an XCD takes nh consecutive heads (the query heads of
  // a kv head meet in one L2), a group of them at a time.
  const int nhb = a.Hq * a.B, nqb = gridDim.x / nhb;
  int qblk = nqb - 1 - (int)blockIdx.x / nhb, hb = (int)blockIdx.x % nhb;
  if (a.group) {
    const int nh = nhb / 8, n = (int)blockIdx.x / 8;
    const int first = n / (a.group * nqb) * a.group, cur = min(a.group, nh - first), r = n - first * nqb;
    qblk = nqb - 1 - r / cur;
    hb = (int)blockIdx.x % 8 * nh + first + r % cur;
  }
  const int h = hb % a.Hq, b = hb / a.Hq;
  const int hk = h / (a.Hq / a.Hkv);
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  const int T = a.T;
  const int q0 = qblk * QB, qw0 = q0 + QW * w;
  const uint32_t span = (uint32_t)T * D * 2;
  const __amdgpu_buffer_rsrc_t rq = make_rsrc(a.q + ((long)b * a.Hq + h) * T * D, span);
  const __amdgpu_buffer_rsrc_t rk = make_rsrc(a.k + ((long)b * a.Hkv + hk) * T * D, span);
  const __amdgpu_buffer_rsrc_t rv = make_rsrc(a.v + ((long)b * a.Hkv + hk) * T * D, span);

  // Q^T operands: sub-block qb, step s -> query qw0 + 16 qb + c16, dims 32s + 8g ..
  half8_t qf[NQ][KS];
#pragma unroll
  for (int qb = 0; qb < NQ; ++qb)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint32_t qi = (uint32_t)(qw0 + 16 * qb + c16);
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(rq, (qi * D + 32 * s + 8 * g) * 2, 0, 0);
      __builtin_memcpy(&qf[qb][s], &v, 16);
    }

  const int q_last = min(q0 + QB, T) - 1;
  const int nt = a.causal ? q_last / KT + 1 : (T + KT - 1) / KT;

  // staging: chunk c = threadIdx.x + 256 k -> tensor c / (KT CHR) (K, V), row, 16-byte column
  uint32_t stg[NCH][4];
  auto load_tile = [&](int j) {
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
      const int c = threadIdx.x + 256 * k;
      const int rc = c % (KT * CHR), row = rc / CHR, col = rc % CHR;
      const uint32_t off = ((uint32_t)(j * KT + row) * D + col * 8) * 2;
      // chunks 0 .. KT*CHR-1 are K, the rest V: with 256 threads that is
      // k < NCH / 2, known at compile time (a per-lane choice of resource
      // would make every load a waterfall loop)
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(k < NCH / 2 ? rk : rv, off, 0, 0);
      stg[k][0] = v[0]; stg[k][1] = v[1]; stg[k][2] = v[2]; stg[k][3] = v[3];
    }
  };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
      const int c = threadIdx.x + 256 * k;
      const int rc = c % (KT * CHR), row = rc / CHR, col = rc % CHR;
      char* dst = lds + buf * BUF + (k < NCH / 2 ? row * KRS : KBUF + row * VRS) + col * 16;
      *reinterpret_cast<uint4*>(dst) = make_uint4(stg[k][0], stg[k][1], stg[k][2], stg[k][3]);
    }
  };

  float m_run[NQ], l_run[NQ];
  float4_t o[NQ][DT];
#pragma unroll
  for (int qb = 0; qb < NQ; ++qb) {
    m_run[qb] = kLow;
    l_run[qb] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[qb][dt] = float4_t{0.f, 0.f, 0.f, 0.f};
  }

  load_tile(0);
  store_tile(0);
  __syncthreads();
  if (nt > 1) load_tile(1);

  for (int j = 0; j < nt; ++j) {
    const char* kb = lds + (j & 1) * BUF;
    const char* vb = kb + KBUF;
    const int t0 = j * KT;
    if (!a.causal || t0 <= qw0 + QW - 1) {  // some query of the wave sees this tile
      // ---- S^T = K_hat Q^T (raised wave priority over the MFMA blocks: a wave
      // with products to issue goes before the CU's other waves' softmax)
      __builtin_amdgcn_s_setprio(1);
      float4_t s[TT][NQ];
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
#pragma unroll
        for (int qb = 0; qb < NQ; ++qb) s[tt][qb] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          half8_t ak;
          *reinterpret_cast<uint4*>(&ak) = *reinterpret_cast<const uint4*>(kb + (16 * tt + c16) * KRS + (32 * ks + 8 * g) * 2);
#pragma unroll
          for (int qb = 0; qb < NQ; ++qb) s[tt][qb] = mfma16x32(ak, qf[qb][ks], s[tt][qb]);
        }
      }
      __builtin_amdgcn_s_setprio(0);
      // ---- mask (the wave's diagonal and the end of the sequence), then
      // the base-2 logits x = s * log2(e)/sqrt(D) folded into the exponent:
      // max x = c * max s for c > 0 (rounding is monotone), and
      // exp2(x - m) is taken as exp2(fma(s, c, -m))
      const bool edge = (a.causal && t0 + KT - 1 > qw0) || t0 + KT > T;
      const float c = a.sm_log2;
      half8_t bp[NQ];
      if (edge) {
#pragma unroll
        for (int qb = 0; qb < NQ; ++qb) {
          const int qi = qw0 + 16 * qb + c16;
          // token 16 tt + i of the lane's rows is t0 + 4g + 16 tt + i; the
          // limits pass through an empty asm so that the compares stay on
          // this branch (most tiles are not edge tiles)
          int lim_t = T - t0 - 4 * g, lim_q = a.causal ? qi - t0 - 4 * g : 0x3fffffff;
          asm volatile("" : "+v"(lim_t), "+v"(lim_q));
#pragma unroll
          for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int o = 16 * tt + i;
              if (o >= lim_t || o > lim_q) s[tt][qb][i] = -INFINITY;
            }
        }
      }
      // A column's maximum moves where one of its own lanes holds a larger
      // score: only such a tile reduces it over the lane groups and rescales
      // (the first always does).  Columns of the wave that keep theirs get a
      // factor of exactly 1, so a row's bits do not depend on its neighbours.
      float mx[NQ];
      bool over[NQ], any_over = false;
#pragma unroll
      for (int qb = 0; qb < NQ; ++qb) {
        mx[qb] = -INFINITY;  // a chain of three-operand maxima over the lane's 8 scores
#pragma unroll
        for (int k = 0; k < 4 * TT; k += 2) mx[qb] = fmaxf(fmaxf(mx[qb], s[k / 4][qb][k % 4]), s[k / 4][qb][k % 4 + 1]);
        over[qb] = mx[qb] * c > m_run[qb];
        any_over |= over[qb];
      }
      if (__any(any_over)) {
#pragma unroll
        for (int qb = 0; qb < NQ; ++qb) {
          if (!__any(over[qb])) continue;
          const float m_new = fmaxf(m_run[qb], pair32_max(pair16_max(mx[qb])) * c);
          const float f = __builtin_amdgcn_exp2f(m_run[qb] - m_new);
          m_run[qb] = m_new;
          l_run[qb] *= f;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) o[qb][dt] *= f;
        }
      }
      // the weights, and this lane's sums of them (its tokens; over the lane groups at the end)
#pragma unroll
      for (int qb = 0; qb < NQ; ++qb) {
        float ls = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float p = __builtin_amdgcn_exp2f(fmaf(s[i / 4][qb][i % 4], c, -m_run[qb]));
          ls += p;
          bp[qb][i] = (_Float16)p;
        }
        l_run[qb] += ls;
      }
      __builtin_amdgcn_s_setprio(1);
      // ---- O^T += V_hat^T P^T, 32 tokens per step
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        // source lane c16 of group g reads row 32u + 4g + c16/4 (and +16), dims 16dt + 4(c16%4) ..
        const __attribute__((address_space(3))) char* vrow =
            (const __attribute__((address_space(3))) char*)vb + (32 * u + 4 * g + (c16 >> 2)) * VRS + (c16 & 3) * 8;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const short4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(vrow + 32 * dt));
          const short4_t v2 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(vrow + 16 * VRS + 32 * dt));
          half8_t av;
          __builtin_memcpy(&av, &v1, 8);
          __builtin_memcpy(reinterpret_cast<char*>(&av) + 8, &v2, 8);
#pragma unroll
          for (int qb = 0; qb < NQ; ++qb) o[qb][dt] = mfma16x32(av, bp[qb], o[qb][dt]);
        }
      }
    }
    __builtin_amdgcn_s_setprio(0);
    if (j + 1 < nt) store_tile((j + 1) & 1);
    if (j + 2 < nt) load_tile(j + 2);
    __syncthreads();
  }

  // ---- normalise and write (lane: query qw0 + 16qb + c16, dims 16dt + 4g ..)
#pragma unroll
  for (int qb = 0; qb < NQ; ++qb) {
    const float lt = pair32_sum(pair16_sum(l_run[qb]));
    const float inv = 1.f / lt;
    const int qi = qw0 + 16 * qb + c16;
    if (qi < T) {
      uint16_t* dst = a.out + (((long)b * a.Hq + h) * T + qi) * D + 4 * g;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const uint32_t lo = (uint32_t)f2h(o[qb][dt][0] * inv) | ((uint32_t)f2h(o[qb][dt][1] * inv) << 16);
        const uint32_t hi = (uint32_t)f2h(o[qb][dt][2] * inv) | ((uint32_t)f2h(o[qb][dt][3] * inv) << 16);
        *reinterpret_cast<uint2*>(dst + 16 * dt) = make_uint2(lo, hi);
      }
      if (a.lse && g == 0) a.lse[((long)b * a.Hq + h) * T + qi] = (m_run[qb] + __log2f(lt)) * 0.69314718f;
    }
  }
}

// x_hat = half(code * scale) per group of 32 (quantizer.py:67-82): the
// product of an int8 code and an fp16 scale is exact in fp32 and is rounded
// once to fp16.
__global__ void dequantize_rows_kernel(const int8_t* __restrict__ codes, const uint16_t* __restrict__ scale,
                                       long n, int D, uint16_t* __restrict__ out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long r = i / D;
  const int d = (int)(i % D);
  out[i] = f2h((float)codes[i] * h2f(scale[r * (D / 32) + d / 32]));
}

}  // namespace carekv

using namespace carekv;

extern "C" int carekv_prefill_attn(const carekv_prefill_params* pp, const uint16_t* q, const uint16_t* k,
                                   const uint16_t* v, uint16_t* out, float* lse, void* stream) {
  CAREKV_REQUIRE(pp && q && k && v && out, "null argument");
  CAREKV_REQUIRE(pp->head_dim == 64 || pp->head_dim == 128, "head_dim must be 64 or 128");
  CAREKV_REQUIRE(pp->batch > 0 && pp->n_heads > 0 && pp->n_kv_heads > 0, "batch and head counts must be positive");
  CAREKV_REQUIRE(pp->n_heads % pp->n_kv_heads == 0, "n_heads must be a multiple of n_kv_heads");
  CAREKV_REQUIRE(pp->seq_len > 0, "seq_len must be positive");
  // 32-bit buffer offsets reach one query block and one key tile past the end
  CAREKV_REQUIRE(((long)pp->seq_len + 128) * pp->head_dim * 2 < (1L << 31), "one head's sequence exceeds 2 GiB");
  PrefillArgs a{};
  a.q = q; a.k = k; a.v = v; a.out = out; a.lse = lse;
  a.B = pp->batch; a.Hq = pp->n_heads; a.Hkv = pp->n_kv_heads; a.T = pp->seq_len; a.causal = pp->causal != 0;
  a.sm_log2 = pp->sm_scale * 1.4426950408889634f;
  const long hb = (long)pp->n_heads * pp->batch, T = pp->seq_len;
  const long nblk = (T + 127) / 128 * hb;
  CAREKV_REQUIRE(nblk < (1L << 31), "too many query blocks");
  // Heads per XCD that run together: about 32768 of their queries, 2 2/3 rounds
  // of the XCD's resident work-groups, so that a few heads' K/V tiles stay in
  // its L2 and the longest blocks still start early enough (the last group has
  // the heads that are left).  4 x 40 heads, T = 8192: 2894 us against
  // 3402 with every head at once; B = 8, 32 / 4 heads, D = 64: 2657 against 2840
  // at T = 8192, 194 against 208 at T = 2047.  Head counts that 8 does not divide
  // would load the XCDs unevenly and keep every head at once.
  if (hb % 8 == 0) {
    const long nh = hb / 8, n_groups = std::max(1L, nh * T / 32768);
    a.group = (int)((nh + n_groups - 1) / n_groups);
  }
  const dim3 grid((unsigned)nblk);
  hipStream_t s = (hipStream_t)stream;
  if (pp->head_dim == 128) hipLaunchKernelGGL(prefill_attn_kernel<128>, grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(prefill_attn_kernel<64>, grid, dim3(256), 0, s, a);
  CAREKV_CHECK_LAUNCH("prefill_attn");
  return CAREKV_OK;
}

extern "C" int carekv_dequantize_rows(const int8_t* codes, const uint16_t* scale, int32_t rows, int32_t D,
                                      int32_t group, uint16_t* out, void* stream) {
  CAREKV_REQUIRE(codes && scale && out, "null argument");
  CAREKV_REQUIRE(group == 32 && D % 32 == 0 && D > 0, "kernels support group_size=32 and D % 32 == 0");
  if (rows <= 0) return CAREKV_OK;
  const long n = (long)rows * D;
  hipLaunchKernelGGL(dequantize_rows_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     codes, scale, n, D, out);
  CAREKV_CHECK_LAUNCH("dequantize_rows");
  return CAREKV_OK;
}

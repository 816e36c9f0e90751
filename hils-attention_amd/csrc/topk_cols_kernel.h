// The one-pass prefill selection of KV heads with one query head, up to 256 chunks in sight (topk_group.hip launches it).
//
// One wavefront owns 16 consecutive queries of a (batch, head).  The scores are formed transposed, S^T = K q^T: the 16
// queries are the columns of the matrix product, and a lane holds, of one query, the chunks nt*16 + 4j + i (accumulator
// register i of block nt in lane (query, j)): a query's scores lie in four lanes, 4*NB in each.  All 16 queries are worked
// on at once and a reduction over a query is in-lane work and two row swaps.  (With the queries as rows, the layout that
// two to eight heads need, a query's scores lie in the 16 lanes of a lane row and four queries are worked on at a time: 16
// queries take four selections, whose reductions, searches and write-outs were 80 % of 2690 vector instructions a wavefront
// at 128 chunks, vector ALU 97 % busy.)
//
// Selection.  The threshold is searched by value: probe c, count the scores from c up, stop at exactly K.  The first probe
// is the quantile of a normal distribution with the row's maximum and sum of exponentials (what the log-sum-exp has
// anyway), the second shifts by the quantile difference of the count seen, the others interpolate between the two nearest
// probes, every fourth halves the range of the scores' order-preserving integer images (so that the search ends whatever
// the scores are), and once every query is one score off, the next probe is the score that is too many or missing: about
// five probes for normal, uniform or exponential scores, where halving the integer images takes sixteen for the slowest of
// 16 queries.  Ties at the threshold go to the lower chunk indices.
//
// us, queries as rows / as columns, top-32, heads of 64: B8 L8192 16 heads 294 / 165; L16000 16 heads 62 + 87 / 35 + 60 (up to
// 128 chunks + up to 256; held to the 168 registers of three wavefronts per SIMD the second spills four, 69 at two);
// B2 L3000 4 heads with a bias, top-16, 22.4 / 14.0.
#pragma once
#include "topk_group_kernel.h"

#define TC_WAVES 2  // wavefronts per workgroup (they never synchronise)

__device__ __forceinline__ int tc_rows_sum_i(int x) {
  hils_uint2v a = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)x, false, false);
  x = (int)(a.x + a.y);
  hils_uint2v b = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)x, false, false);
  return (int)(b.x + b.y);
}
// Sum over the four lanes of a query and the sum over those before this one (j = lane >> 4).
__device__ __forceinline__ unsigned tc_rows_scan(unsigned x, int j, unsigned& total) {
  hils_uint2v a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  const unsigned pair = a.x + a.y;
  hils_uint2v b = __builtin_amdgcn_permlane32_swap(pair, pair, false, false);
  total = b.x + b.y;
  return ((j & 1) ? a.x : 0u) + ((j & 2) ? b.x : 0u);
}
// z with P(normal > z) = p (rational approximation, Abramowitz and Stegun 26.2.23: error below 5e-4)
__device__ __forceinline__ float tc_normal_quantile(float p) {
  const float h = fminf(p, 1.f - p);
  const float t = __builtin_amdgcn_sqrtf(-2.f * HILS_LN2 * __builtin_amdgcn_logf(h));
  const float num = fmaf(t, fmaf(t, 0.010328f, 0.802853f), 2.515517f);
  const float den = fmaf(t, fmaf(t, fmaf(t, 0.001308f, 0.189269f), 1.432788f), 1.f);
  const float z = t - num * __builtin_amdgcn_rcpf(den);
  return p < 0.5f ? z : -z;
}

template <int KS, int NB, bool BIAS>
__global__ void __launch_bounds__(64 * TC_WAVES) __attribute__((amdgpu_waves_per_eu(NB <= 8 ? 4 : 3)))
topk_fwd_cols_kernel(TgArgs a, int bs_shift) {
  constexpr int D = KS * 32;
  constexpr int NV = 4 * NB;  // scores of a lane
  constexpr int NM = NV / 32;  // words of its winner mask
  static_assert(NB % 8 == 0 && NB <= 16, "whole mask words; two copies of the scores in registers");
  __shared__ __align__(16) uint32_t stage_w[TC_WAVES][16 * 32];  // winners, [query][slot]: chunk << 16 | bf16 score
  __shared__ __align__(16) float bias_s[BIAS ? NB * 16 : 4];     // of this (batch, head)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane & 15, j = lane >> 4;
  const int hk = blockIdx.y, N = a.N, topk = a.topk;
  const long b = blockIdx.z;
  const int t0 = a.t_base + (blockIdx.x * TC_WAVES + wave) * 16;
  if constexpr (BIAS) {
    for (int c = threadIdx.x; c < NB * 16; c += 64 * TC_WAVES) bias_s[c] = c < N ? a.bias[(b * N + c) * (long)a.h_kv + hk] : 0.f;
    __syncthreads();
  }
  if (t0 >= a.t_end) return;
  uint32_t* stage = stage_w[wave];

  // this lane's query
  const int tq = t0 + col;
  const bool ok = tq < a.t_end;
  const int tc = ok ? tq : t0;
  int lim;
  {
    const int x = a.window_size > 0 ? tc + a.q_offset - a.window_size + 1 : tc + a.q_offset;
    int lm = a.causal ? (bs_shift >= 0 ? (x >> bs_shift) : floordiv(x, a.block_size)) : N;
    lm = lm < 0 ? 0 : (lm > N ? N : lm);
    lim = ok ? lm - 4 * j : -1000000;  // chunk nt*16 + 4j + i is in sight while nt*16 + i < lim
  }
  const long row = (b * a.L + tc) * (long)a.h_kv + hk;
  bf16x8_t qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qf[ks] = *(const bf16x8_t*)(a.q + row * D + ks * 32 + j * 8);
  const float swa = a.lse_bf16 ? bf2f(((const bf16_t*)a.lse_swa)[row]) : a.lse_swa[row];

  // ---- the logits, -inf where the chunk is not in sight; a block's keys are loaded one block ahead ----
  typedef unsigned tc_u4 __attribute__((ext_vector_type(4)));
  const int nb_real = (N + 15) / 16;
  const uint4* pbase = a.pk + ((b * a.h_kv + hk) * (long)nb_real * KS) * 64 + lane;
  float x[NB][4];
  auto load = [&](int nt, tc_u4 (&d)[KS]) __attribute__((always_inline)) {
    const int nn = nt < nb_real ? nt : nb_real - 1;  // blocks past the tensor re-read its last one and are masked
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) d[ks] = *(const tc_u4*)&pbase[((long)nn * KS + ks) * 64];
  };
  auto use = [&](int nt, const tc_u4 (&d)[KS]) __attribute__((always_inline)) {
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, d[ks]), qf[ks], acc, 0, 0, 0);
    f32x4_t bv = {0.f, 0.f, 0.f, 0.f};
    if constexpr (BIAS) bv = *(const f32x4_t*)&bias_s[nt * 16 + 4 * j];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = __fmul_rn(acc[i], a.sm_scale);
      if constexpr (BIAS) v = __fadd_rn(v, bv[i]);
      x[nt][i] = (nt * 16 + i < lim) ? v : HILS_NEG_INF;
    }
  };
  {
    tc_u4 k0[KS], k1[KS], k2[KS], k3[KS];  // four blocks in flight
    load(0, k0);
    load(1, k1);
    load(2, k2);
    load(3, k3);
#pragma unroll
    for (int nt = 0; nt < NB; nt += 4) {
      __builtin_amdgcn_sched_barrier(0);
      use(nt, k0);
      if (nt + 4 < NB) load(nt + 4, k0);
      __builtin_amdgcn_sched_barrier(0);
      use(nt + 1, k1);
      if (nt + 5 < NB) load(nt + 5, k1);
      __builtin_amdgcn_sched_barrier(0);
      use(nt + 2, k2);
      if (nt + 6 < NB) load(nt + 6, k2);
      __builtin_amdgcn_sched_barrier(0);
      use(nt + 3, k3);
      if (nt + 7 < NB) load(nt + 7, k3);
    }
  }

  // ---- lse_total = logaddexp(lse_swa, logsumexp of the visible logits), as in topk_fwd_group_kernel ----
  float hi_x = HILS_NEG_INF;
#pragma unroll
  for (int nt = 0; nt < NB; ++nt) hi_x = fmaxf(hi_x, fmaxf(fmaxf(x[nt][0], x[nt][1]), fmaxf(x[nt][2], x[nt][3])));
  hi_x = rows_max(hi_x);
  const float ref2 = hi_x > HILS_NEG_INF ? hi_x * HILS_LOG2E : 0.f;
  float l = 0.f;
#pragma unroll
  for (int nt = 0; nt < NB; ++nt)
#pragma unroll
    for (int i = 0; i < 4; ++i) l += __builtin_amdgcn_exp2f(fmaf(x[nt][i], HILS_LOG2E, -ref2));
  l = rows_sum(l);
  float lse_tot;
  {
    const float hils2 = (l > 0.f) ? ref2 + __builtin_amdgcn_logf(l) : HILS_NEG_INF;  // log2 domain
    const float swa2 = swa * HILS_LOG2E;
    const float mx = fmaxf(swa2, hils2), mn = fminf(swa2, hils2);
    float tot2 = mx;
    if (mn > HILS_NEG_INF) tot2 = mx + __builtin_amdgcn_logf(1.f + __builtin_amdgcn_exp2f(mn - mx));
    const float lt = tot2 * HILS_LN2;
    if (a.lse_total && j == 0 && ok) a.lse_total[row] = lt;
    lse_tot = tot2 > HILS_NEG_INF ? lt : 0.f;  // (all logits are -inf: -inf - -inf would be a NaN)
  }

  // ---- selection scores (compared as floats) and the number of finite ones ----
  float key[NB][4];
  int nvalid = 0;
#pragma unroll
  for (int nt = 0; nt < NB; ++nt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      key[nt][i] = __fsub_rn(x[nt][i], lse_tot);
      nvalid += key[nt][i] > HILS_NEG_INF ? 1 : 0;
    }
  nvalid = tc_rows_sum_i(nvalid);
  const float hi = __fsub_rn(hi_x, lse_tot);
  auto count_from = [&](float c) __attribute__((always_inline)) -> int {
    int n0 = 0, n1 = 0;
#pragma unroll
    for (int nt = 0; nt < NB; ++nt) {
      n0 += key[nt][0] >= c ? 1 : 0;
      n1 += key[nt][1] >= c ? 1 : 0;
      n0 += key[nt][2] >= c ? 1 : 0;
      n1 += key[nt][3] >= c ? 1 : 0;
    }
    return tc_rows_sum_i(n0 + n1);
  };

  // The winners are the scores from Tf up, except `cut` of a tie.  Invariants of a live query: more than K scores from lo
  // up (nlo of them), fewer than K from up up (nup), lo < up.
  constexpr float LOWEST = -3.402823466e38f;
  float Tf = LOWEST;  // a query that keeps all its scores
  bool live = nvalid > topk;
  bool tied = false;
  float lo = LOWEST, up = live ? tg_key_score(tg_score_key(hi) + 1u) : 0.f;
  int nlo = nvalid, nup = 0;
  if (__any(live)) {
    const float n_f = (float)nvalid, rn = __builtin_amdgcn_rcpf(n_f);
    const float z_max = tc_normal_quantile(0.56f * rn), z_k = tc_normal_quantile((float)topk * rn);
    // mean and deviation of normal scores with maximum 0 = mean + z_max sd and log mean exp = mean + sd^2 / 2
    const float lme = HILS_LN2 * __builtin_amdgcn_logf(l * rn), disc = fmaf(z_max, z_max, 2.f * lme);
    const float sd = disc > 0.f ? z_max - __builtin_amdgcn_sqrtf(disc) : z_max;
    float c = hi + sd * (z_k - z_max);
    for (int n = 1; __any(live); ++n) {
      bool chosen = n == 1;
      if (n > 2 && !__any(live & (nlo > topk + 1) & (nup < topk - 1))) {
        // one off everywhere: the smallest score from lo up is one too many, or the largest below up the one missing
        // (lo or up moves there with it, so that a tie leaves nothing between them)
        const bool drop = nlo == topk + 1;
        const uint32_t flip = drop ? 0u : 0x80000000u;
        const float bar = drop ? lo : tg_key_score(tg_score_key(-up) + 1u);
        float best = __builtin_inff();
#pragma unroll
        for (int nt = 0; nt < NB; ++nt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float y = __uint_as_float(__float_as_uint(key[nt][i]) ^ flip);
            best = fminf(best, y >= bar ? y : __builtin_inff());
          }
        best = -rows_max(-best);
        if (live) {
          const float at = drop ? best : -best, above = tg_key_score(tg_score_key(at) + 1u);
          c = drop ? above : at;
          if (drop) lo = at; else up = above;
        }
        chosen = true;
      }
      const uint32_t klo = tg_score_key(lo), kup = tg_score_key(up);
      const float mid = tg_key_score(klo + (kup - klo) / 2);
      if (!chosen) {
        if (n == 2) {
          const float p = (float)(nlo == nvalid ? nup : nlo) * rn;  // what the first probe counted
          c += sd * (z_k - tc_normal_quantile(fminf(fmaxf(p, 0.5f * rn), 1.f - 0.5f * rn)));
        } else if ((n & 3) == 0) {
          c = mid;
        } else {
          // (no lower probe yet: twice as far from the maximum as the last one)
          const float wl = (float)(nlo - topk), wu = (float)(topk - nup);
          c = lo > LOWEST ? lo + (up - lo) * (wl * __builtin_amdgcn_rcpf(wl + wu)) : up - 2.f * (hi - up);
        }
      }
      if (!(c > lo && c < up)) c = mid;
      // no score between them: the scores at lo are tied over the K-th place.  (Every fourth probe halves a range of
      // 2^32, so no finite scores come near the other limit; it ends the loop whatever the scores are.)
      const bool closed = kup - klo <= 1u || n > 200;
      const int cnt = count_from(c);
      if (live & closed) {
        Tf = lo;
        tied = true;
        live = false;
      }
      if (live) {
        if (cnt == topk) {
          Tf = c;
          live = false;
        } else if (cnt > topk) {
          lo = c;
          nlo = cnt;
        } else {
          up = c;
          nup = cnt;
        }
      }
    }
  }

  // ---- winner masks: bit nt*4 + i of the lane's words ----
  uint32_t mask[NM];
#pragma unroll
  for (int w = 0; w < NM; ++w) {
    uint32_t m = 0u;
#pragma unroll
    for (int e = 31; e >= 0; --e) m = (m << 1) | (key[w * 8 + e / 4][e & 3] >= Tf ? 1u : 0u);
    mask[w] = m;
  }
  if (__any(tied)) {
    // the scores equal to Tf beyond the lowest `need` chunk indices are taken out again
    int need = topk - nup, at = 0;  // `at`: ties at lower indices, over the lanes
#pragma unroll
    for (int nt = 0; nt < NB; ++nt) {
      int mine = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) mine += key[nt][i] == Tf ? 1 : 0;
      unsigned all;
      int before = at + (int)tc_rows_scan((unsigned)mine, j, all);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool eq = key[nt][i] == Tf;
        if (tied & eq & (before >= need)) mask[nt / 8] &= ~(1u << ((nt & 7) * 4 + i));
        before += eq ? 1 : 0;
      }
      at += (int)all;
    }
  }

  // ---- slots: winners in blocks before, in this block's lanes before, in this lane before ----
#pragma unroll
  for (int e = 0; e < 2; ++e) ((uint4*)stage)[e * 64 + lane] = make_uint4(0xffffff80u, 0xffffff80u, 0xffffff80u, 0xffffff80u);
  __builtin_amdgcn_wave_barrier();
  unsigned first = 0u;  // winners of the words before
#pragma unroll
  for (int w = 0; w < NM; ++w) {
    // counts per block in nibbles, the even and the odd blocks' in bytes (a query's block has at most 16)
    uint32_t n4 = mask[w] - ((mask[w] >> 1) & 0x55555555u);
    n4 = (n4 & 0x33333333u) + ((n4 >> 2) & 0x33333333u);
    unsigned tot_e, tot_o;
    const unsigned bef_e = tc_rows_scan(n4 & 0x0f0f0f0fu, j, tot_e), bef_o = tc_rows_scan((n4 >> 4) & 0x0f0f0f0fu, j, tot_o);
    const unsigned both = tot_e + tot_o;
    const unsigned pre = both * 0x01010100u + first * 0x01010101u;  // (bytes below 2^8: at most 128 + 32)
    const unsigned base_e = pre + bef_e, base_o = pre + tot_e + bef_o;
    first += (both * 0x01010101u) >> 24;
#pragma unroll
    for (int n8 = 0; n8 < 8; ++n8) {
      const int nt = w * 8 + n8;
      unsigned slot = (((n8 & 1) ? base_o : base_e) >> ((n8 >> 1) * 8)) & 255u;
      f32x4_t bv = {0.f, 0.f, 0.f, 0.f};
      if constexpr (BIAS) bv = *(const f32x4_t*)&bias_s[nt * 16 + 4 * j];  // the returned scores carry no bias
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if ((mask[w] >> (n8 * 4 + i)) & 1u) {
          const float raw = BIAS ? __fsub_rn(x[nt][i], bv[i]) : x[nt][i];
          if (slot < 32u) stage[col * 32 + slot] = (uint32_t)f2bf(raw) | ((uint32_t)(nt * 16 + 4 * j + i) << 16);
          ++slot;
        }
      }
    }
  }
  __builtin_amdgcn_wave_barrier();

  // ---- write out: indices (B,L,H,topk) int32, scores (B,L,H,1,topk) bf16 ----
  const long row0 = (b * a.L + t0) * (long)a.h_kv + hk;
#pragma unroll
  for (int e0 = 0; e0 < 16 * 32; e0 += 64) {
    const int e = e0 + lane, qi = e >> 5, k = e & 31;
    const uint32_t u = stage[e];
    if ((k < topk) & (t0 + qi < a.t_end)) {
      const long o = (row0 + (long)qi * a.h_kv) * topk + k;
      a.indices[o] = (int)u >> 16;  // (no winner: -1)
      a.scores[o] = (bf16_t)u;
    }
  }
}

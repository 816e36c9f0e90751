// Prefill top-k chunk selection, one pass over the chunk keys.
//
// One wavefront owns 16/GMAX consecutive queries of a (batch, KV head): the 16 rows of its MFMA
// tile are (queries x the GMAX heads of the KV head).  It streams the chunk keys once (B operands,
// 16 chunks per block, repacked into operand order by topk_pack_lmk_kernel) and keeps every scaled
// logit in registers: accumulator register i of block nt in lane (col, j) is row 4j+i, chunk
// nt*16+col, so a query's logits for up to 512 chunks lie in the 16 lanes of one lane row, 32 per
// lane (up to 1024: 64 per lane, one wavefront per SIMD).  From there, without touching memory again:
//   * the log-sum-exp of every row (in-lane maxima and sums, one 16-lane reduction per row),
//   * the selection score of every (query, chunk): max over the heads of logit - lse_total, a float
//     (in-lane: the heads of a query are registers of one lane),
//   * the top-K per query, the four lane rows working on four queries at once: the K-th largest
//     score is bracketed from the two largest scores of every lane (their minimum over the lanes is
//     a lower bound with at least 32 scores above it), the scores above the bound (about 1.5 K of
//     512) are compacted through LDS to at most 8 per lane (12 or 16 as records, from 32 blocks on), turned into order-preserving unsigned
//     keys, and the threshold is found on those by a bitwise search whose counts are 16-lane DPP
//     reductions (no ballots, no scalar round trip) and which stops at the first probe that counts
//     exactly K; ties at the threshold go to the lower chunk indices,
//   * the ascending order of the winners from the votes of the blocks (rank = winners voted before and in
//     lower columns) and their raw scores straight from the logits; with records (most kernels of 32 and 64 blocks) from a
//     map of the winning chunks in LDS and from the records.
// Five to eight query heads per KV head (HALF below) take two wavefronts per four queries, one for the
// heads 0..3 and one for the rest: each forms the partial selection scores of its heads, the two
// trade them through LDS, and both then select on the same scores and write their own heads' outputs.
// Covers G = 1..8, D in {64, 128}, N <= 1024, topk <= 32, an optional additive bias per
// (chunk, head) (the layer's prior bias), no Gumbel noise / drop mask; everything else runs on the
// kernels of topk.hip.  With a bias the registers hold the biased logits (what the log-sum-exp and
// the selection work on) and a winner's raw score is its logit minus the bias again.
#include "topk_group_kernel.h"
#include "topk_cols_kernel.h"

// plain: no Gumbel noise and no drop mask (a bias is fine)
bool hils_topk_group_covers(int N, int G, int D, int topk, int per_qhead, bool plain) {
  if (per_qhead && (G < 2 || G > 8)) return false;  // (one head a group: the keys are shared anyway)
  return plain && G >= 1 && G <= 8 && (D == 64 || D == 128) && N <= 16 * TG_NB && topk <= 32;
}

// queries that see 513 to 1024 chunks (topk_group_wide.hip)
void tg_launch_wide(int GM, int D, bool perq, bool half, bool exp, dim3 grid, hipStream_t st, const TgArgs& a);

// lmk_packed: the chunk keys in topk_pack_lmk_kernel's order.  The queries are split by how many
// chunks they can see (at most 8, 16, 24, 32 or 64 blocks of 16) into one launch each.
int hils_topk_group_launch(const void* q, const void* lmk_packed, const float* lse_swa, const float* bias,
                           int32_t* indices,
                           void* scores, float* lse_total, float* sel_logits, int B, int L, int N, int h_kv,
                           int G, int D, int topk, int block_size, int window_size, int causal, int q_offset,
                           float sm_scale, int lse_bf16, int per_qhead, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  // rows of a tile: queries x 1, 2 or 4 heads (three heads, and two with a key per query head, whose
  // wavefronts are one per head of four: padding rows)
  const int GM = (G == 1) ? 1 : ((G == 2 && !per_qhead) ? 2 : 4);
  const bool halves = G > 4;  // two wavefronts per four queries
  const int QGROUPS = halves ? (per_qhead ? 4 : 1) : (per_qhead ? 4 : TG_WAVES);  // wavefronts (pairs) of a workgroup with queries of their own
  const int NQ = 16 / GM;
  const bool exp = sel_logits != nullptr;
  auto limit_of = [&](int tq) -> int {
    int lm = causal ? visible_limit(tq + q_offset, window_size, block_size) : N;
    return lm < 0 ? 0 : (lm > N ? N : lm);
  };
  int t = 0;
  while (t < L) {
    // the bucket of query t and the last query that still falls into it (limits grow with t)
    int NB = exp && N <= 512 ? 32 : 64, t_hi = L;
    if (!exp) {
      const int lm = limit_of(t);
      NB = lm <= 128 ? 8 : (lm <= 256 ? 16 : (lm <= 384 ? 24 : (lm <= 512 ? 32 : 64)));
      if (NB < 64) {
        int lo = t, hi = L;  // first query whose limit exceeds 16 * NB
        while (lo < hi) {
          const int mid = lo + (hi - lo) / 2;
          if (limit_of(mid) <= 16 * NB) lo = mid + 1; else hi = mid;
        }
        t_hi = lo;
      }
    }
    dim3 grid((t_hi - t + NQ * QGROUPS - 1) / (NQ * QGROUPS), h_kv, B);
    const TgArgs a{(const bf16_t*)q, (const uint4*)lmk_packed, lse_swa, bias, indices, (bf16_t*)scores, lse_total,
                   sel_logits, L, N, h_kv, G, topk, block_size, window_size, causal, q_offset, sm_scale, t, t_hi, lse_bf16};
    if (GM == 1 && NB <= 16 && !exp) {
      // one head per KV head: queries as columns, 16 at once (B4 L8192 16/16 heads of 64, top-32: 174 -> 98 us; past 256
      // chunks two copies of the scores do not fit the registers)
      const int bs_shift = (block_size > 0 && (block_size & (block_size - 1)) == 0) ? __builtin_ctz(block_size) : -1;
      grid.x = (t_hi - t + 16 * TC_WAVES - 1) / (16 * TC_WAVES);
      auto cols = [&](auto ks, auto bi) {
        if (NB == 8) hipLaunchKernelGGL((topk_fwd_cols_kernel<ks.value, 8, bi.value>), grid, dim3(64 * TC_WAVES), 0, st, a, bs_shift);
        else hipLaunchKernelGGL((topk_fwd_cols_kernel<ks.value, 16, bi.value>), grid, dim3(64 * TC_WAVES), 0, st, a, bs_shift);
      };
      auto with_bias = [&](auto ks) {
        if (bias) cols(ks, std::true_type{}); else cols(ks, std::false_type{});
      };
      if (D == 64) with_bias(std::integral_constant<int, 2>{}); else with_bias(std::integral_constant<int, 4>{});
    } else if (NB == 64) {
      tg_launch_wide(GM, D, per_qhead != 0, halves, exp, grid, st, a);
    } else {
      tg_dispatch(GM, D, bias != nullptr, per_qhead != 0, halves, [&](auto gm, auto ks, auto bi, auto pq, auto hf) {
#define TG_NBS(NB_, EX_) tg_call<gm.value, ks.value, NB_, EX_, bi.value, pq.value, hf.value>(grid, st, a)
        if (exp) TG_NBS(32, true);
        else if (NB == 32) {
          // Records shorten a wavefront's serial chain, but with a bias and wide heads they spill: past one round of
          // wavefronts (two per SIMD, four workgroups a compute unit), where the instructions count, votes are ahead
          // (records / votes, 32/8 heads of 128, 512 chunks, top-8: 1024 queries 28.5 / 31.8 us, 1536 48.5 / 46.6,
          // 4096 94 / 91, 8192 168 / 159)
          if constexpr (gm.value == 4 && ks.value == 4 && bi.value && !pq.value && !hf.value) {
            if ((long)grid.x * grid.y * grid.z > 4L * hils_device_cus()) {
              tg_call<4, 4, 32, false, true, false, false, false>(grid, st, a);
              return;
            }
          }
          TG_NBS(32, false);
        }
        else if (NB == 24) TG_NBS(24, false);
        else if constexpr (gm.value > 1) {  // (one head: above)
          if (NB == 16) TG_NBS(16, false);
          else TG_NBS(8, false);
        }
#undef TG_NBS
      });
    }
    t = t_hi;
  }
  return HILS_OK;
}

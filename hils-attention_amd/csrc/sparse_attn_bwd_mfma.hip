// Sparse attention backward on bf16 MFMA (chunk size 64, D and Dv in {64, 128}).
//
// dK and dV of a chunk are sums over every (query, head) row that selected the chunk, so
// that side is computed chunk-major: an inverse index (for each (batch, KV head, chunk) the
// list of (query, slot) pairs that hold it) is built by a counting sort, then a workgroup per
// segment of a chunk's pairs streams its rows in rounds of 64, recomputes P and dS with the scores in the
// orientation rows x tokens, and keeps dK, dV of the chunk in MFMA accumulators: no atomics,
// one write per element (a chunk cut into several segments: one per segment, added up afterwards).
//
//   S  = Q K^T            (16x16x32 MFMA over d)
//   dP = dO V^T           (16x16x32 MFMA over dv)
//   P  = exp2(S c2 - lse2),  delta = sum_tokens P dP,  dS = w P (dP - delta)
//   dV += (w P)^T dO      (tokens x Dv, 16x16x32 MFMA over 32 rows)
//   dK += scale dS^T Q    (tokens x D,  16x16x32 MFMA over 32 rows)
//
// An accumulator-layout tile (lane: column = token, registers = rows 4j..4j+3) is, two row tiles
// side by side, exactly the A operand of the 16x16x32 MFMA with the roles (row m = token, k = 32
// rows), so P and dS feed the second pair of products without leaving registers.  Their B operands
// (k = rows, n = feature) are columns of the gathered Q and dO rows: the workgroup stages the rows
// row-major in LDS once per round for all four wavefronts, and the column reads
// are the hardware's transposing LDS loads (a 16-lane group fetches a 4 x 16 block and every lane
// receives one column of it).
#include "decode_rows.h"
#include "../../include/hils_amd.h"

#define BW_S 64
typedef short bw_s4 __attribute__((ext_vector_type(4)));
typedef unsigned bw_u4 __attribute__((ext_vector_type(4)));  // a 16-byte piece as a register value

__global__ void bw_fill_int_kernel(int* p, int value, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = value;
}

// ---------------------------------------------------------------------------
// Inverse index: pairs (query << 8 | slot) grouped by (batch, KV head, chunk).
// ---------------------------------------------------------------------------
// The index entries (query t_lo + r, slot s) of one KV head for the queries of a segment, walked by a
// workgroup of 1024: thread tid takes entries tid, tid + 1024, ... of the segment's rows x K entries
// (consecutive threads read consecutive slots of a row).  (r, s) advance by (1024 / K, 1024 % K) per
// step, so that nothing is divided inside the loop, and four loads are in flight per thread (a
// clamped row is loaded for a step past the end and skipped).  f(t, slot, chunk).
template <class F>
__device__ __forceinline__ void bw_walk_indices(const int32_t* __restrict__ seg0, int t_lo, int rows, int H, int K,
                                                F f) {
  const int qK = 1024 / K, rK = 1024 % K;
  int r = (int)threadIdx.x / K, sl = (int)threadIdx.x - r * K;
  const long rstride = (long)H * K;
  while (r < rows) {
    int rr[4], ss[4], cc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      rr[u] = r;
      ss[u] = sl;
      sl += rK;
      r += qK;
      if (sl >= K) { sl -= K; ++r; }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) cc[u] = seg0[(long)(rr[u] < rows ? rr[u] : rows - 1) * rstride + ss[u]];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (rr[u] < rows) f(t_lo + rr[u], ss[u], cc[u]);
  }
}

// counts[((b*H + h) * ranges + t / range) * nchunk + c] = number of valid entries equal to c; one workgroup per
// (batch, KV head, segment of queries of one range), LDS histogram first.
__global__ void __launch_bounds__(1024)
bw_count_kernel(const int32_t* __restrict__ indices, int* __restrict__ counts, int L, int H, int K,
                int nchunk, int seg_len, int range, int n_range) {
  extern __shared__ int hist[];
  const int h = blockIdx.y;
  const long b = blockIdx.z;
  const int t_lo = blockIdx.x * seg_len;
  const int t_hi = (t_lo + seg_len < L) ? t_lo + seg_len : L;
  for (int i = threadIdx.x; i < nchunk; i += 1024) hist[i] = 0;
  __syncthreads();
  const int32_t* seg0 = indices + ((b * L + t_lo) * H + h) * (long)K;
  bw_walk_indices(seg0, t_lo, t_hi - t_lo, H, K, [&](int, int, int c) {
    if (c >= 0 && c < nchunk) atomicAdd(&hist[c], 1);
  });
  __syncthreads();
  int* out = counts + ((b * H + h) * n_range + t_lo / range) * (long)nchunk;
  for (int i = threadIdx.x; i < nchunk; i += 1024)
    if (hist[i]) atomicAdd(&out[i], hist[i]);
}

// Work items of the dK/dV kernel (null: none wanted): every cell (batch, KV head, range of queries, chunk) is cut
// into segments of at most seg_pairs pairs.  With one range a cell is a chunk: one that is not cut is written by its
// item, which also zeroes the gradients of an empty one.  With several, every item leaves a partial result and an
// empty cell has none.
struct BwItems {
  int2* list;     // (cell, segment)
  int* total;     // number of items
  int* part_off;  // [cell] first partial result of a cell
  int seg_pairs;
  int n_range;
  __device__ __forceinline__ int segs(int x) const { return x > seg_pairs ? (x + seg_pairs - 1) / seg_pairs : n_range == 1 || x ? 1 : 0; }
};

// exclusive scan of n counts into offsets[0..n] (offsets[n] = total) and the item list; one workgroup, four
// counts per thread and step.  The arrays are 16-byte aligned and padded to a multiple of four entries.
__global__ void __launch_bounds__(1024)
bw_scan_kernel(const int* __restrict__ counts, int* __restrict__ offsets, int* __restrict__ cursor, int n, BwItems it) {
  __shared__ __align__(16) int wsum[3][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto parts = [&](int ns) -> int { return ns > 1 || it.n_range > 1 ? ns : 0; };
  int carry[3] = {0, 0, 0};  // pairs, items, partial results before this step's
  int4 next = tid * 4 < n ? *(const int4*)&counts[tid * 4] : make_int4(0, 0, 0, 0);
  for (int base = 0; base < n; base += 4096) {
    const int i0 = base + tid * 4;  // (the arrays are padded to whole groups of four)
    const int4 c4 = next;
    if (i0 + 4096 < n) next = *(const int4*)&counts[i0 + 4096];
    int x[4] = {0, 0, 0, 0};
    if (i0 < n) {
      x[0] = c4.x;
      x[1] = i0 + 1 < n ? c4.y : 0;
      x[2] = i0 + 2 < n ? c4.z : 0;
      x[3] = i0 + 3 < n ? c4.w : 0;
    }
    int s[3] = {0, 0, 0};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[0] += x[e];
      if (it.list && i0 + e < n) {
        const int ns = it.segs(x[e]);
        s[1] += ns;
        s[2] += parts(ns);
      }
    }
    int pos[3], incl[3] = {s[0], s[1], s[2]};
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        const int y = __shfl_up(incl[e], o, 64);
        if (lane >= o) incl[e] += y;
      }
    }
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      if (lane == 63) wsum[e][wave] = incl[e];
      pos[e] = carry[e] + incl[e] - s[e];
    }
    __syncthreads();
    // (all sums read at once and kept by every thread: two barriers a step; 18.8 -> 16.7 us for 16384 counts)
#pragma unroll
    for (int e = 0; e < 3; ++e) {
#pragma unroll
      for (int w = 0; w < 16; w += 4) {
        const int4 y = *(const int4*)&wsum[e][w];
        const int ys[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          pos[e] += w + u < wave ? ys[u] : 0;
          carry[e] += ys[u];
        }
      }
    }
    if (i0 < n) {
      int4 o4, p4;
      int* op = (int*)&o4;
      int* pp = (int*)&p4;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        op[e] = pos[0];
        pos[0] += x[e];
        pp[e] = pos[2];
        if (it.list && i0 + e < n) {
          const int ns = it.segs(x[e]);
          for (int k = 0; k < ns; ++k) it.list[pos[1] + k] = make_int2(i0 + e, k);
          pos[1] += ns;
          pos[2] += parts(ns);
        }
      }
      *(int4*)&offsets[i0] = o4;  // (offsets[n], when it lies in the group, is written below)
      *(int4*)&cursor[i0] = o4;
      if (it.list) *(int4*)&it.part_off[i0] = p4;
    }
    __syncthreads();
  }
  if (tid == 0) {
    offsets[n] = carry[0];
    if (it.list) *it.total = carry[1];
  }
}

// Pairs grouped by (b, h, c).  A workgroup reads its segment's entries once, at most BW_SCATTER / 1024 per thread, and
// takes every entry's place among its chunk's with an LDS atomic; one global atomic per chunk reserves the range in the
// chunk's list.  Written straight from there a wavefront's 64 entries go to 64 lines, and the L2's rate of requests
// bounds the kernel (33.5 M pairs, B8 L8192 16 KV heads, top-32, 128 chunks: 153 us).  STAGE: the pairs are laid out
// in LDS by chunk first and leave in runs.  With 8192 entries and 16 wavefronts 117 us; 101 with the workgroups of a
// unit on one XCD, whose L2 then merges the runs' partial lines; 61 with 4096 entries and 8 wavefronts (four workgroups
// on a compute unit, whose phases overlap; 71 with 2048 and 4).
#define BW_SCATTER 4096  // entries per workgroup
#define BW_SCATTER_NT 512
template <bool STAGE>
__global__ void __launch_bounds__(BW_SCATTER_NT)
bw_scatter_kernel(const int32_t* __restrict__ indices, int* __restrict__ cursor,
                  uint32_t* __restrict__ pairs, int L, int H, int K, int nchunk, int seg_len, int range, int n_range, int n_wg) {
  constexpr int NT = BW_SCATTER_NT, E = BW_SCATTER / NT;
  extern __shared__ __attribute__((aligned(16))) int bs_smem[];
  int* hist = bs_smem;               // [nchunk] entries of a chunk; then where they go, less their place in LDS (STAGE)
  int* first = hist + nchunk;        // [nchunk] a chunk's first place in LDS (STAGE)
  int2* out = (int2*)(bs_smem + ((2 * nchunk + 3) & ~3));  // [entry] pair, where it goes (STAGE)
  __shared__ int wsum[NT / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wg = (int)(blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8);  // (an XCD takes whole units)
  if (wg >= n_wg) return;
  const int nseg = (L + seg_len - 1) / seg_len;
  const int seg = wg % nseg, unit = wg / nseg;
  const int h = unit % H;
  const long b = unit / H;
  const int t_lo = seg * seg_len;
  const int rows = t_lo + seg_len < L ? seg_len : L - t_lo;
  int* cur = cursor + ((b * H + h) * n_range + t_lo / range) * (long)nchunk;
  const int32_t* seg0 = indices + ((b * L + t_lo) * H + h) * (long)K;
  const long rstride = (long)H * K;
  const int qK = NT / K, rK = NT % K;
  int r = tid / K, sl = tid - r * K;
  int cc[E], rank[E];
  uint32_t pr[E];
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const bool in = r < rows;
    const int c = seg0[(long)(in ? r : rows - 1) * rstride + sl];
    cc[u] = in && c >= 0 && c < nchunk ? c : -1;
    pr[u] = ((uint32_t)(t_lo + r) << 8) | (uint32_t)sl;
    sl += rK;
    r += qK;
    if (sl >= K) { sl -= K; ++r; }
  }
  for (int i = tid; i < nchunk; i += NT) hist[i] = 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < E; ++u)
    if (cc[u] >= 0) rank[u] = atomicAdd(&hist[cc[u]], 1);
  __syncthreads();
  if constexpr (!STAGE) {
    for (int i = tid; i < nchunk; i += NT) {
      const int cnt = hist[i];
      hist[i] = cnt ? atomicAdd(&cur[i], cnt) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < E; ++u)
      if (cc[u] >= 0) pairs[hist[cc[u]] + rank[u]] = pr[u];
    return;
  }
  int total = 0;
  for (int base = 0; base < nchunk; base += NT) {
    const int i = base + tid;
    const int cnt = i < nchunk ? hist[i] : 0;
    const int dst = cnt ? atomicAdd(&cur[i], cnt) : 0;
    int incl = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(incl, o, 64);
      if (lane >= o) incl += y;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int pos = total + incl - cnt;
    for (int w = 0; w < NT / 64; ++w) {
      const int x = wsum[w];
      pos += w < wave ? x : 0;
      total += x;
    }
    if (i < nchunk) {
      first[i] = pos;
      hist[i] = dst - pos;
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < E; ++u)
    if (cc[u] >= 0) {
      const int pos = first[cc[u]] + rank[u];
      out[pos] = make_int2((int)pr[u], hist[cc[u]] + pos);
    }
  __syncthreads();
  for (int i = tid; i < total; i += NT) pairs[out[i].y] = (uint32_t)out[i].x;
}

// ---------------------------------------------------------------------------
// dK, dV: one workgroup of four wavefronts per work item, a segment of the pairs of a (batch, KV head,
// chunk).  A chunk near the start of the sequence is selected two to three times as often as the average
// one, and with one workgroup per chunk and all of them resident at once the kernel ran as long as its
// fullest chunk (B2 L8192 32/4 heads of 64, top-32: 1300 us; in segments 1035).  The segments of
// a cut chunk leave fp32 partial results that bw_dkdv_sum_kernel adds up.
// Rows of many heads (16 MiB for these four KV heads' queries) are fetched again by every chunk: 5.3 GB past the L2.
// The items then go by ranges of queries (bw_range): 926 -> 735 us.  With the gathers as global instead of flat loads,
// whose data every wait for the LDS had waited for, and a round's reads ahead of its products: 712 us; B8 L8192 16/16
// heads of 64: 1435 -> 1400, vector ALU 42 % and matrix cores 29 % busy, LDS 42 %.
// ---------------------------------------------------------------------------
struct BwDims {
  int L, Lkv, HQ, H, K, NW, nchunk, mask_last;
  float sm_scale;
  int out16;  // dk, dv are bf16 tensors that this kernel overwrites (else fp32, added to)
  int B;
  const float* slope;  // per query head, or null: scores lose slope * max(0, 62 - token) before the softmax
  BwItems items;
  float* part;  // [partial result][64 tokens][D + DV]
};

// Tokens of a wavefront.  Every staged row is read (row-wise and column-wise) by each wavefront that has
// other tokens, and those LDS reads are what bounds the kernel: 144 KiB a round of 64 rows at D = 64 with
// 16 tokens per wavefront.  Narrow heads have the registers for 32: two wavefronts share the tokens, each
// takes half of the rows and the two add up at the end (80 KiB a round; two wavefronts per SIMD instead of
// four: held to 168 registers the kernel spills 63 and takes twice the time).  With one multiply-add per
// row address, delta as the start of the dP accumulators and the mask left to the output: 1527 -> 1439 us
// at B8 L8192 16/16 heads of 64, top-32, 1035 -> 930 at B2 L8192 32/4.
constexpr int bw_tt(int D, int DV) { return (D <= 64 && DV <= 64) ? 2 : 1; }

template <int D, int DV, int G>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
bw_dkdv_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
               const bf16_t* __restrict__ weights, const float* __restrict__ lse,
               const float* __restrict__ delta, const bf16_t* __restrict__ d_o,
               const int* __restrict__ offsets, const uint32_t* __restrict__ pairs,
               void* __restrict__ dk_out, void* __restrict__ dv_out, BwDims dm) {
  // delta (B,L,HQ,NW) fp32: sum_tokens P dP of every (row, slot), written by the dQ kernel
  constexpr int KS = D / 32, VS = DV / 32;    // k-steps of the two 16x16x32 products
  constexpr int DT = D / 16, VT = DV / 16;    // 16-wide column tiles of dK, dV
  constexpr int TT = bw_tt(D, DV);            // 16-token tiles of a wavefront
  constexpr int ROWS = 32 * TT;               // rows staged per round: 32 for each wavefront with the same tokens
  constexpr int PPR = ROWS / G;               // pairs per round
  // staging: padded row (bytes).  32 bytes: the 16-byte reads of 16 rows take 4 cycles, 8 with 16 (dK/dV at L32768 32/8 heads
  // of 128 4264 -> 3749 us, L8192 32/4 of 128 850 -> 768, B2 L8192 32/4 of 64 712 -> 688)
  constexpr int QROW = D * 2 + 32;
  constexpr int OROW = DV * 2 + 32;
  constexpr int BUF = ROWS * (QROW + OROW) + 3 * ROWS * 4;  // one staging buffer (bytes)
  extern __shared__ __attribute__((aligned(16))) char bw_smem[];  // two staging buffers
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, j = lane >> 4;
  // XCD-aware order: hardware hands consecutive workgroup ids to the 8 XCDs in turn; an XCD works
  // through one contiguous share of the items, i.e. of the (batch, KV head) pairs, so the query and dO
  // rows that its workgroups gather (the same L rows for every chunk of the head) stay in its L2.
  const int n_items = *dm.items.total;
  const int vid = (int)(blockIdx.x % 8) * ((n_items + 7) / 8) + (int)(blockIdx.x / 8);
  if ((int)(blockIdx.x / 8) >= (n_items + 7) / 8 || vid >= n_items) return;
  const int2 item = dm.items.list[vid];
  const int cell = item.x, c = cell % dm.nchunk, unit = cell / dm.nchunk / dm.items.n_range;
  const int hk = unit % dm.H;
  const long b = unit / dm.H;
  const int c_lo = offsets[cell], c_hi = offsets[cell + 1];  // the cell's pairs
  const bool whole = dm.items.n_range == 1 && c_hi - c_lo <= dm.items.seg_pairs;
  const int p_lo = c_lo + item.y * dm.items.seg_pairs;
  const int p_hi = c_hi - p_lo <= dm.items.seg_pairs ? c_hi : p_lo + dm.items.seg_pairs;
  if (p_lo == p_hi) {
    if (dm.out16) {  // nobody selected the chunk: its gradients are zero
      bf16_t* dk16 = (bf16_t*)dk_out + ((b * dm.Lkv + (long)c * BW_S) * dm.H + hk) * D;
      bf16_t* dv16 = (bf16_t*)dv_out + ((b * dm.Lkv + (long)c * BW_S) * dm.H + hk) * DV;
      for (int i = tid; i < BW_S * (D / 8); i += 256)
        *(uint4*)(dk16 + (long)(i / (D / 8)) * dm.H * D + (i % (D / 8)) * 8) = make_uint4(0, 0, 0, 0);
      for (int i = tid; i < BW_S * (DV / 8); i += 256)
        *(uint4*)(dv16 + (long)(i / (DV / 8)) * dm.H * DV + (i % (DV / 8)) * 8) = make_uint4(0, 0, 0, 0);
    }
    return;
  }

  // this wavefront's 16 * TT tokens of the chunk as B operands (k = feature, n = token), and its rows
  const int tw = TT == 2 ? (wave & 1) : wave, rw = TT == 2 ? (wave >> 1) : 0;
  uint4 kb[TT][KS], vb[TT][VS];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) {
    const long tok = (long)c * BW_S + tw * (16 * TT) + tt * 16 + col;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      kb[tt][ks] = *(const uint4*)(k + ((b * dm.Lkv + tok) * dm.H + hk) * D + ks * 32 + j * 8);
#pragma unroll
    for (int ks = 0; ks < VS; ++ks)
      vb[tt][ks] = *(const uint4*)(v + ((b * dm.Lkv + tok) * dm.H + hk) * DV + ks * 32 + j * 8);
  }

  f32x4_t acc_k[TT][DT], acc_v[TT][VT];
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) {
#pragma unroll
    for (int t = 0; t < DT; ++t) acc_k[tt][t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < VT; ++t) acc_v[tt][t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  }
  const float c2 = dm.sm_scale * HILS_LOG2E;

  // Staging roles: thread -> (row, 16-byte piece), NQ (NO) items per thread and round.
  constexpr int QPP = D / 8, OPP = DV / 8;
  constexpr int NQ = ROWS * QPP / 256, NO = ROWS * OPP / 256;
  constexpr int QRS = 256 / QPP, ORS = 256 / OPP;  // row step between a thread's items
  const int q_row0 = tid / QPP, q_pc = tid % QPP;
  const int o_row0 = tid / OPP, o_pc = tid % OPP;
  const int npair = p_hi - p_lo;
  const int nround = (npair + PPR - 1) / PPR;

  // Loads below are unconditional from clamped addresses, the pair entries as relaxed atomic
  // loads: a load inside a branch is waited for inside it, and a plain load may be moved next to
  // its use; either way the gathers of a round would queue up behind one another's latency.
  auto pair_ok = [&](int round, int row) __attribute__((always_inline)) -> bool {  // false for padding rows
    return row < ROWS && round * PPR + row / G < npair;
  };
  auto pair_of = [&](int round, int row) __attribute__((always_inline)) -> uint32_t {  // pair of a round's row (pair 0 of the chunk for padding rows)
    const int pi = round * PPR + row / G;
    return __hip_atomic_load(pairs + p_lo + (pair_ok(round, row) ? pi : 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  uint32_t pk_q[NQ], pk_o[NO], pk_r;
  bw_u4 xq[NQ], xo[NO];
  float r_l2 = INFINITY, r_dl = 0.f;
  bf16_t r_wb = 0;
  bool r_ok = false;
  auto load_pairs = [&](int round) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NQ; ++u) pk_q[u] = pair_of(round, q_row0 + u * QRS);
#pragma unroll
    for (int u = 0; u < NO; ++u) pk_o[u] = D == DV ? pk_q[u < NQ ? u : 0] : pair_of(round, o_row0 + u * ORS);  // (the same rows)
    pk_r = pair_of(round, tid);
  };
  // Row addresses are this lane's base plus query * stride, one 32 x 32 + 64 multiply-add each (the row
  // steps of a thread are multiples of 16: its head is the same for all its rows).
  static_assert(QRS % 16 == 0 && ORS % 16 == 0, "a thread stages rows of one head");
  const char* q_lane = (const char*)(q + (b * dm.L * (long)dm.HQ + hk * G + q_row0 % G) * D + q_pc * 8);
  const char* o_lane = (const char*)(d_o + (b * dm.L * (long)dm.HQ + hk * G + o_row0 % G) * DV + o_pc * 8);
  const long row_lane = b * dm.L * (long)dm.HQ + hk * G + (tid < ROWS ? tid % G : 0);  // (one address for the threads without a row)
  const float* l_lane = lse + row_lane * dm.K;
  const bf16_t* w_lane = weights + row_lane * dm.NW;
  const float* d_lane = delta + row_lane * dm.NW;
  const unsigned q_step = (unsigned)dm.HQ * D * 2u, o_step = (unsigned)dm.HQ * DV * 2u;
  const unsigned l_step = (unsigned)(dm.HQ * dm.K), w_step = (unsigned)(dm.HQ * dm.NW);
  // (as global pointers: an integer made a generic pointer is read by flat loads, which every wait for the LDS waits for)
  typedef const __attribute__((address_space(1))) bw_u4* bw_gptr;
  auto mad64 = [](unsigned a, unsigned b2, unsigned long c3) __attribute__((always_inline)) -> unsigned long {
    return (unsigned long)a * b2 + c3;
  };
  auto fetch = [&](int round) __attribute__((always_inline)) {  // gathers of `round`, whose pairs load_pairs(round) fetched
#pragma unroll
    for (int u = 0; u < NQ; ++u) {
      // padding rows read the row of the chunk's first pair (finite values): their P is 0, so they add nothing
      xq[u] = *(bw_gptr)mad64(pk_q[u] >> 8, q_step, (unsigned long)q_lane);
    }
#pragma unroll
    for (int u = 0; u < NO; ++u) {
      xo[u] = *(bw_gptr)mad64(pk_o[u] >> 8, o_step, (unsigned long)o_lane);
    }
    {
      // raw values; what a padding row gets instead is decided where they are staged, so that
      // nothing here has to wait for a load
      r_ok = pair_ok(round, tid);
      const uint32_t pk = pk_r;
      const unsigned long le = mad64(pk >> 8, l_step, pk & 255), we = mad64(pk >> 8, w_step, pk & 255);
      r_l2 = l_lane[le];
      r_wb = w_lane[we];
      r_dl = d_lane[we];
    }
  };
  // staging of the gathered rows of a round (in registers since fetch(round)) into buffer `buf`
  auto stage = [&](int buf) __attribute__((always_inline)) {
    char* q_rm = bw_smem + buf * BUF;       // ROWS x QROW
    char* o_rm = q_rm + ROWS * QROW;        // ROWS x OROW
    float* row_lse = (float*)(o_rm + ROWS * OROW);
    float* row_w = row_lse + ROWS;
    float* row_delta = row_w + ROWS;
#pragma unroll
    for (int u = 0; u < NQ; ++u) *(bw_u4*)(q_rm + (q_row0 + u * QRS) * QROW + q_pc * 16) = xq[u];
#pragma unroll
    for (int u = 0; u < NO; ++u) *(bw_u4*)(o_rm + (o_row0 + u * ORS) * OROW + o_pc * 16) = xo[u];
    if (tid < ROWS) {  // padding rows and empty slots: P = 0
      row_lse[tid] = (r_ok && r_l2 != HILS_NEG_INF) ? r_l2 : INFINITY;
      row_w[tid] = r_ok ? bf2f(r_wb) : 0.f;
      row_delta[tid] = r_ok ? -r_dl : 0.f;  // negated: the accumulators of dP start from it
    }
  };
  // column reads of a staged tile: rows r0 + 4j .. r0 + 4j + 3 of columns c0 .. c0 + 15, this
  // lane's column, and the same of the 16 rows behind.  (Transposing load: lane l of a 16-lane group addresses row l/4,
  // columns 4*(l%4) .. +3 of the 4 x 16 block and receives column l of it.)
  typedef short bw_tr4 __attribute__((ext_vector_type(4)));
  auto col_pair = [&](const char* base, int rowb, int r0, int c0) __attribute__((always_inline)) -> bw_u4 {
    const char* p = base + (r0 + 4 * j + (col >> 2)) * rowb + (c0 + 4 * (col & 3)) * 2;
    const uint2 a = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bw_tr4*)p));
    const uint2 b2 = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bw_tr4*)(p + 16 * rowb)));
    return (bw_u4){a.x, a.y, b2.x, b2.y};
  };
  load_pairs(0);
  fetch(0);
  load_pairs(1);
  stage(0);
  if (nround > 1) {
    fetch(1);
    load_pairs(2);
  }
  lds_barrier();

  for (int round = 0; round < nround; ++round) {
    const char* q_rm = bw_smem + (round & 1) * BUF;
    const char* o_rm = q_rm + ROWS * QROW;
    const float* row_lse = (const float*)(o_rm + ROWS * OROW);
    const float* row_w = row_lse + ROWS;
    const float* row_delta = row_w + ROWS;
    const int rows_here = ((npair - round * PPR < PPR) ? npair - round * PPR : PPR) * G;
    // This wavefront's two 16-row tiles: their P and dS, side by side, are the A operands (m = token,
    // k = 32 rows) of one 16x16x32 product per column tile and token tile; k index 8j + e stands for row
    // 4j + e of the first tile (e < 4) or row 4j + e - 4 of the second.
    // A SIMD holds two wavefronts and a round is a chain (rows, scores, exponentials, column reads, products): the
    // reads of a link are issued ahead of the link before it, fenced so that the scheduler does not sink them.
    const int r0 = rw * 32;
    if (r0 < rows_here) {
      bw_u4 qa[2][KS], oa[2][VS];
      f32x4_t l4[2], w4[2], d4[2];
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qa[h2][ks] = *(const bw_u4*)(q_rm + (r0 + h2 * 16 + col) * QROW + (ks * 32 + j * 8) * 2);
      }
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) {
        const int r = r0 + h2 * 16 + 4 * j;
        d4[h2] = *(const f32x4_t*)&row_delta[r];
#pragma unroll
        for (int ks = 0; ks < VS; ++ks) oa[h2][ks] = *(const bw_u4*)(o_rm + (r0 + h2 * 16 + col) * OROW + (ks * 32 + j * 8) * 2);
        l4[h2] = *(const f32x4_t*)&row_lse[r];
        w4[h2] = *(const f32x4_t*)&row_w[r];
      }
      __builtin_amdgcn_sched_barrier(0);
      // ---- S and dP of 32 rows x this wavefront's tokens
      f32x4_t s[2][TT], dp[2][TT];
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) s[h2][tt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
          for (int tt = 0; tt < TT; ++tt)
            s[h2][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, qa[h2][ks]), *(const bf16x8_t*)&kb[tt][ks], s[h2][tt], 0, 0, 0);
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) dp[h2][tt] = d4[h2];  // dP - delta
#pragma unroll
      for (int ks = 0; ks < VS; ++ks)
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
          for (int tt = 0; tt < TT; ++tt)
            dp[h2][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, oa[h2][ks]), *(const bf16x8_t*)&vb[tt][ks], dp[h2][tt], 0, 0, 0);
      if (dm.slope) {  // distance penalty (16 % G == 0: row 4j + i is the same head in every 16-row tile)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float sl = dm.slope[hk * G + (4 * j + i) % G];
#pragma unroll
          for (int tt = 0; tt < TT; ++tt) {
            const int dist = BW_S - 2 - (tw * (16 * TT) + tt * 16 + col);
            s[0][tt][i] -= sl * (float)(dist > 0 ? dist : 0);
            s[1][tt][i] -= sl * (float)(dist > 0 ? dist : 0);
          }
        }
      }
      bw_u4 bo[VT], bq[DT];
#pragma unroll
      for (int t = 0; t < VT; ++t) bo[t] = col_pair(o_rm, OROW, r0, t * 16);
      __builtin_amdgcn_sched_barrier(0);
      uint4 a_p[TT], a_ds[TT];
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        // accumulator layout: column = token `col`, registers = rows 4j..4j+3
        uint2 xp[2], xds[2];
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2) {
          float pv[4], ds[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) pv[i] = __builtin_amdgcn_exp2f(fmaf(s[h2][tt][i], c2, -l4[h2][i]));
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            pv[i] *= w4[h2][i];
            ds[i] = pv[i] * dp[h2][tt][i];
          }
          xp[h2].x = pack_bf2(pv[0], pv[1]);
          xp[h2].y = pack_bf2(pv[2], pv[3]);
          xds[h2].x = pack_bf2(ds[0], ds[1]);
          xds[h2].y = pack_bf2(ds[2], ds[3]);
        }
        a_p[tt] = make_uint4(xp[0].x, xp[0].y, xp[1].x, xp[1].y);
        a_ds[tt] = make_uint4(xds[0].x, xds[0].y, xds[1].x, xds[1].y);
      }
      // ---- dV += (wP)^T dO, dK += dS^T Q: contraction over the 32 rows
#pragma unroll
      for (int t = 0; t < DT; ++t) bq[t] = col_pair(q_rm, QROW, r0, t * 16);
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
          acc_v[tt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t*)&a_p[tt], __builtin_bit_cast(bf16x8_t, bo[t]), acc_v[tt][t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
          acc_k[tt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t*)&a_ds[tt], __builtin_bit_cast(bf16x8_t, bq[t]), acc_k[tt][t], 0, 0, 0);
    }
    // the next round's rows (gathered while this round computed) go to the other buffer, which
    // was last read a round ago (before the previous barrier); its gathers follow
    if (round + 1 < nround) {
      stage((round + 1) & 1);
      if (round + 2 < nround) {
        fetch(round + 2);
        load_pairs(round + 3);
      }
    }
    lds_barrier();
  }
  // The two wavefronts with the same tokens add up their row halves: each hands the token tile that the
  // other keeps over through LDS (the last round's barrier is behind the staging buffers' last use).
  constexpr int NT = DT + VT;
  static_assert(TT == 1 || 4 * NT * 64 * 16 <= 2 * BUF, "the exchange fits the staging buffers");
  f32x4_t* xch = (f32x4_t*)bw_smem;  // [wavefront][column tile][lane]
  auto give = [&](const f32x4_t (&ak)[DT], const f32x4_t (&av)[VT]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < DT; ++t) xch[(wave * NT + t) * 64 + lane] = ak[t];
#pragma unroll
    for (int t = 0; t < VT; ++t) xch[(wave * NT + DT + t) * 64 + lane] = av[t];
  };
  // accumulators: column = feature t*16 + col, rows = tokens 4j + i of the tile
  auto finish = [&](f32x4_t (&ak)[DT], f32x4_t (&av)[VT], int tok0) __attribute__((always_inline)) {
    if constexpr (TT == 2) {
      const int other = wave ^ 2;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const f32x4_t x = xch[(other * NT + t) * 64 + lane];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (t < DT) ak[t < DT ? t : 0][i] += x[i];
          else av[t < DT ? 0 : t - DT][i] += x[i];
        }
      }
    }
    // a masked last token's own row of sums is the only place its probabilities went: it becomes 0 here
    if (dm.mask_last && tok0 == BW_S - 16 && j == 3) {
#pragma unroll
      for (int t = 0; t < DT; ++t) ak[t][3] = 0.f;
#pragma unroll
      for (int t = 0; t < VT; ++t) av[t][3] = 0.f;
    }
    if (!whole) {
      float* out = dm.part + (long)(dm.items.part_off[cell] + item.y) * (BW_S * (D + DV));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float* row = out + (tok0 + 4 * j + i) * (D + DV) + col;
#pragma unroll
        for (int t = 0; t < DT; ++t) row[t * 16] = ak[t][i];
#pragma unroll
        for (int t = 0; t < VT; ++t) row[D + t * 16] = av[t][i];
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const long tk = (long)c * BW_S + tok0 + 4 * j + i;
      const long rk = ((b * dm.Lkv + tk) * dm.H + hk) * D, rv = ((b * dm.Lkv + tk) * dm.H + hk) * DV;
      if (dm.out16) {
        bf16_t* dkr = (bf16_t*)dk_out + rk;
        bf16_t* dvr = (bf16_t*)dv_out + rv;
#pragma unroll
        for (int t = 0; t < DT; ++t) dkr[t * 16 + col] = f2bf(ak[t][i] * dm.sm_scale);
#pragma unroll
        for (int t = 0; t < VT; ++t) dvr[t * 16 + col] = f2bf(av[t][i]);
      } else {
        float* dkr = (float*)dk_out + rk;
        float* dvr = (float*)dv_out + rv;
#pragma unroll
        for (int t = 0; t < DT; ++t) dkr[t * 16 + col] += ak[t][i] * dm.sm_scale;
#pragma unroll
        for (int t = 0; t < VT; ++t) dvr[t * 16 + col] += av[t][i];
      }
    }
  };
  if constexpr (TT == 2) {
    if (rw == 0) give(acc_k[1], acc_v[1]); else give(acc_k[0], acc_v[0]);
    lds_barrier();
    if (rw == 0) finish(acc_k[0], acc_v[0], tw * 32); else finish(acc_k[1], acc_v[1], tw * 32 + 16);
  } else {
    finish(acc_k[0], acc_v[0], tw * 16);
  }
}

// The partial results of the cut chunks, four features per thread, ranges and their segments in order.  Their bytes are
// the floor; the loads of four ranges' first segments, then of a range's others, are in flight together (one after the
// other / so: 16.4 / 7.0 us at B1 L2048 16/2 heads of 64, top-32, 33 / 31 in ranges at B2 L8192 32/4).
template <int D, int DV>
__global__ void __launch_bounds__(256)
bw_dkdv_sum_kernel(const int* __restrict__ offsets, void* __restrict__ dk_out, void* __restrict__ dv_out, BwDims dm) {
  const int c = blockIdx.x % dm.nchunk, unit = blockIdx.x / dm.nchunk;
  const int nr = dm.items.n_range;
  const int cell0 = unit * nr * dm.nchunk + c;  // of the first range
  if (nr == 1 && offsets[cell0 + 1] - offsets[cell0] <= dm.items.seg_pairs) return;
  const int hk = unit % dm.H;
  const long b = unit / dm.H;
  constexpr int F4 = (D + DV) / 4, N = BW_S * F4;
  constexpr int U = 4;  // loads in flight
  for (int i = blockIdx.y * 256 + threadIdx.x; i < N; i += gridDim.y * 256) {
    f32x4_t x = {0.f, 0.f, 0.f, 0.f};
    auto add = [&](const f32x4_t& y) {
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] += y[e];
    };
    for (int r0 = 0; r0 < nr; r0 += U) {
      int ns[U];
      const f32x4_t* src[U];
      f32x4_t first[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int cell = cell0 + (r0 + u < nr ? r0 + u : r0) * dm.nchunk;
        ns[u] = r0 + u < nr ? dm.items.segs(offsets[cell + 1] - offsets[cell]) : 0;
        src[u] = (const f32x4_t*)(dm.part + (long)dm.items.part_off[cell] * (BW_S * (D + DV))) + i;
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (ns[u]) first[u] = *src[u];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (ns[u]) add(first[u]);
        int k = 1;
        for (; k + 1 < ns[u]; k += U) {
          f32x4_t y[U];
#pragma unroll
          for (int w = 0; w < U; ++w) y[w] = src[u][(long)(k + w < ns[u] ? k + w : k) * N];
#pragma unroll
          for (int w = 0; w < U; ++w)
            if (k + w < ns[u]) add(y[w]);
        }
        if (k < ns[u]) add(src[u][(long)k * N]);
      }
    }
    const int t = i / F4, f = (i - t * F4) * 4;
    const long row = (b * dm.Lkv + (long)c * BW_S + t) * dm.H + hk;
    const bool is_k = f < D;
    const float sc = is_k ? dm.sm_scale : 1.f;
    const long o = is_k ? row * D + f : row * DV + f - D;
    void* out = is_k ? dk_out : dv_out;
    if (dm.out16) {
      uint2 pk;
      pk.x = pack_bf2(x[0] * sc, x[1] * sc);
      pk.y = pack_bf2(x[2] * sc, x[3] * sc);
      *(uint2*)((bf16_t*)out + o) = pk;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) ((float*)out)[o + e] += x[e] * sc;
    }
  }
}

// ---------------------------------------------------------------------------
// dQ, dW: query-block-major, like the forward kernel.  One workgroup owns T consecutive
// queries of a (batch, KV head), sorts the T*K (query, slot) pairs by chunk in LDS, and its
// wavefronts take chunks from a shared counter.  Per 16-row tile of a visit, with the scores
// in the orientation tokens x rows:
//   S^T  = K Q^T,  dP^T = V dO^T      (16x16x32 MFMAs, K and V of the chunk as A operands)
//   P = exp2(S c2 - lse2), delta = sum_tokens P dP (= dW of the pair), dS = w P (dP - delta)
//   dQ  += scale dS K                 (dS^T in accumulator layout is the A operand; K of the chunk
//                                      pre-transposed as B operand)
// dQ tiles are added into an LDS tile of the block as 32-bit fixed point (integer LDS atomics),
// scaled by a power of two from the bound  scale * 2 * max_row(sum_k|w| * |dO|_1) * max|V| * max|K|.
// ---------------------------------------------------------------------------
#define BQ_THREADS 512
#define BQ_STAGE_THREADS 768
#define BQ_MAXP 16  // (query, slot) pairs of a block per thread

struct BqDims {
  int L, Lkv, HQ, H, B, K, NW, T, nblk, nchunk, mask_last;
  float sm_scale;
  const float* slope;  // as in BwDims
  uint32_t k_magic;    // hils_udiv_magic(K)
};

typedef __attribute__((address_space(3))) int bq_lds_int;

// Rows behind the output tile that padding rows add to: as many as one address serves (the heads of a query among the
// four rows of a lane group).
constexpr int bq_spare(int G) { return G < 4 ? G : 4; }

// floor(x + 0.5) as an integer, one instruction (__float2int_rn is two).  The compiler counts no wait states between a
// matrix product and inline assembly that reads its result: bq_settle waits out the 12 behind the last one.
__device__ __forceinline__ void bq_settle(f32x4_t (&a)[4]) {
  asm volatile("s_nop 11" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]));
}
__device__ __forceinline__ int bq_round(float x) {
  int i;
  asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(i) : "v"(x));
  return i;
}

// a tile's rows, this lane's: pair (query of the block << 8 | slot), pieces of its q and dO, lse, weight
template <int KS, int VS>
struct BqRows {
  bw_u4 q[KS], o[VS];
  float l2;
  bf16_t wb;
  unsigned pk;
};

// STAGE: the block's own query and dO rows are copied into LDS once (coalesced) and every tile
// takes its row operands from there instead of gathering them from global memory once per (row,
// slot) pair (narrow heads; bq_stage_pays has the rule).  A tile is vector-ALU and LDS work with a matrix product at
// either end, one wavefront's pieces hardly overlap, so the rows' short way from the LDS buys a third wavefront per
// SIMD: their registers are loaded at their use, S before dP, and 12 wavefronts of at most 168 registers run instead of
// 8.  B8 L8192 16/16 heads of 64, top-32, dQ: 1800 us with the rows off their 16-byte boundaries (a ds_read_b128 then
// takes three times as long), 1550 on them, 1530 with 200 vector instructions a tile for 259 (row addresses without
// clamps in full tiles, one-instruction rounding, nothing copied between tiles), 1480 with 12 wavefronts; 280 of it are
// the block's set-up and end.
template <int D, int DV, int G, bool STAGE, int NT>
__global__ void __launch_bounds__(NT)
bw_dq_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ d_o, const bf16_t* __restrict__ ka,
             const bf16_t* __restrict__ va, const bf16_t* __restrict__ kt, const float* __restrict__ vmax,
             const float* __restrict__ kmax, const bf16_t* __restrict__ weights,
             const int32_t* __restrict__ indices, const float* __restrict__ lse, bf16_t* __restrict__ dq,
             float* __restrict__ dw, BqDims dm) {
  constexpr int KS = D / 32, VS = DV / 32;
  constexpr int DT = D / 16;
  constexpr int QT = 16 / G;
  constexpr int MAXP = BQ_MAXP;
  extern __shared__ __align__(16) int smem_i[];  // (16-byte row pieces are read from it)
  const int R = dm.T * G;
  constexpr int SPARE = bq_spare(G);
  int* q_acc = smem_i;                       // (R + SPARE) x D fixed point; padding rows add to the last SPARE
  int* cur = q_acc + (size_t)(R + SPARE) * D;  // nchunk: histogram -> running ends
  unsigned short* pairs = (unsigned short*)(cur + ((dm.nchunk + 3) & ~3));  // T*K pairs (query << 8 | slot) grouped by chunk (T, K <= 256)
  constexpr int QROWB = D * 2 + 16, OROWB = DV * 2 + 16;       // staged rows, padded (bytes)
  char* rows_q = (char*)pairs + (((size_t)dm.T * dm.K * 2 + 15) & ~(size_t)15);  // STAGE: R x QROWB
  char* rows_o = rows_q + (size_t)R * QROWB;                                     //        R x OROWB
  __shared__ float red[32];
  __shared__ int scan_s[NT / 64];
  __shared__ int next_s;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, j = lane >> 4;
  const int total = dm.nblk * dm.H * dm.B;
  const int per_xcd = (total + 7) / 8;
  const int vid = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  if (vid >= total) return;
  const int unit = vid / dm.nblk;
  const int blk = dm.nblk - 1 - (vid - unit * dm.nblk);
  const int hk = unit % dm.H;
  const long b = unit / dm.H;
  const int t0 = blk * dm.T;
  const int K = dm.K;
  const int npair = dm.T * K;

  // selected chunk of every (query, slot) pair of the block
  int creg[MAXP], preg[MAXP];
#pragma unroll
  for (int e = 0; e < MAXP; ++e) {
    const int i = tid + e * NT;
    int c = -1;
    preg[e] = 0;
    if (i < npair) {
      const int ql = (int)hils_udiv((uint32_t)i, (uint32_t)K, dm.k_magic), slot = i - ql * K;
      preg[e] = (ql << 8) | slot;
      if (t0 + ql < dm.L) c = indices[((b * dm.L + t0 + ql) * dm.H + hk) * (long)K + slot];
    }
    if (c < 0 || c >= dm.nchunk) c = -1;
    creg[e] = c;
  }
  // row bound: sum_k |w| * |dO|_1
  float rb = 0.f;
  for (int row = tid; row < R; row += NT) {
    const int ql = row / G, g = row - ql * G;
    if (t0 + ql < dm.L) {
      const long rowi = (b * dm.L + t0 + ql) * (long)dm.HQ + hk * G + g;
      const float a = hils_abs_row_sum_bf16(weights, rowi * dm.NW, K, (long)dm.B * dm.L * dm.HQ * dm.NW);
      float l1 = 0.f;
#pragma unroll
      for (int p8 = 0; p8 < DV / 8; ++p8) {
        float f[8];
        unpack8(*(const uint4*)(d_o + rowi * DV + p8 * 8), f);
#pragma unroll
        for (int e = 0; e < 8; ++e) l1 += fabsf(f[e]);
      }
      rb = fmaxf(rb, a * l1);
    }
  }
  for (int i = tid; i < (R + SPARE) * D; i += NT) q_acc[i] = 0;
  for (int i = tid; i < dm.nchunk; i += NT) cur[i] = 0;
  if (tid == 0) next_s = 0;
  if (STAGE) {
    // rows beyond the sequence end are never addressed by a pair: they re-read the last row.  Four
    // loads in flight per thread and none inside a branch (a load inside a branch is waited for there).
    auto stage_rows = [&](const bf16_t* src, char* dst, int rowb, int npc) __attribute__((always_inline)) {
      const int n = R * npc;
      for (int i0 = 0; i0 < n; i0 += 4 * NT) {
        bw_u4 t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int i = i0 + u * NT + tid;
          const int ic = i < n ? i : n - 1;
          const int row = ic / npc, pc = ic - row * npc;
          int tq = t0 + row / G;
          tq = tq < dm.L ? tq : dm.L - 1;
          t[u] = *(const bw_u4*)(src + ((b * dm.L + tq) * (long)dm.HQ + hk * G + row % G) * (npc * 8) + pc * 8);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int i = i0 + u * NT + tid;
          if (i < n) {
            const int row = i / npc, pc = i - row * npc;
            *(bw_u4*)(dst + row * rowb + pc * 16) = t[u];
          }
        }
      }
    };
    stage_rows(q, rows_q, QROWB, D / 8);
    stage_rows(d_o, rows_o, OROWB, DV / 8);
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < MAXP; ++e)
    if (creg[e] >= 0) atomicAdd(&cur[creg[e]], 1);
  rb = block_max(rb, red);  // barrier: histogram complete
  float vm = 0.f, km = 0.f;
  const int per_thr = (dm.nchunk + NT - 1) / NT;
  const int c_lo = tid * per_thr;
  int local = 0;
  for (int c = c_lo; c < c_lo + per_thr && c < dm.nchunk; ++c) {
    const int h = cur[c];
    if (h > 0) {
      // (the sign marks a chunk with a NaN or an infinity)
      vm = fmaxf(vm, fabsf(vmax[(b * dm.H + hk) * (long)dm.nchunk + c]));
      km = fmaxf(km, fabsf(kmax[(b * dm.H + hk) * (long)dm.nchunk + c]));
    }
    local += h;
  }
  int incl = local;
#pragma unroll
  for (int o2 = 1; o2 < 64; o2 <<= 1) {
    const int x = __shfl_up(incl, o2, 64);
    if (lane >= o2) incl += x;
  }
  if (lane == 63) scan_s[wave] = incl;
  vm = block_max(vm, red);  // barrier: scan_s visible, all histogram reads done
  km = block_max(km, red);
  int base = incl - local;
  for (int w2 = 0; w2 < wave; ++w2) base += scan_s[w2];
  for (int c = c_lo; c < c_lo + per_thr && c < dm.nchunk; ++c) {
    const int h = cur[c];
    cur[c] = base;
    base += h;
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < MAXP; ++e)
    if (creg[e] >= 0) pairs[atomicAdd(&cur[creg[e]], 1)] = (unsigned short)preg[e];
  __syncthreads();  // now chunk c owns pairs[cur[c-1] .. cur[c])

  const float bound = 2.f * dm.sm_scale * rb * vm * km;
  float fx_scale = 1.f;
  if (bound > 0.f && bound < 3.0e38f) {
    int e2 = 28 - ilogbf(bound);
    e2 = e2 > 90 ? 90 : (e2 < -90 ? -90 : e2);
    fx_scale = ldexpf(1.f, e2);
  }
  const float fx_inv = 1.f / fx_scale;
  const float c2 = dm.sm_scale * HILS_LOG2E;
  const float out_scale = dm.sm_scale * fx_scale;
  // rows of lse, weights and dw from the block's first query on, with 32-bit element offsets (hils_bw_run)
  const char* lse_blk = (const char*)(lse + (b * dm.L + t0) * (long)dm.HQ * K);
  const char* w_blk = (const char*)(weights + (b * dm.L + t0) * (long)dm.HQ * dm.NW);
  float* dw_blk = dw + (b * dm.L + t0) * (long)dm.HQ * dm.NW;
  const bf16_t* q_blk = q + (b * dm.L + t0) * (long)dm.HQ * D;
  const bf16_t* do_blk = d_o + (b * dm.L + t0) * (long)dm.HQ * DV;
  const int qs = r / G, g = r - qs * G;  // this lane's row of a tile: query slot, head
  const int hq = hk * G + g;
  const float sl = dm.slope ? dm.slope[hq] : 0.f;
  const unsigned l_row = (unsigned)(hq * K), w_row0 = (unsigned)(hq * dm.NW);  // ... of query 0 and this lane's head
  const unsigned l_step = (unsigned)(dm.HQ * K), w_step = (unsigned)(dm.HQ * dm.NW);
  const int npair_valid = cur[dm.nchunk - 1];
  // LDS addresses of this lane's column r in the four output rows of its lane group, for query 0 of the block (rows of
  // one query are consecutive heads: one address, up to SPARE rows from it), and in the spare rows
  unsigned acc_lane = (unsigned)(size_t)(bq_lds_int*)(q_acc + ((4 * j) % G) * D + r);
  unsigned spare_lane = (unsigned)(size_t)(bq_lds_int*)(q_acc + R * D + r);
  asm volatile("" : "+v"(acc_lane), "+v"(spare_lane));  // (kept as registers: or the constant parts are added per use)

  for (;;) {
    int c = 0;
    if (lane == 0) c = atomicAdd(&next_s, 1);
    c = __builtin_amdgcn_readfirstlane(c);
    if (c >= dm.nchunk) break;
    const int vs = c ? cur[c - 1] : 0;
    if (vs >= npair_valid) break;
    const int ve = cur[c];
    if (vs == ve) continue;
    const long chunk = (b * dm.H + hk) * (long)dm.nchunk + c;
    const bf16_t* ka_c = ka + chunk * (long)BW_S * D + lane * 8;
    const bf16_t* va_c = va + chunk * (long)BW_S * DV + lane * 8;
    const bf16_t* kt_c = kt + chunk * (long)BW_S * D + lane * 8;
    // Operands of the chunk: K and V as A operands of the two score products, K transposed as B
    // operand of dQ = dS K.  With 64-wide heads all three stay in registers for every tile of the
    // visit; wider heads reload them per tile (K transposed into the registers of the first set).
    constexpr bool KEEP = D <= 64 && DV <= 64;
    bw_u4 xa[4 * KS], ya[4 * VS], xt[KEEP ? 2 * DT : 1];
    if (KEEP) {
#pragma unroll
      for (int u = 0; u < 4 * KS; ++u) xa[u] = *(const bw_u4*)(ka_c + u * 512);
#pragma unroll
      for (int u = 0; u < 4 * VS; ++u) ya[u] = *(const bw_u4*)(va_c + u * 512);
#pragma unroll
      for (int u = 0; u < 2 * DT; ++u) xt[u] = *(const bw_u4*)(kt_c + u * 512);
    }
    auto load_rows = [&](int p, BqRows<KS, VS>& x) __attribute__((always_inline)) {
      const int last = ((ve - p < QT) ? ve - p : QT) - 1;  // padding rows repeat the tile's last pair
      x.pk = pairs[p + (qs < last ? qs : last)];
      const unsigned ql_r = x.pk >> 8, slot_r = x.pk & 255u;
      if (!STAGE) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          x.q[ks] = *(const bw_u4*)(q_blk + (__umul24(ql_r, (unsigned)(dm.HQ * D)) + (unsigned)(hq * D + ks * 32 + j * 8)));
#pragma unroll
        for (int ks = 0; ks < VS; ++ks)
          x.o[ks] = *(const bw_u4*)(do_blk + (__umul24(ql_r, (unsigned)(dm.HQ * DV)) + (unsigned)(hq * DV + ks * 32 + j * 8)));
      }
      // (byte offsets below 2^32: a uniform base and one register)
      x.l2 = *(const float*)(lse_blk + (__umul24(ql_r, l_step) + l_row + slot_r) * 4u);
      x.wb = *(const bf16_t*)(w_blk + (__umul24(ql_r, w_step) + w_row0 + slot_r) * 2u);
    };
    // one tile, its rows in x; the next tile's rows, if there is one, are loaded into nx behind its arithmetic
    auto tile = [&](int p, BqRows<KS, VS>& x, BqRows<KS, VS>& nx) __attribute__((always_inline)) {
      const int n = (ve - p < QT) ? ve - p : QT;  // pairs of the tile
      if (!KEEP) {
        load_rows(p, x);
#pragma unroll
        for (int u = 0; u < 4 * KS; ++u) xa[u] = *(const bw_u4*)(ka_c + u * 512);
#pragma unroll
        for (int u = 0; u < 4 * VS; ++u) ya[u] = *(const bw_u4*)(va_c + u * 512);
      }
      // (with staged rows always, a visit's last tile its own again: behind a branch the wait for these loads is one for the
      // next tile's too; B2 L8192 32/4 heads of 64 711 -> 664 us.  With gathered rows they cost more, 138 -> 144 at L8192 16/8)
      if (KEEP && (STAGE || p + QT < ve)) load_rows(p + QT < ve ? p + QT : p, nx);
      if (STAGE) {
        const unsigned row_l = (x.pk >> 8) * G + g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) x.q[ks] = *(const bw_u4*)(rows_q + row_l * QROWB + (ks * 32 + j * 8) * 2);
      }
      // LDS addresses of the output rows 4j .. 4j + 3, this lane's column
      constexpr int NP = G >= 4 ? 1 : 4 / G;  // pairs they belong to
      const unsigned short* op = pairs + p + (4 * j) / G;
      unsigned at[NP];
      if (n == QT) {
#pragma unroll
        for (int u = 0; u < NP; ++u) at[u] = __umul24((unsigned)op[u] >> 8, (unsigned)(G * D * 4)) + acc_lane;
      } else {  // padding rows add to the spare rows
        const int last = n - 1 - (4 * j) / G;
#pragma unroll
        for (int u = 0; u < NP; ++u) {
          const unsigned real = __umul24((unsigned)op[u <= last ? u : last] >> 8, (unsigned)(G * D * 4)) + acc_lane;
          at[u] = u <= last ? real : spare_lane;
        }
      }
      const float l2 = x.l2 == HILS_NEG_INF ? INFINITY : x.l2;
      // ---- S^T and dP^T: tokens x rows, four token tiles each
      f32x4_t st[4], dpt[4];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        st[mt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        dpt[mt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
          st[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, xa[mt * KS + ks]),
                                                           __builtin_bit_cast(bf16x8_t, x.q[ks]), st[mt], 0, 0, 0);
      if (STAGE) {
        __builtin_amdgcn_sched_barrier(0);
        const unsigned row_l = (x.pk >> 8) * G + g;
#pragma unroll
        for (int ks = 0; ks < VS; ++ks) x.o[ks] = *(const bw_u4*)(rows_o + row_l * OROWB + (ks * 32 + j * 8) * 2);
      }
#pragma unroll
      for (int ks = 0; ks < VS; ++ks)
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
          dpt[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ya[mt * VS + ks]),
                                                            __builtin_bit_cast(bf16x8_t, x.o[ks]), dpt[mt], 0, 0, 0);
      if (!KEEP) {  // K of the chunk as B operand of dQ = dS K replaces the first operand set
#pragma unroll
        for (int u = 0; u < 2 * DT; ++u) xa[u] = *(const bw_u4*)(kt_c + u * 512);
      }
      if (dm.slope) {
        float sl_v = sl;
        int j_v = j;
        asm volatile("" : "+v"(sl_v), "+v"(j_v) : : "memory");  // (a branch that keeps no registers between tiles)
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int dist = BW_S - 2 - (mt * 16 + j_v * 4 + i);
            st[mt][i] -= sl_v * (float)(dist > 0 ? dist : 0);
          }
      }
      // ---- P, delta, dS (this lane: row r of the tile, tokens mt*16 + 4j + i)
      float delta = 0.f;
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float pv = __builtin_amdgcn_exp2f(st[mt][i] * c2 - l2);
          st[mt][i] = pv;
          delta += pv * dpt[mt][i];
        }
      if (dm.mask_last && j == 3) {  // token 63 = tile 3, lane group 3, register 3
        delta -= st[3][3] * dpt[3][3];
        st[3][3] = 0.f;
      }
      delta = rows_sum(delta);
      if (j == 0 && qs < n) dw_blk[__umul24(x.pk >> 8, w_step) + w_row0 + (x.pk & 255u)] = delta;
      const float f = __uint_as_float((unsigned)x.wb << 16) * out_scale;
      bf16x8_t ap[2];
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        // (the difference first: a product rounded before the cancellation leaves its error behind)
        auto ds = [&](int mt, int i) __attribute__((always_inline)) { return f * st[mt][i] * (dpt[mt][i] - delta); };
        uint4 y;
        y.x = pack_bf2(ds(2 * s2, 0), ds(2 * s2, 1));
        y.y = pack_bf2(ds(2 * s2, 2), ds(2 * s2, 3));
        y.z = pack_bf2(ds(2 * s2 + 1, 0), ds(2 * s2 + 1, 1));
        y.w = pack_bf2(ds(2 * s2 + 1, 2), ds(2 * s2 + 1, 3));
        ap[s2] = __builtin_bit_cast(bf16x8_t, y);
      }
      // ---- dQ tile += dS K: four column tiles at a time
#pragma unroll
      for (int d0 = 0; d0 < DT; d0 += 4) {
        f32x4_t acc[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[u] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const bw_u4 kb2 = KEEP ? xt[KEEP ? (d0 + u) * 2 + s2 : 0] : xa[(d0 + u) * 2 + s2];
            acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ap[s2], __builtin_bit_cast(bf16x8_t, kb2), acc[u], 0, 0, 0);
          }
        bq_settle(acc);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            __hip_atomic_fetch_add((bq_lds_int*)(at[i * NP / 4] + (unsigned)((i % (4 / NP)) * D + (d0 + u) * 16) * 4u),
                                   bq_round(acc[u][i]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    };
    BqRows<KS, VS> xa_r, xb_r;
    if (KEEP) load_rows(vs, xa_r);
    for (int p = vs;;) {  // two row sets in turn: nothing is copied from one to the other
      tile(p, xa_r, xb_r);
      p += QT;
      if (p >= ve) break;
      tile(p, xb_r, xa_r);
      p += QT;
      if (p >= ve) break;
    }
  }
  __syncthreads();
  constexpr int C8 = D / 8;
  for (int i = tid; i < R * C8; i += NT) {
    const int row = i / C8, c8 = i - row * C8;
    const int ql = row / G, g2 = row - ql * G;
    const int t = t0 + ql;
    if (t < dm.L) {
      const int* src = q_acc + (size_t)row * D + c8 * 8;
      uint4 x;
      x.x = pack_bf2((float)src[0] * fx_inv, (float)src[1] * fx_inv);
      x.y = pack_bf2((float)src[2] * fx_inv, (float)src[3] * fx_inv);
      x.z = pack_bf2((float)src[4] * fx_inv, (float)src[5] * fx_inv);
      x.w = pack_bf2((float)src[6] * fx_inv, (float)src[7] * fx_inv);
      *(uint4*)(dq + ((b * dm.L + t) * (long)dm.HQ + hk * G + g2) * D + c8 * 8) = x;
    }
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static size_t bw_round(size_t n) { return (n + 255) & ~(size_t)255; }

// sm_n (an extra term in every chunk's softmax denominator) reaches the backward only through
// the saved per-chunk LSE, so any sm_n >= 0 is covered.
bool hils_bw_covers(int L, int Lkv, int HQ, int H, int D, int Dv, int K, int S, int q_block, int WH,
                    float sm_n, const float* slope) {
  if (H <= 0 || HQ % H != 0) return false;
  const int G = HQ / H;
  return S == BW_S && (D == 64 || D == 128) && (Dv == 64 || Dv == 128) &&
         (G == 1 || G == 2 || G == 4 || G == 8 || G == 16) && q_block == 1 && WH == HQ && sm_n >= 0.f &&
         Lkv >= S && K <= 256 && L < (1 << 24) && Lkv / S <= 12288;
}

void hils_bw_pack_launch(const void* k, const void* v, bf16_t* ka, bf16_t* va, bf16_t* kt, float* kmax, float* vmax,
                         int B, int Lkv, int H, int D, int Dv, void* stream);

// T queries per workgroup of the dQ kernel such that the fixed-point tile, the chunk histogram
// and the pair list (and, with `stage`, the block's own query and dO rows) fit in LDS; 0 when the
// shape does not fit.
static size_t bq_smem_bytes(int T, int G, int D, int Dv, int K, int nchunk, bool stage) {
  size_t n = (size_t)(T * G + bq_spare(G)) * D * 4 + (size_t)((nchunk + 3) & ~3) * 4 + (((size_t)T * K * 2 + 15) & ~(size_t)15);
  if (stage) n += (size_t)T * G * ((size_t)D * 2 + 16 + (size_t)Dv * 2 + 16);
  return n;
}
static int bq_pick_T(int L, int G, int D, int Dv, int K, int nchunk, bool stage, size_t* smem_out) {
  // the largest block that fits: the more rows share a visit, the fewer K/V bytes per row
  const size_t limit = 156 * 1024;
  const size_t per_q = (size_t)G * D * 4 + (size_t)K * 2 + (stage ? (size_t)G * ((size_t)(D + Dv) * 2 + 32) : 0);
  const size_t fixed = (size_t)bq_spare(G) * D * 4 + (size_t)((nchunk + 3) & ~3) * 4 + 16;  // spare rows, histogram, alignment
  if (fixed + per_q > limit) return 0;
  long T = (long)((limit - fixed) / per_q);
  if (T > 256) T = 256;  // a pair is (query << 8 | slot) in 16 bits
  if (T * K > BQ_MAXP * BQ_THREADS) T = (BQ_MAXP * BQ_THREADS) / K;
  if (T > L) T = L;
  if (T >= 8) T &= ~7L;
  if (T < 1) return 0;
  *smem_out = bq_smem_bytes((int)T, G, D, Dv, K, nchunk, stage);
  return (int)T;
}

struct BwLayout {
  size_t counts, offsets, cursor, pairs, ka, va, kt, vmax, kmax, items, n_items, part_off, part, total;
  int seg_pairs, range, n_range;
  size_t max_items;
};
// Queries per range of the dK/dV kernel: the gathered rows of a unit (batch, KV head) should stay in an XCD's L2 (4 MiB,
// and the workgroups of one range overlap with those of the next).  Where a unit's rows are more than 3 MiB the items go
// range by range of 2 MiB, at the price of a partial result of 64 (D + Dv) floats per (range, chunk): as many bytes,
// written and read, as the gathers of 256 rows, and ranges times chunks grow with the square of the length.  Hence only
// where such a cell has 1024 rows on average (a causal call reaches about half of the cells) and the partial results stay
// within 1 GiB; with fewer than eight units the XCDs share a unit's items, whose rows are unequal (the first ranges have
// few chunks and full cells), and it takes 2048.  Rows of one or two heads are bound by requests and gain nothing.
// Whole backward, us, one range / ranges of 2 MiB (in brackets, rows of a cell): top-32, B2 L8192 32/4 heads of 64 [2048]
// 1583 / 1449, B1 L8192 32/8 of 128 [1024] 1800 / 1759, B2 L8192 16/4 of 128 [1024] 1783 / 1757, B1 L16384 32/8 of 128
// [512] 3757 / 3984, L32768 [256] 9314 / 10019; few units: B1 L8192 16/2 of 64 [2048] 526 / 497, B1 L8192 32/4 of 128
// [1024] 1820 / 1908 (the rule costs here: B1 L16384 32/4 of 64 [1024] 1974 / 1859); top-8: B2 L8192 32/4 of 64 [512] 621 / 649, B1 L8192 32/8 of 128 [256] 726 / 790, B1 L16384 16/2 of 64
// [256] 396 / 481; one or two heads: B2 L16384 16/16 of 64 [1024] 1863 / 2056, B8 L8192 32/16 of 64 [2048] 5570 / 5965.
// Ranges of other lengths, dK/dV + sum, B2 L8192 32/4 of 64: 857 in ranges of 1 MiB, 806 of 2, 912 of 3, 914 of 4.
static int bw_range(size_t units, int L, int nchunk, int G, int D, int Dv, int K) {
  const size_t row = (size_t)G * (D + Dv) * 2;
  if (G < 4 || (size_t)L * row <= ((size_t)3 << 20)) return L;
  int r = (int)(((size_t)2 << 20) / row) & ~255;
  r = r > 256 ? r : 256;
  const size_t rows = (size_t)r * K * G / nchunk;  // of a cell
  const size_t parts = units * nchunk * ((L + r - 1) / r) * (BW_S * (size_t)(D + Dv) * 4);
  return rows >= (units >= 8 ? 1024u : 2048u) && parts <= ((size_t)1 << 30) ? r : L;
}
// Pairs per work item of the dK/dV kernel: about 2048 items of equal size in all (some four rounds of the
// workgroups that fit the chip), but no less than 512 rows (a cell may have fewer), whose gathers are four times the
// partial result's bytes.
static BwLayout bw_layout(int B, int L, int Lkv, int G, int H, int D, int Dv, int K) {
  const size_t chunks = (size_t)B * H * (Lkv / BW_S);
  const size_t pairs = (size_t)B * L * H * K;
  size_t seg = (pairs + 2047) / 2048;
  const size_t least = G < 8 ? 512 / G : 64;
  seg = ((seg > least ? seg : least) + 63) & ~(size_t)63;
  BwLayout lo;
  lo.range = bw_range((size_t)B * H, L, Lkv / BW_S, G, D, Dv, K);
  lo.n_range = (L + lo.range - 1) / lo.range;
  const size_t cells = chunks * lo.n_range;
  size_t o = 0;
  lo.counts = o; o += bw_round((cells + 1) * 4);
  lo.offsets = o; o += bw_round((cells + 1) * 4);
  lo.cursor = o; o += bw_round((cells + 1) * 4);
  lo.pairs = o; o += bw_round((size_t)B * L * H * K * 4);
  lo.ka = o; o += bw_round(chunks * BW_S * D * 2);
  lo.va = o; o += bw_round(chunks * BW_S * Dv * 2);
  lo.kt = o; o += bw_round(chunks * BW_S * D * 2);
  lo.vmax = o; o += bw_round(chunks * 4);
  lo.kmax = o; o += bw_round(chunks * 4);
  const bool cut = (size_t)lo.range > seg;  // (no cell has more pairs than its range queries unless one names a chunk twice)
  lo.seg_pairs = cut ? (int)seg : 0x7fffffff;
  lo.max_items = cells + (cut ? pairs / seg : 0);
  lo.items = o; o += bw_round(lo.max_items * sizeof(int2));
  lo.n_items = o; o += bw_round(4);
  lo.part_off = o; o += bw_round((cells + 1) * 4);
  // one range: a cell of n > seg pairs has ceil(n / seg) <= 2 n / seg partial results; several: every item has one
  const size_t parts = lo.n_range > 1 ? lo.max_items < pairs ? lo.max_items : pairs : cut ? 2 * (pairs / seg + 1) : 0;
  lo.part = o; o += bw_round(parts * BW_S * (size_t)(D + Dv) * 4);
  lo.total = o;
  return lo;
}

size_t hils_bw_workspace_bytes(int B, int L, int Lkv, int HQ, int H, int D, int Dv, int K, int S,
                               int q_block, int WH, float sm_n) {
  if (!hils_bw_covers(L, Lkv, HQ, H, D, Dv, K, S, q_block, WH, sm_n, nullptr)) return 0;
  size_t smem;
  if (bq_pick_T(L, HQ / H, D, Dv, K, Lkv / S, false, &smem) == 0) return 0;
  return bw_layout(B, L, Lkv, HQ / H, H, D, Dv, K).total;
}

template <int D, int DV>
static int bw_launch_dkdv(int G, dim3 grid, hipStream_t st, const bf16_t* q, const bf16_t* k,
                          const bf16_t* v, const bf16_t* w, const float* lse, const float* delta,
                          const bf16_t* d_o, const int* offsets, const uint32_t* pairs, void* dk, void* dv,
                          const BwDims& dm) {
#define BW_CALL(G_)                                                                                         \
  do {                                                                                                      \
    auto kern = bw_dkdv_kernel<D, DV, G_>;                                                                  \
    static HilsLdsReserve reserved;                                                                         \
    if (int rc = hils_reserve_lds(&reserved, (const void*)kern, smem, "hils_sparse_attn_bwd")) return rc;   \
    hipLaunchKernelGGL(kern, grid, dim3(256), smem, st, q, k, v, w, lse, delta, d_o, offsets, pairs, dk, dv, dm); \
  } while (0)
  constexpr size_t ROWS = 32 * bw_tt(D, DV);
  const size_t smem = 2 * (ROWS * (D * 2 + 32) + ROWS * (DV * 2 + 32) + 3 * ROWS * sizeof(float));  // two staging buffers
  switch (G) {
    case 1: BW_CALL(1); break;
    case 2: BW_CALL(2); break;
    case 4: BW_CALL(4); break;
    case 8: BW_CALL(8); break;
    case 16: BW_CALL(16); break;
    default: return -1;
  }
#undef BW_CALL
  if (dm.items.n_range > 1 || dm.items.seg_pairs != 0x7fffffff)  // some chunk may have been cut
    hipLaunchKernelGGL((bw_dkdv_sum_kernel<D, DV>), dim3((unsigned)((long)dm.B * dm.H * dm.nchunk), 8), dim3(256), 0, st,
                       offsets, dk, dv, dm);
  return HILS_OK;
}

template <int D, int DV, int G, bool STAGE, int NT>
static int bq_launch(dim3 grid, size_t smem, hipStream_t st, const bf16_t* q, const bf16_t* d_o,
                     const bf16_t* ka, const bf16_t* va, const bf16_t* kt, const float* vmax,
                     const float* kmax, const bf16_t* w, const int32_t* idx, const float* lse, bf16_t* dq,
                     float* dw, const BqDims& dm) {
  auto kern = bw_dq_kernel<D, DV, G, STAGE, NT>;
  static HilsLdsReserve reserved;  // per instantiation
  if (int rc = hils_reserve_lds(&reserved, (const void*)kern, smem, "hils_sparse_attn_bwd")) return rc;
  hipLaunchKernelGGL(kern, grid, dim3(NT), smem, st, q, d_o, ka, va, kt, vmax, kmax, w, idx, lse, dq, dw, dm);
  return HILS_OK;
}

template <int D, int DV>
static int bq_dispatch_g(int G, bool stage, dim3 grid, size_t smem, hipStream_t st, const bf16_t* q,
                         const bf16_t* d_o, const bf16_t* ka, const bf16_t* va, const bf16_t* kt,
                         const float* vmax, const float* kmax, const bf16_t* w, const int32_t* idx,
                         const float* lse, bf16_t* dq, float* dw, const BqDims& dm) {
  if constexpr (D <= 64 && DV <= 64) {
    if (stage) switch (G) {
      case 1: return bq_launch<D, DV, 1, true, BQ_STAGE_THREADS>(grid, smem, st, q, d_o, ka, va, kt, vmax, kmax, w, idx, lse, dq, dw, dm);
      case 2: return bq_launch<D, DV, 2, true, BQ_STAGE_THREADS>(grid, smem, st, q, d_o, ka, va, kt, vmax, kmax, w, idx, lse, dq, dw, dm);
      case 4: return bq_launch<D, DV, 4, true, BQ_STAGE_THREADS>(grid, smem, st, q, d_o, ka, va, kt, vmax, kmax, w, idx, lse, dq, dw, dm);
      case 8: return bq_launch<D, DV, 8, true, BQ_STAGE_THREADS>(grid, smem, st, q, d_o, ka, va, kt, vmax, kmax, w, idx, lse, dq, dw, dm);
      case 16: return bq_launch<D, DV, 16, true, BQ_STAGE_THREADS>(grid, smem, st, q, d_o, ka, va, kt, vmax, kmax, w, idx, lse, dq, dw, dm);
      default: return -1;
    }
  }
  switch (G) {
    case 1: return bq_launch<D, DV, 1, false, BQ_THREADS>(grid, smem, st, q, d_o, ka, va, kt, vmax, kmax, w, idx, lse, dq, dw, dm);
    case 2: return bq_launch<D, DV, 2, false, BQ_THREADS>(grid, smem, st, q, d_o, ka, va, kt, vmax, kmax, w, idx, lse, dq, dw, dm);
    case 4: return bq_launch<D, DV, 4, false, BQ_THREADS>(grid, smem, st, q, d_o, ka, va, kt, vmax, kmax, w, idx, lse, dq, dw, dm);
    case 8: return bq_launch<D, DV, 8, false, BQ_THREADS>(grid, smem, st, q, d_o, ka, va, kt, vmax, kmax, w, idx, lse, dq, dw, dm);
    case 16: return bq_launch<D, DV, 16, false, BQ_THREADS>(grid, smem, st, q, d_o, ka, va, kt, vmax, kmax, w, idx, lse, dq, dw, dm);
  }
  return -1;
}

// Staging the block's rows in LDS halves the block or more (its rows take as much as its output tile), but the rows of
// all blocks of an XCD together would not stay in its L2 beside the operands, and every (row, slot) pair gathers one:
// gathered / staged, dQ alone at B2 L8192, 4 KV heads of 64, top-32: 236 / 202 us with 2 query heads per KV head,
// 514 / 382 with 4, 785 / 650 with 8, 1646 / 1283 with 16.  Calls whose gathering blocks fit one round of the chip keep
// them (B1 L3001 32/4: 96 / 107 us, B2 L1024 16/2: 24.6 / 26.5).  Wide heads have no registers for a visit's operands
// and no room for the rows.
static bool bq_stage_pays(long units, int L, int G, int D, int Dv, int K, int nchunk) {
  if (D > 64 || Dv > 64) return false;
  size_t a, b2;
  const int t_plain = bq_pick_T(L, G, D, Dv, K, nchunk, false, &a);
  const int t_stage = bq_pick_T(L, G, D, Dv, K, nchunk, true, &b2);
  return t_plain > 0 && t_stage > 0 && units * ((L + t_plain - 1) / t_plain) > hils_device_cus();
}

// Inverse index of an index tensor (B, L, H, K) with values in [0, nchunk) or < 0: counts,
// offsets (cells + 1 ints, cells = B*H*nchunk), cursor (scratch) and the pairs (t << 8 | slot)
// grouped by (b, h, chunk).  Also used by the top-k backward.
static int bw_build_index(const int32_t* indices, int* counts, int* offsets, int* cursor, uint32_t* pairs,
                           const BwItems& items, int B, int L, int H, int K, int nchunk, int range, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  const int n_range = (L + range - 1) / range;
  const long cells = (long)B * H * nchunk * n_range;
  {
    const long n = cells + 1;
    hipLaunchKernelGGL(bw_fill_int_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, counts, 0, n);
  }
  // segments of queries per workgroup: short enough for a few thousand workgroups (the LDS atomics of
  // a workgroup on one chunk's counter serialise), long enough that a workgroup's one global atomic per
  // chunk stays cheap
  int seg_len = n_range > 1 ? 256 : L;  // (a segment lies in one range)
  while ((long)B * H * ((L + seg_len - 1) / seg_len) < 4096 && seg_len > 128) seg_len = (seg_len + 1) / 2;
  dim3 gs((L + seg_len - 1) / seg_len, H, B);
  hipLaunchKernelGGL(bw_count_kernel, gs, dim3(1024), (size_t)nchunk * 4, st, indices, counts, L, H, K, nchunk, seg_len, range, n_range);
  hipLaunchKernelGGL(bw_scan_kernel, dim3(1), dim3(1024), 0, st, counts, offsets, cursor, (int)cells, items);
  // The scatter keeps a segment's entries in registers.  Staging them pays where a chunk has several of them and where
  // there are many (direct / staged: 33.5 M pairs 153 / 61 us, 2 M 13.1 / 8.8, 128 K 4.6 / 5.5, 16 K 3.8 / 5.0).
  while ((long)seg_len * K > BW_SCATTER && seg_len > 1) seg_len = (seg_len + 1) / 2;
  const long n_wg = (long)B * H * ((L + seg_len - 1) / seg_len);
  const dim3 gc((unsigned)((n_wg + 7) / 8 * 8));
  const size_t staged = (size_t)((2 * nchunk + 3) & ~3) * 4 + (size_t)seg_len * K * sizeof(int2);
  if ((long)B * L * H * K >= 1 << 19 && (long)seg_len * K >= 4L * nchunk && staged <= 80 * 1024) {
    static HilsLdsReserve reserved;
    if (int rc = hils_reserve_lds(&reserved, (const void*)bw_scatter_kernel<true>, staged, "hils_sparse_attn_bwd")) return rc;
    hipLaunchKernelGGL(bw_scatter_kernel<true>, gc, dim3(BW_SCATTER_NT), staged, st, indices, cursor, pairs, L, H, K, nchunk, seg_len, range, n_range, (int)n_wg);
  } else {
    hipLaunchKernelGGL(bw_scatter_kernel<false>, gc, dim3(BW_SCATTER_NT), (size_t)nchunk * 4, st, indices, cursor, pairs, L, H, K, nchunk, seg_len, range, n_range, (int)n_wg);
  }
  return HILS_OK;
}

int hils_build_chunk_index(const int32_t* indices, int* counts, int* offsets, int* cursor, uint32_t* pairs,
                           int B, int L, int H, int K, int nchunk, void* stream) {
  return bw_build_index(indices, counts, offsets, cursor, pairs, BwItems{nullptr, nullptr, nullptr, 0, 1}, B, L, H, K,
                        nchunk, L, stream);
}

// Whole backward on the MFMA kernels: dq (bf16, written), dw (fp32, written at the valid slots),
// dk / dv (fp32, accumulated into the caller's buffers; or, with kv16, bf16 tensors that are overwritten).
int hils_bw_run(const void* q, const void* k, const void* v, const void* weights, const int32_t* indices,
                const float* slope, const float* lse, const void* d_o, void* dq, void* dk, void* dv,
                float* dw, void* workspace, int B, int L, int Lkv, int HQ, int H, int D, int Dv, int K, int NW,
                float sm_scale, int mask_last, int kv16, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  const int nchunk = Lkv / BW_S;
  const BwLayout lo = bw_layout(B, L, Lkv, HQ / H, H, D, Dv, K);
  char* ws = (char*)workspace;
  int* counts = (int*)(ws + lo.counts);
  int* offsets = (int*)(ws + lo.offsets);
  int* cursor = (int*)(ws + lo.cursor);
  uint32_t* pairs = (uint32_t*)(ws + lo.pairs);
  bf16_t* ka = (bf16_t*)(ws + lo.ka);
  bf16_t* va = (bf16_t*)(ws + lo.va);
  bf16_t* kt = (bf16_t*)(ws + lo.kt);
  float* vmax = (float*)(ws + lo.vmax);
  float* kmax = (float*)(ws + lo.kmax);
  const int G = HQ / H;
  if (H > 65535 || B > 65535 || (size_t)B * H * nchunk * lo.n_range > (1u << 30)) return -1;
  // (24-bit row strides and 32-bit offsets inside a block of up to 256 queries)
  if ((long)HQ * (D > Dv ? D : Dv) >= (1 << 23) || (long)HQ * NW >= (1 << 22) || (long)HQ * K >= (1 << 22)) return -1;
  hils_bw_pack_launch(k, v, ka, va, kt, kmax, vmax, B, Lkv, H, D, Dv, stream);  // operands of the dQ kernel
  // ---- dQ, dW
  {
    size_t smem;
    const bool stage = bq_stage_pays((long)B * H, L, G, D, Dv, K, nchunk);
    int T = bq_pick_T(L, G, D, Dv, K, nchunk, stage, &smem);
    if (T == 0) return -1;
    // small problems: rather a block for every compute unit than the largest blocks (64 blocks of 64 queries ->
    // 256 of 16 at B2 L1024 16/2 heads of 64: 63 -> 26 us)
    const long cus = hils_device_cus(), units = (long)B * H, per_unit = cus / units;
    if (units * ((L + T - 1) / T) < cus && per_unit > 0) {
      const long t = ((L + per_unit - 1) / per_unit + 7) & ~7L;
      if (t < T) T = (int)t;
      smem = bq_smem_bytes(T, G, D, Dv, K, nchunk, stage);
    }
    const int nblk = (L + T - 1) / T;
    const long total = (long)nblk * H * B;
    if (total > (1L << 30)) return -1;
    BqDims dm{L, Lkv, HQ, H, B, K, NW, T, nblk, nchunk, mask_last, sm_scale, slope, hils_udiv_magic((uint32_t)K)};
    dim3 grid((unsigned)(((total + 7) / 8) * 8));
    int rc = -1;
#define BQ_D(D_, DV_)                                                                                 \
  rc = bq_dispatch_g<D_, DV_>(G, stage, grid, smem, st, (const bf16_t*)q, (const bf16_t*)d_o, ka, va, kt, vmax, \
                              kmax, (const bf16_t*)weights, indices, lse, (bf16_t*)dq, dw, dm)
    if (D == 64 && Dv == 64) BQ_D(64, 64);
    else if (D == 128 && Dv == 128) BQ_D(128, 128);
    else if (D == 64 && Dv == 128) BQ_D(64, 128);
    else if (D == 128 && Dv == 64) BQ_D(128, 64);
#undef BQ_D
    if (rc != HILS_OK) return rc;
  }
  // ---- inverse index, then dK, dV
  const BwItems items{(int2*)(ws + lo.items), (int*)(ws + lo.n_items), (int*)(ws + lo.part_off), lo.seg_pairs, lo.n_range};
  if (int rc = bw_build_index(indices, counts, offsets, cursor, pairs, items, B, L, H, K, nchunk, lo.range, stream)) return rc;
  BwDims dm{L, Lkv, HQ, H, K, NW, nchunk, mask_last, sm_scale, kv16, B, slope, items, (float*)(ws + lo.part)};
  if (kv16 && Lkv > nchunk * BW_S) {  // tokens behind the last whole chunk are never attended
    for (int b2 = 0; b2 < B; ++b2) {
      const long nk = (long)(Lkv - nchunk * BW_S) * H * D / 2, nv = (long)(Lkv - nchunk * BW_S) * H * Dv / 2;
      int* pk = (int*)((bf16_t*)dk + ((long)b2 * Lkv + (long)nchunk * BW_S) * H * D);
      int* pv = (int*)((bf16_t*)dv + ((long)b2 * Lkv + (long)nchunk * BW_S) * H * Dv);
      hipLaunchKernelGGL(bw_fill_int_kernel, dim3((unsigned)((nk + 255) / 256)), dim3(256), 0, st, pk, 0, nk);
      hipLaunchKernelGGL(bw_fill_int_kernel, dim3((unsigned)((nv + 255) / 256)), dim3(256), 0, st, pv, 0, nv);
    }
  }
  const long grid_n = ((long)lo.max_items + 7) / 8 * 8;
  if (grid_n > 2147483647L) return -1;
  dim3 grid((unsigned)grid_n);
  int rc = -1;
#define BW_D(D_, DV_)                                                                              \
  rc = bw_launch_dkdv<D_, DV_>(G, grid, st, (const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v,   \
                               (const bf16_t*)weights, lse, dw, (const bf16_t*)d_o, offsets, pairs, dk, dv, dm)
  if (D == 64 && Dv == 64) BW_D(64, 64);
  else if (D == 128 && Dv == 128) BW_D(128, 128);
  else if (D == 64 && Dv == 128) BW_D(64, 128);
  else if (D == 128 && Dv == 64) BW_D(128, 64);
#undef BW_D
  return rc;
}

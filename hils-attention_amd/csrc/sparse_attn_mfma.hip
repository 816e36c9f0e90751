// Sparse attention forward on bf16 MFMA for prefill-sized query counts.
//
// The work is regrouped by chunk, not by query.  One workgroup owns T consecutive queries
// of one (batch, KV head).  It sorts the T*K (query, slot) pairs by chunk index in LDS, so
// that all queries of the block that selected chunk c sit next to each other ("a visit").
// A wavefront takes up to 16/G queries of a visit (16 rows: queries x the G heads of the
// KV head), loads the chunk's K rows and the gathered query rows straight into MFMA
// operands, forms S^T = K Q^T (tokens x rows) with 16x16x32 MFMAs, does the per-chunk
// softmax along the accumulator registers, and feeds P back as the A operand of
// O = P V without leaving registers (the contraction order over tokens is permuted to
// the accumulator layout; V is pre-transposed per chunk in the same order).  The
// (rows x Dv) partial outputs are summed into a fixed-point output tile in LDS with integer
// LDS atomics, which is what lets rows of different visits be arbitrary subsets of the block.
// What fixed point cannot hold is kept out of it: a block that visits a chunk with a NaN or an
// infinity in V (or meets such a weight) sums in floating point instead, and a row whose softmax
// is not a number comes out as NaN.
#include "common.h"
#include "../../include/hils_amd.h"
#include <type_traits>

#define GA_THREADS 512
#ifndef GA_THREADS_NARROW
#define GA_THREADS_NARROW 768  // D = Dv = 64
#endif
#define GA_WAVES (GA_THREADS / 64)
#define GA_S 64                 // chunk size this kernel is built for
#define GA_MAXP 16              // (query, slot) pairs of a block per thread
#define GA_KEY_INVALID 0xFFFFFFFFu
#define GA_PAIR_BITS 12

// ---------------------------------------------------------------------------
// Operand packing.  Each 64-token chunk of K and V of a (batch, KV head) is rewritten once
// into the exact register order of the 16x16x32 MFMA operands the forward kernel needs, so
// that every operand load of a wavefront is one contiguous 1 KiB burst (8 full cache lines)
// instead of 16 half-used lines at a 2*H*D-byte stride:
//   kp[chunk][mt][ks][lane][8] = K[token mt*16 + (lane&15)][d = ks*32 + (lane>>4)*8 + e]
//   vp[chunk][dt][s][lane][8]  = V[token tok(s, lane>>4, e)][dv = dt*16 + (lane&15)]
// with tok(s, j, e) = 32*s + 16*(e/4) + 4*j + e%4, the order in which an accumulator-layout
// P supplies tokens when it is fed back as the A operand of O = P V.
// Also records max|V| of every chunk (it bounds the fixed-point output accumulation), NaNs left out,
// with the sign bit set when the chunk holds a NaN or an infinity.
// BWD: what the backward's dQ kernel needs, in one pass over K and V: kp, vp in the order of kp, kt = K
// in the order that vp has otherwise, and both maxima.
//
// Memory-bound.  Every 16-byte piece of the chunk is loaded once, all of a thread's before any is used, in
// the order of kp; the transposed matrix goes by way of row-major rows in LDS and the transposing load.
// B8 L8192 16 heads of 64: 89 us (6.0 TB/s; the chunks' bytes one by one through LDS: 90), the backward's arrays
// 123 us (two passes of 90); B1 L2048 2 heads 5.1 -> 3.7 us.
// ---------------------------------------------------------------------------
template <int D, int DV, bool BWD>
__global__ void __launch_bounds__(256)
pack_kv_kernel(const bf16_t* __restrict__ k, const bf16_t* __restrict__ v, bf16_t* __restrict__ kp,
               bf16_t* __restrict__ vp, bf16_t* __restrict__ kt, float* __restrict__ kmax, float* __restrict__ vmax,
               int Lkv, int H, int nchunk) {
  typedef short pk_s4 __attribute__((ext_vector_type(4)));
  typedef short pk_s8 __attribute__((ext_vector_type(8)));
  constexpr int DT = BWD ? D : DV, PITCH = DT * 2 + 16;  // the transposed matrix
  constexpr int NK = D / 32, NV = DV / 32;               // pieces of a thread
  __shared__ __align__(16) unsigned char tile[GA_S * PITCH];
  __shared__ uint32_t red[2][4];  // largest magnitude, bit 31: not all numbers
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 15, j = lane >> 4;
  const int c = blockIdx.x, h = blockIdx.y;
  const long b = blockIdx.z;
  const long chunk = (b * H + h) * (long)nchunk + c;
  const long row0 = (b * Lkv + (long)c * GA_S) * H + h;
  // (piece i of a matrix: ((mt * KS + ks) * 64 + lane), a wavefront's u-th at i = u * 256 + tid)
  uint4 kx[NK], vx[NV];
#pragma unroll
  for (int u = 0; u < NK; ++u) {
    const int blk = u * 4 + wave;
    kx[u] = *(const uint4*)(k + (row0 + (long)(blk / (D / 32) * 16 + col) * H) * D + blk % (D / 32) * 32 + j * 8);
  }
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int blk = u * 4 + wave;
    vx[u] = *(const uint4*)(v + (row0 + (long)(blk / (DV / 32) * 16 + col) * H) * DV + blk % (DV / 32) * 32 + j * 8);
  }
  const auto& tx = [&]() -> const auto& { if constexpr (BWD) return kx; else return vx; }();
#pragma unroll
  for (int u = 0; u < DT / 32; ++u) {
    const int blk = u * 4 + wave;
    *(uint4*)(tile + (blk / (DT / 32) * 16 + col) * PITCH + blk % (DT / 32) * 64 + j * 16) = tx[u];
  }
#pragma unroll
  for (int u = 0; u < NK; ++u) *(uint4*)(kp + chunk * (long)GA_S * D + (long)(u * 256 + tid) * 8) = kx[u];
  if constexpr (BWD) {
#pragma unroll
    for (int u = 0; u < NV; ++u) *(uint4*)(vp + chunk * (long)GA_S * DV + (long)(u * 256 + tid) * 8) = vx[u];
  }
  // ---- maxima (bf16 bits: the order of the magnitudes)
  auto largest = [&](const auto& x, int m) {
    uint32_t mx = 0, odd = 0;
    for (const uint4& y : x) {
      const uint32_t w[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t mag = (e & 1 ? w[e / 2] >> 16 : w[e / 2]) & 0x7fffu;
        odd |= mag >= 0x7f80u;
        mx = mag <= 0x7f80u && mag > mx ? mag : mx;
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const uint32_t y = __shfl_xor((int)mx, o, 64);
      mx = y > mx ? y : mx;
    }
    const bool any = __ballot(odd != 0) != 0;
    if (lane == 0) red[m][wave] = mx | (any ? 0x80000000u : 0u);
  };
  largest(vx, 0);
  if constexpr (BWD) largest(kx, 1);
  __syncthreads();
  if (tid < (BWD ? 2 : 1)) {
    uint32_t mx = 0, odd = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint32_t x = red[tid][w], m = x & 0x7fffffffu;
      odd |= x & 0x80000000u;
      mx = m > mx ? m : mx;
    }
    const float top = __uint_as_float(mx << 16);
    (tid ? kmax : vmax)[chunk] = odd ? -top : top;
  }
  // ---- transposed: piece ((dt * 2 + s) * 64 + lane)
  bf16_t* out = (BWD ? kt : vp) + chunk * (long)GA_S * DT;
#pragma unroll
  for (int u = 0; u < DT / 32; ++u) {
    const int blk = u * 4 + wave, dt = blk >> 1, s = blk & 1;
    const unsigned char* p = tile + (32 * s + 4 * j + (col >> 2)) * PITCH + (col & 3) * 8 + dt * 32;
    const pk_s4 y0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) pk_s4*)p);
    const pk_s4 y1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) pk_s4*)(p + 16 * PITCH));
    *(uint4*)(out + (long)(u * 256 + tid) * 8) = __builtin_bit_cast(uint4, (pk_s8)__builtin_shufflevector(y0, y1, 0, 1, 2, 3, 4, 5, 6, 7));
  }
}

template <bool BWD>
static void pack_kv_launch(const void* k, const void* v, bf16_t* kp, bf16_t* vp, bf16_t* kt, float* kmax, float* vmax,
                           int B, int Lkv, int H, int D, int Dv, hipStream_t st) {
  const int nchunk = Lkv / GA_S;
#define PACK(D_, DV_)                                                                                              \
  hipLaunchKernelGGL((pack_kv_kernel<D_, DV_, BWD>), dim3(nchunk, H, B), dim3(256), 0, st, (const bf16_t*)k,       \
                     (const bf16_t*)v, kp, vp, kt, kmax, vmax, Lkv, H, nchunk)
  if (D == 64 && Dv == 64) PACK(64, 64);
  else if (D == 64) PACK(64, 128);
  else if (Dv == 64) PACK(128, 64);
  else PACK(128, 128);
#undef PACK
}

// Fixed point by accumulator bias: a product accumulated onto GA_FX_BIAS = 1.5 * 2^23 comes out
// as a float whose unit in the last place is 1, so (bits - bits of the bias) is the sum rounded
// to an integer, for |sum| < 2^22.  The kernel adds the raw bits and counts the adds of every
// output row; the biases leave in the epilogue (all of it modulo 2^32).
#define GA_FX_BIAS 12582912.0f
#define GA_FX_BIAS_BITS 0x4B400000
#define GA_FX_LOG2_MAX 21  // sums are scaled below 2^21: one bit of head room for the rounding of P
// The fine variant converts the products to integers instead: 29 bits below the bound for an instruction per
// accumulator element (32K prefill, 32/8 heads of 128: 2126 -> 2210 us; B4 L8192, 16/16 of 64: 645 -> 662).
#define GA_FX_LOG2_MAX_FINE 30
// Entries of nadd[]: adds of the row (at most a tile's 16 a slot) and, above them, rows that are not numbers
#define GA_ODD_ROW (1 << 16)
#define GA_FX_LIMIT 1.0e18f  // row weight sums and |V| past this go the floating-point way

struct GaDims {
  int L, Lkv, HQ, H, B, K, NW, T, nblk, nchunk, mask_last;
  float sm_scale;
  // indices (and weights) are shared by q_block consecutive queries (T % q_block == 0); weights
  // have WH = HQ or H heads; sm_n * exp(-max) joins every chunk's softmax denominator
  int q_block, WH;
  float sm_n;
  int merge_col;  // with a local-branch output given: the weight column that scales it
  uint32_t k_magic, qb_magic;  // hils_udiv_magic of K and q_block (pair index < 2^16, query index < 2^24)
};

// The bits of a value that may be a NaN.  This file is compiled without NaN handling: the compiler would reason a test of
// the bits of a float it has computed back into one that no NaN passes, so they come through an empty asm statement.
__device__ __forceinline__ unsigned ga_bits(float x) {
  unsigned u = __float_as_uint(x);
  asm("" : "+v"(u));
  return u;
}

// Power-of-two fixed-point scale for sums bounded by `bound`: bound * scale < 2^log2_max.
__device__ __forceinline__ float ga_fx_scale(float bound, int log2_max) {
  if (bound == 0.f) return 1.f;
  int e2 = log2_max - 1 - ilogbf(bound);
  e2 = e2 > 90 ? 90 : (e2 < -90 ? -90 : e2);
  return ldexpf(1.f, e2);
}

// ---- explicit operand loads --------------------------------------------------------------
// The tile stream below keeps several global loads in flight across loop iterations (the next
// tile's query rows, the next visit's K and V).  Which of them are outstanding at a use depends on
// wavefront-uniform branches (does the chunk change?), and the compiler's wait-count insertion
// merges such paths to "wait for nearly everything", which exposed one full memory latency per
// tile.  So the loads of the stream are issued by inline assembly, which that pass does not track,
// and the kernel waits itself: vector-memory loads return in issue order, so
// `s_waitcnt vmcnt(N)` with N = the loads issued after the wanted one (a lower bound is always
// safe; stores are never counted) guarantees it has landed.  A register that a load is still
// writing must not be read or copied before its wait: the waits are followed by empty asm
// statements that "modify" the registers, which orders every use behind the wait.
typedef unsigned ga_u32x4 __attribute__((ext_vector_type(4)));

template <int OFF>
__device__ __forceinline__ void ga_load128(ga_u32x4& dst, unsigned voff, const void* sbase) {
  asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "+v"(dst) : "v"(voff), "s"(sbase), "n"(OFF));
}
__device__ __forceinline__ void ga_load16(unsigned& dst, unsigned voff, const void* sbase) {
  asm volatile("global_load_ushort %0, %1, %2" : "+v"(dst) : "v"(voff), "s"(sbase));
}
template <int N>
__device__ __forceinline__ void ga_vmwait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N));
}
__device__ __forceinline__ void ga_pin(ga_u32x4& a) { asm volatile("" : "+v"(a)); }
__device__ __forceinline__ void ga_pin(unsigned& a) { asm volatile("" : "+v"(a)); }
__device__ __forceinline__ bf16x8_t ga_bf(const ga_u32x4& x) { return __builtin_bit_cast(bf16x8_t, x); }

// One tile of the stream a wavefront works through: up to 16/G (query, slot) pairs of a visit.
template <int KS>
struct GaTile {
  ga_u32x4 bq[KS];  // gathered query rows (B operand of S^T = K Q^T), this lane's pieces
  unsigned wbits;   // this lane's row: its weight (bf16 bits)
  float rs;         // ... and the fixed-point scale of its output row
  int pk;           // ... and its pair (query of the block << 8 | slot)
  int n;            // real pairs in the tile
  int orow[4];      // output-tile element offsets of this lane's four accumulator rows
};

// Output tiles are accumulated in LDS as 32-bit fixed point: integer LDS atomics run at
// full rate on this hardware (float LDS atomics do not), and integer addition is
// associative, so the result does not depend on the order in which wavefronts add.
// The scale is chosen per output row from bound = sum_k |w_row,k| * max_visited|V|, which
// bounds every element of the row because each P row is a convex combination: a row keeps
// 20 bits below its own bound however small its weights are beside its neighbours'.
// FINE: 29 bits, which a column whose V is small beside the largest keeps its precision with: for the calls
// that would otherwise run on the decode kernels, whose sums are fp32.
template <int D, int DV, int G, bool SLOPE, int NT, bool FINE>
__global__ void __launch_bounds__(NT)
sparse_attn_fwd_gather(const bf16_t* __restrict__ q, bf16_t* qp, const bf16_t* __restrict__ kp,
                       const bf16_t* __restrict__ vp, const float* __restrict__ vmax,
                       const bf16_t* __restrict__ weights, const int32_t* __restrict__ indices,
                       const float* __restrict__ slope, const bf16_t* __restrict__ swa_o,
                       bf16_t* __restrict__ o, float* __restrict__ lse, GaDims dm) {
  constexpr int KS = D / 32;    // k-steps of S^T = K Q^T
  constexpr int DT = DV / 16;   // 16-wide output column tiles
  constexpr int QT = 16 / G;    // queries per 16-row tile
  constexpr int MAXP = GA_MAXP;  // pairs per thread: T*K <= MAXP * GA_THREADS
  typedef GaTile<KS> Tile;
  extern __shared__ __align__(16) int smem_i[];
  const int R = dm.T * G;
  int* o_acc = smem_i;                       // R x DV fixed point
  int* cur = o_acc + (size_t)R * DV;         // nchunk: histogram -> running ends
  int* pairs = cur + dm.nchunk;              // T*K pairs (query << 8 | slot) grouped by chunk
  int* nadd = pairs + dm.T * dm.K;           // R: tiles added to each output row, and how many were not numbers
  float* rscale = (float*)(nadd + R);        // R: sum_k |w| of the row, then its fixed-point scale
  __shared__ float red[32];
  __shared__ int scan_s[NT / 64];
  __shared__ int next_s;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, j = lane >> 4;
  // XCD-aware order: hardware hands consecutive workgroup ids to the 8 XCDs in turn, so
  // id -> (xcd, slot); each XCD walks one contiguous share of the (batch, head, block)
  // list, latest query blocks first, and its L2 sees one head's K/V at a time.
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
  const long LB = dm.L / dm.q_block;          // rows of indices / weights per batch element
  const bool w_per_q = dm.WH == dm.HQ;        // weights per query head (else per KV head)

  // ---- prologue.  All global loads of the block set-up are issued before anything waits:
  // the query rows to repack, the selected chunk indices, and the weight rows.
  // (0) Packed copy of this block's query rows: within the G heads of a (query, KV head) the
  // 16-byte pieces are interleaved head-minor, [piece][head][8], so that the B-operand loads
  // of the G lanes that hold the heads of one query are contiguous (whole cache lines; read in
  // place, a row's four lanes would touch half a line each).  Only this workgroup reads what it
  // writes here (made visible by the barriers below).
  constexpr int PPR = D / 8;
  constexpr int QPK = 10;  // pieces per thread in flight (a 72-query block of 4 heads, D = 128, has 9)
  const int npiece = dm.T * G * PPR;
  uint4 qtmp[QPK];
#pragma unroll
  for (int e = 0; e < QPK; ++e) {
    const int i = tid + e * NT;
    const int ql = i / (G * PPR), rem = i - ql * (G * PPR);
    const int g2 = rem / PPR, pc = rem - g2 * PPR;
    const bool ok = i < npiece && t0 + ql < dm.L;
    const long blk_e = ((b * dm.L + (ok ? t0 + ql : t0)) * (long)dm.HQ + hk * G) * D;  // t0 < L always
    // relaxed atomic loads: the compiler keeps them here, ahead of the loads below, instead of
    // moving them next to their use behind the weight loop (a second exposed latency)
    const unsigned long long* src = (const unsigned long long*)(q + blk_e + g2 * D + pc * 8);
    const unsigned long long lo = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    const unsigned long long hi = __hip_atomic_load(src + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    qtmp[e] = make_uint4((unsigned)lo, (unsigned)(lo >> 32), (unsigned)hi, (unsigned)(hi >> 32));
  }
  // (1) selected chunk of every (query, slot) pair of the block
  int creg[MAXP], preg[MAXP];
#pragma unroll
  for (int e = 0; e < MAXP; ++e) {
    const int i = tid + e * NT;
    int c = -1;
    preg[e] = 0;
    if (i < npair) {
      const int ql = (int)hils_udiv((uint32_t)i, (uint32_t)K, dm.k_magic), slot = i - ql * K;
      preg[e] = (ql << 8) | slot;
      if (t0 + ql < dm.L) c = indices[((b * LB + (long)hils_udiv((uint32_t)(t0 + ql), (uint32_t)dm.q_block, dm.qb_magic)) * dm.H + hk) * (long)K + slot];
    }
    creg[e] = c;
  }
  // (2) weight rows, for the bound of the fixed-point scale: a row's sum of |w| over the K slots
  // (aligned dword loads, all in flight together)
  bool no_fx = false;  // something fixed point cannot hold (told by the bits: NaNs compare as the largest)
  for (int row = tid; row < R; row += NT) {
    const int ql = row / G, g = row - ql * G;
    float a = 0.f;
    if (t0 + ql < dm.L) {
      const long e0 = ((b * LB + (long)hils_udiv((uint32_t)(t0 + ql), (uint32_t)dm.q_block, dm.qb_magic)) * (long)dm.WH + (w_per_q ? hk * G + g : hk)) *
                      dm.NW;  // first element
      a = hils_abs_row_sum_bf16(weights, e0, K, (long)dm.B * LB * dm.WH * dm.NW);
    }
    no_fx = no_fx || ga_bits(a) > __float_as_uint(GA_FX_LIMIT);
    rscale[row] = a;  // only this thread touches the entry until the barrier behind the scan
  }
  // The packed copy goes through LDS (the output tile is not in use yet): pieces arrive in the
  // order of the source rows and leave in packed order, so that loads and stores are both
  // contiguous 1 KiB per wavefront instruction.  The staged pieces fit the output tile: a row has
  // D / 8 pieces of 16 bytes against DV * 4 bytes of accumulators (D <= 2 * DV).
  static_assert(D <= 2 * DV, "the staged query pieces must fit inside the output tile");
  uint4* stage = (uint4*)o_acc;
#pragma unroll
  for (int e = 0; e < QPK; ++e) {
    const int i = tid + e * NT;
    const int ql = i / (G * PPR), rem = i - ql * (G * PPR);
    const int g2 = rem / PPR, pc = rem - g2 * PPR;
    if (i < npiece) stage[ql * (G * PPR) + pc * G + g2] = qtmp[e];
  }
  for (int i = QPK * NT + tid; i < npiece; i += NT) {  // blocks with more pieces (rare shapes)
    const int ql = i / (G * PPR), rem = i - ql * (G * PPR);
    const int g2 = rem / PPR, pc = rem - g2 * PPR;
    const long blk_e = ((b * dm.L + (t0 + ql < dm.L ? t0 + ql : t0)) * (long)dm.HQ + hk * G) * D;
    stage[ql * (G * PPR) + pc * G + g2] = *(const uint4*)(q + blk_e + g2 * D + pc * 8);
  }
  for (int i = tid; i < dm.nchunk; i += NT) cur[i] = 0;
  for (int i = tid; i < R; i += NT) nadd[i] = 0;
  if (tid == 0) next_s = 0;
  lds_barrier();
  for (int i = tid; i < npiece; i += NT) {
    const int ql = i / (G * PPR);
    const uint4 x = stage[i];
    stage[i] = make_uint4(0, 0, 0, 0);  // this thread's share of clearing the output tile
    if (t0 + ql < dm.L)
      *(uint4*)(qp + ((b * dm.L + t0 + ql) * (long)dm.HQ + hk * G) * D + (i - ql * (G * PPR)) * 8) = x;
  }
  for (int i = npiece * 4 + tid; i < R * DV; i += NT) o_acc[i] = 0;  // the rest of the tile
  // (LDS-only barriers up to the last one of the prologue: the packed-query stores above stay in
  // flight behind the sort instead of being waited for here)
  lds_barrier();
  // histogram of the selected chunks
#pragma unroll
  for (int e = 0; e < MAXP; ++e) {
    int c = creg[e];
    if (c < -1 || c >= dm.nchunk) c = -1;
    if (c < 0 && lse) {
      const int i = tid + e * NT;
      const int ql = (int)hils_udiv((uint32_t)i, (uint32_t)K, dm.k_magic), slot = i - ql * K;
      if (i < npair && t0 + ql < dm.L) {
#pragma unroll
        for (int g = 0; g < G; ++g)
          lse[((b * dm.L + t0 + ql) * dm.HQ + hk * G + g) * (long)K + slot] = HILS_NEG_INF;
      }
    }
    creg[e] = c;
    if (c >= 0) atomicAdd(&cur[c], 1);
  }
  lds_barrier();  // histogram complete
  // max |V| over the visited chunks; exclusive scan of the histogram on the way
  float vm = 0.f;
  const int per_thr = (dm.nchunk + NT - 1) / NT;
  const int c_lo = tid * per_thr;
  int local = 0;
  for (int c = c_lo; c < c_lo + per_thr && c < dm.nchunk; ++c) {
    const int h = cur[c];
    if (h > 0) {
      const float cm = vmax[(b * dm.H + hk) * (long)dm.nchunk + c];
      no_fx = no_fx || ga_bits(cm) > __float_as_uint(GA_FX_LIMIT);  // (a set sign bit too)
      vm = fmaxf(vm, cm);
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
  vm = block_max_lds(no_fx ? INFINITY : vm, red);  // barrier: scan_s visible, all histogram reads done
  const bool flt = __builtin_amdgcn_readfirstlane((int)(vm > GA_FX_LIMIT)) != 0;  // of the whole block
  int base = incl - local;
  for (int w2 = 0; w2 < wave; ++w2) base += scan_s[w2];
  for (int c = c_lo; c < c_lo + per_thr && c < dm.nchunk; ++c) {
    const int h = cur[c];
    cur[c] = base;
    base += h;
  }
  for (int row = tid; row < R; row += NT) rscale[row] = flt ? 1.f : ga_fx_scale(rscale[row] * vm, FINE ? GA_FX_LOG2_MAX_FINE : GA_FX_LOG2_MAX);
  lds_barrier();
#pragma unroll
  for (int e = 0; e < MAXP; ++e)
    if (creg[e] >= 0) pairs[atomicAdd(&cur[creg[e]], 1)] = preg[e];
  __syncthreads();  // now chunk c owns pairs[cur[c-1] .. cur[c])

  const float c2 = dm.sm_scale * HILS_LOG2E;
  const int qs = r / G, g = r - qs * G;  // this lane's row of a tile: query slot, head
  const int hq = hk * G + g;
  const float sl = SLOPE ? slope[hq] : 0.f;
  // rows of a tile are addressed from the block's first query with 32-bit byte offsets into the
  // packed copy, in which the G heads of a query are interleaved per 16-byte piece: the lanes of
  // one query read contiguous bytes
  const char* qb = (const char*)(qp + ((b * dm.L + t0) * (long)dm.HQ + hk * G) * D);
  const bf16_t* wb = weights + ((b * LB + t0 / dm.q_block) * (long)dm.WH + (w_per_q ? hk * G : hk)) * dm.NW;
  float* lse_blk = lse ? lse + (b * dm.L + t0) * (long)dm.HQ * K : nullptr;  // the block's first row
  const unsigned q_lane = (unsigned)((j * G + g) * 8) * 2u, w_lane = w_per_q ? (unsigned)(g * dm.NW) : 0u;
  const unsigned q_step = (unsigned)dm.HQ * D * 2u;  // bytes per query of the block
  const int w_step = dm.WH * dm.NW;                  // elements per group of q_block queries

  // ---- visits: a wavefront takes chunks from a shared counter; a visit is all pairs of the
  // block on one chunk, processed as tiles of up to QT pairs.  The tile stream of a wavefront
  // is software-pipelined so that no operand load is waited for right after it is issued:
  //   step i:  issue Q(i+1);  O += P(i-1) V  [then V(chunk i) replaces V in place];
  //            S(i) = K Q(i)^T  [then K(chunk i+1) replaces K in place];  softmax -> P(i).
  // K and V of a chunk are reloaded only when the next tile belongs to another chunk.  Two tile
  // records alternate between "current" and "next / previous", so nothing is copied per step.
  ga_u32x4 ka[4][KS], vb[DT][2];
  constexpr int NK = 4 * KS;   // loads of a K reload
  constexpr int NV = 2 * DT;   // loads of a V reload
  constexpr int NA = KS + 1;   // loads of a tile issue (query pieces + weight)
  // operand loads: a wavefront-uniform 64-bit base plus this lane's 32-bit byte offset; the
  // instruction's immediate offset reaches 4 KiB, so a chunk is addressed from 4 KiB-spaced bases
  const unsigned lane_b = lane * 16;
  const char* kp_unit = (const char*)(kp + (b * dm.H + hk) * (long)dm.nchunk * GA_S * D);
  const char* vp_unit = (const char*)(vp + (b * dm.H + hk) * (long)dm.nchunk * GA_S * DV);
  auto load_k_all = [&](int c) {
    const char* kbase = kp_unit + (long)c * (GA_S * D * 2);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        constexpr int dummy = 0; (void)dummy;
        const int piece = mt * KS + ks;  // 1 KiB pieces
        const char* sb = kbase + (piece / 4) * 4096;
        switch (piece % 4) {
          case 0: ga_load128<0>(ka[mt][ks], lane_b, sb); break;
          case 1: ga_load128<1024>(ka[mt][ks], lane_b, sb); break;
          case 2: ga_load128<2048>(ka[mt][ks], lane_b, sb); break;
          default: ga_load128<3072>(ka[mt][ks], lane_b, sb); break;
        }
      }
  };
  auto load_v_half = [&](int c, int d0, int nd) {  // column tiles d0 .. d0+nd-1
    const char* vbase = vp_unit + (long)c * (GA_S * DV * 2);
#pragma unroll
    for (int u = 0; u < nd; ++u)
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const int piece = (d0 + u) * 2 + s2;
        const char* sb = vbase + (piece / 4) * 4096;
        switch (piece % 4) {
          case 0: ga_load128<0>(vb[d0 + u][s2], lane_b, sb); break;
          case 1: ga_load128<1024>(vb[d0 + u][s2], lane_b, sb); break;
          case 2: ga_load128<2048>(vb[d0 + u][s2], lane_b, sb); break;
          default: ga_load128<3072>(vb[d0 + u][s2], lane_b, sb); break;
        }
      }
  };
  auto pin_k = [&]() {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) ga_pin(ka[mt][ks]);
  };
  auto pin_v = [&]() {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      ga_pin(vb[dt][0]);
      ga_pin(vb[dt][1]);
    }
  };
  const int npair_valid = cur[dm.nchunk - 1];  // pairs with a valid chunk
  // next non-empty visit: chunk id (or -1) and its pair range
  auto grab = [&](int& vs_o, int& ve_o) -> int {
    for (;;) {
      int c = 0;
      if (lane == 0) c = atomicAdd(&next_s, 1);
      c = __builtin_amdgcn_readfirstlane(c);
      if (c >= dm.nchunk) return -1;
      vs_o = c ? cur[c - 1] : 0;
      if (vs_o >= npair_valid) return -1;  // every pair lies in an earlier chunk
      ve_o = cur[c];
      if (vs_o != ve_o) return c;
    }
  };
  // tile after (c, p, ve)
  auto advance = [&](int& c, int& p, int& ve) {
    if (p + QT < ve) { p += QT; return; }
    int vs2, ve2;
    c = grab(vs2, ve2);
    p = vs2;
    ve = ve2;
  };
  // A tile's gathered query rows (B operands), weight, row scale: NA loads.  Padding rows of a
  // visit's last tile repeat the tile's last pair with weight 0: their P is exactly 0 and is
  // added to that pair's output rows.
  const char* wb_c = (const char*)wb;
  auto issue_tile = [&](Tile& t, int p, int ve) {
    t.n = (ve - p < QT) ? ve - p : QT;
    const int last = t.n - 1;
    t.pk = pairs[p + (qs < last ? qs : last)];
    const unsigned ql = (unsigned)t.pk >> 8;
    const unsigned qoff = __umul24(ql, q_step) + q_lane;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      switch (ks) {
        case 0: ga_load128<0>(t.bq[ks], qoff, qb); break;
        case 1: ga_load128<4 * G * 16>(t.bq[ks], qoff, qb); break;
        case 2: ga_load128<2 * 4 * G * 16>(t.bq[ks], qoff, qb); break;
        default: ga_load128<3 * 4 * G * 16>(t.bq[ks], qoff, qb); break;
      }
    }
    const unsigned woff =
        (__umul24(dm.q_block == 1 ? ql : ql / (unsigned)dm.q_block, (unsigned)w_step) + w_lane + (t.pk & 255)) * 2u;
    ga_load16(t.wbits, woff, wb_c);
    t.rs = rscale[ql * G + g];
  };
  auto pin_tile = [&](Tile& t) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) ga_pin(t.bq[ks]);
    ga_pin(t.wbits);
  };
  // output rows 4j .. 4j+3 of a tile starting at pair p (element offsets of this lane's column)
  auto tile_rows = [&](Tile& t, int p, auto flt_c) __attribute__((always_inline)) {
    const int last = t.n - 1;
    if constexpr (G >= 4) {  // the four rows are consecutive heads of one query
      const int qsl = (4 * j) / G;
      const int pk = pairs[p + (qsl < last ? qsl : last)];
      const int base = ((pk >> 8) * G + (4 * j) % G) * DV + r;
#pragma unroll
      for (int i = 0; i < 4; ++i) t.orow[i] = base + i * DV;
    } else {
      int pk_o[4];
      if (t.n == QT) {  // neighbouring entries, no clamps
        const int* po = pairs + p + (4 * j) / G;
#pragma unroll
        for (int i = 0; i < 4; ++i) pk_o[i] = po[i / G];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int qsl = (4 * j + i) / G;
          pk_o[i] = pairs[p + (qsl < last ? qsl : last)];
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) t.orow[i] = (int)__umul24((unsigned)pk_o[i] >> 8, (unsigned)(G * DV)) + (i % G) * DV + r;
    }
    if constexpr (decltype(flt_c)::value) {  // a padding row's zero times an infinity is no zero: it is left out
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if ((4 * j + i) / G > last) t.orow[i] = -1;
    }
  };
  bf16x8_t ap[2];   // P of the previous tile (A operand of O = P V)
  // S = K Q^T of tile t (its operands have landed), softmax, P -> ap; K(c_next) replaces K when asked
  auto score_stage = [&](Tile& t, bool reload, int c_next) {
    // four independent accumulation chains (token tiles), interleaved so that a chain's next
    // MFMA is issued only after three others
    f32x4_t st[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) st[mt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
        st[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga_bf(ka[mt][ks]), ga_bf(t.bq[ks]), st[mt], 0, 0, 0);
    if (reload) load_k_all(c_next);
    if (SLOPE) {
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int dist = GA_S - 2 - (mt * 16 + j * 4 + i);
          st[mt][i] -= sl * (float)(dist > 0 ? dist : 0);
        }
    }
    if (dm.mask_last && j == 3) st[3][3] = HILS_NEG_INF;  // token 63 = tile 3, lane group 3, register 3
    // (this file is compiled without NaN handling: the maxima are bare v_max3 instructions)
    float m = fmaxf(fmaxf(st[0][0], st[0][1]), st[0][2]);
    m = fmaxf(fmaxf(m, st[0][3]), st[1][0]);
    m = fmaxf(fmaxf(m, st[1][1]), st[1][2]);
    m = fmaxf(fmaxf(m, st[1][3]), st[2][0]);
    m = fmaxf(fmaxf(m, st[2][1]), st[2][2]);
    m = fmaxf(fmaxf(m, st[2][3]), st[3][0]);
    m = fmaxf(fmaxf(m, st[3][1]), st[3][2]);
    m = rows_max(fmaxf(m, st[3][3]));
    const float mc = m * c2;
    float sum = 0.f;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = __builtin_amdgcn_exp2f(st[mt][i] * c2 - mc);
        st[mt][i] = e;
        sum += e;
      }
    sum = rows_sum(sum);
    if (dm.sm_n != 0.f) sum += dm.sm_n * __builtin_amdgcn_exp2f(-mc);
    if (lse && qs < t.n && j == 0) {
      const int ql = t.pk >> 8, slot = t.pk & 255;
      lse_blk[(ql * dm.HQ + hq) * K + slot] = mc + __builtin_amdgcn_logf(sum);
    }
    const float w_row = qs < t.n ? __uint_as_float(t.wbits << 16) : 0.f;
    const float f = w_row * t.rs * __builtin_amdgcn_rcpf(sum);  // fixed-point scale (a power of two) folded into P
    // (padding rows count on the row they are added to)
    if (j == 0) atomicAdd(&nadd[(t.pk >> 8) * G + g], (ga_bits(f) & 0x7f800000u) == 0x7f800000u ? GA_ODD_ROW + 1 : 1);
    // P as the A operand of O = P V: k-step s takes tokens of accumulator tiles 2s, 2s+1
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      uint4 x;
      x.x = pack_bf2(st[2 * s][0] * f, st[2 * s][1] * f);
      x.y = pack_bf2(st[2 * s][2] * f, st[2 * s][3] * f);
      x.z = pack_bf2(st[2 * s + 1][0] * f, st[2 * s + 1][1] * f);
      x.w = pack_bf2(st[2 * s + 1][2] * f, st[2 * s + 1][3] * f);
      ap[s] = *(bf16x8_t*)&x;
    }
  };
  // O += P V for the tile whose rows are `orow` (V has landed); V(c_next) replaces V when asked
  auto add = [&](int* at, float x) __attribute__((always_inline)) { atomicAdd(at, FINE ? (int)x : __float_as_int(x)); };
  auto output_stage = [&](const int* orow, bool reload, int c_next, auto flt_c) __attribute__((always_inline)) {
    constexpr bool FLT = decltype(flt_c)::value;
    constexpr float acc0 = FINE || FLT ? 0.f : GA_FX_BIAS;
    const f32x4_t fx_bias = {acc0, acc0, acc0, acc0};
    // four column tiles at a time: their eight MFMAs interleaved (two-deep chains), then the
    // operand reload, then the fixed-point adds
#pragma unroll
    for (int d0 = 0; d0 < DT; d0 += 4) {
      f32x4_t acc[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] = fx_bias;
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ap[s2], ga_bf(vb[d0 + u][s2]), acc[u], 0, 0, 0);
      if (reload) load_v_half(c_next, d0, 4);
      if constexpr (FLT) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (orow[i] >= 0) unsafeAtomicAdd((float*)&o_acc[orow[i] + (d0 + u) * 16], acc[u][i]);
      } else if constexpr (G >= 4) {
        // the lane's four rows are consecutive heads of one query: one address, the rest are offsets
        // the instruction carries
        int* o0 = o_acc + orow[0];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) add(o0 + i * DV + (d0 + u) * 16, acc[u][i]);
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) add(&o_acc[orow[i] + (d0 + u) * 16], acc[u][i]);
      }
    }
  };

  // ---- the stream.  Issue order of a step i (x_i = "tile i is on another chunk than tile i-1"):
  //   A_i: query rows + weight of tile i+1 (NA loads, when there is a tile i+1)
  //   B_i: V of tile i's chunk (NV loads, when x_i), behind the MFMAs of O += P(i-1) V
  //   C_i: K of tile i+1's chunk (NK loads, when x_{i+1}), behind the MFMAs of S(i)
  // O += P(i-1) V needs B_{i-1}: the loads behind it are C_{i-1} (NK when x_i) and A_i;
  // S(i) needs C_{i-1} and A_{i-1}: the loads behind C_{i-1} are A_i and B_i (NV when x_i).
  // Without a tile i+1 there is no A_i and the step simply waits for everything.
  auto stream = [&](auto flt_c) __attribute__((always_inline)) {
    int c_cur, p_cur = 0, ve_cur = 0;
    c_cur = grab(p_cur, ve_cur);
    if (c_cur >= 0) {
      Tile ta, tb;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) { ta.bq[ks] = (ga_u32x4){0, 0, 0, 0}; tb.bq[ks] = (ga_u32x4){0, 0, 0, 0}; }
      ta.wbits = tb.wbits = 0;
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) ka[mt][ks] = (ga_u32x4){0, 0, 0, 0};
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) vb[dt][0] = vb[dt][1] = (ga_u32x4){0, 0, 0, 0};
      // step 0 (no previous tile): A_{-1} = tile 0, C_{-1} = K(c_0), then A_0, B_0 = V(c_0)
      issue_tile(ta, p_cur, ve_cur);
      tile_rows(ta, p_cur, flt_c);
      load_k_all(c_cur);
      int c_nxt = c_cur, p_nxt = p_cur, ve_nxt = ve_cur;
      advance(c_nxt, p_nxt, ve_nxt);
      if (c_nxt >= 0) {
        issue_tile(tb, p_nxt, ve_nxt);
        tile_rows(tb, p_nxt, flt_c);
      }
      load_v_half(c_cur, 0, DT);
      if (c_nxt >= 0) ga_vmwait<NA + NV>(); else ga_vmwait<NV>();
      pin_k();
      pin_tile(ta);
      score_stage(ta, c_nxt >= 0 && c_nxt != c_cur, c_nxt);
      int c_prev = c_cur;
      // one step: `cu` is the tile whose scores are due (its loads were issued a step ago), `nx`
      // holds the previous tile's output rows until the output stage is through, then the tile
      // after `cu`.
      auto step = [&](Tile& cu, Tile& nx) {
        c_cur = c_nxt; p_cur = p_nxt; ve_cur = ve_nxt;
        advance(c_nxt, p_nxt, ve_nxt);
        const bool more = c_nxt >= 0;
        const bool x = c_cur != c_prev;
        if (more) issue_tile(nx, p_nxt, ve_nxt);  // A_i; leaves nx.orow alone
        if (!more) ga_vmwait<0>(); else if (x) ga_vmwait<NA + NK>(); else ga_vmwait<NA>();
        pin_v();
        output_stage(nx.orow, x, c_cur, flt_c);          // B_i
        if (more) tile_rows(nx, p_nxt, flt_c);
        if (!more) ga_vmwait<0>(); else if (x) ga_vmwait<NA + NV>(); else ga_vmwait<NA>();
        pin_k();
        pin_tile(cu);
        score_stage(cu, more && c_nxt != c_cur, c_nxt);  // C_i
        c_prev = c_cur;
      };
      // the stream: tile 0 = ta (scored above), tile 1 = tb, tile 2 -> ta, ...
      bool last_is_a = true;
      while (c_nxt >= 0) {
        step(tb, ta);
        last_is_a = false;
        if (c_nxt < 0) break;
        step(ta, tb);
        last_is_a = true;
      }
      int orow_last[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) orow_last[i] = last_is_a ? ta.orow[i] : tb.orow[i];
      ga_vmwait<0>();
      pin_v();
      output_stage(orow_last, false, 0, flt_c);
    }
  };
  // (two copies of the stream: a branch at its adds cost 1.5 % with heads of 128)
  if (flt) stream(std::true_type{}); else stream(std::false_type{});
  __syncthreads();
  constexpr int C8 = DV / 8;
  const int wcol = dm.merge_col;
  for (int i = tid; i < R * C8; i += NT) {
    const int row = i / C8, c8 = i - row * C8;
    const int ql = row / G, g2 = row - ql * G;
    const int t = t0 + ql;
    if (t < dm.L) {
      const int* src = o_acc + (size_t)row * DV + c8 * 8;
      const unsigned added = (unsigned)nadd[row];
      const unsigned bias = FINE ? 0u : (added & (GA_ODD_ROW - 1)) * (unsigned)GA_FX_BIAS_BITS;  // wraps like the sums did
      const float fx_inv = 1.f / rscale[row];  // a power of two: exact
      const int4 s0 = *(const int4*)src, s1 = *(const int4*)(src + 4);
      const int sum[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = (float)(int)((unsigned)sum[e] - bias) * fx_inv;
      if (flt) {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = __int_as_float(sum[e]);
      }
      const long orow_g = ((b * dm.L + t) * (long)dm.HQ + hk * G + g2) * DV + c8 * 8;
      if (swa_o) {  // o = remote branch + local branch * its inter-chunk weight, rounded once
        const float wl = bf2f(weights[((b * LB + (long)hils_udiv((uint32_t)t, (uint32_t)dm.q_block, dm.qb_magic)) * (long)dm.WH + (w_per_q ? hk * G + g2 : hk)) *
                                          dm.NW + wcol]);
        float sv[8];
        unpack8(*(const uint4*)(swa_o + orow_g), sv);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = fmaf(sv[e], wl, f[e]);
      }
      uint4 x;
      x.x = pack_bf2(f[0], f[1]);
      x.y = pack_bf2(f[2], f[3]);
      x.z = pack_bf2(f[4], f[5]);
      x.w = pack_bf2(f[6], f[7]);
      if (added >= GA_ODD_ROW) x = make_uint4(0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u);
      *(uint4*)(o + orow_g) = x;
    }
  }
}

template <int D, int DV, int G, bool SLOPE, bool FINE>
static int ga_launch_s(dim3 grid, size_t smem, hipStream_t st, const bf16_t* q, bf16_t* qp, const bf16_t* k,
                       const bf16_t* vt, const float* vmax, const bf16_t* w, const int32_t* idx,
                       const float* slope, const bf16_t* swa_o, bf16_t* o, float* lse, const GaDims& dm) {
  static_assert(D % 32 == 0 && DV % 16 == 0 && 16 % G == 0, "tile shapes of the MFMA forward");
  // Narrow heads leave the wavefronts under 168 registers: twelve of them per workgroup (one workgroup
  // per compute unit, its size is what sets the occupancy) instead of eight.
  constexpr int NT = (D <= 64 && DV <= 64) ? GA_THREADS_NARROW : GA_THREADS;
  auto kern = sparse_attn_fwd_gather<D, DV, G, SLOPE, NT, FINE>;
  static HilsLdsReserve reserved;  // per instantiation
  if (int rc = hils_reserve_lds(&reserved, (const void*)kern, smem, "hils_sparse_attn_fwd")) return rc;
  hipLaunchKernelGGL(kern, grid, dim3(NT), smem, st, q, qp, k, vt, vmax, w, idx, slope, swa_o, o, lse, dm);
  return HILS_OK;
}

template <int D, int DV, int G>
static int ga_launch(dim3 grid, size_t smem, hipStream_t st, const bf16_t* q, bf16_t* qp, const bf16_t* k,
                     const bf16_t* vt, const float* vmax, const bf16_t* w, const int32_t* idx,
                     const float* slope, const bf16_t* swa_o, bf16_t* o, float* lse, bool fine, const GaDims& dm) {
  if constexpr (D == DV && G <= 8)  // (what decode_step takes)
    if (fine && !slope) return ga_launch_s<D, DV, G, false, true>(grid, smem, st, q, qp, k, vt, vmax, w, idx, slope, swa_o, o, lse, dm);
  if (slope) return ga_launch_s<D, DV, G, true, false>(grid, smem, st, q, qp, k, vt, vmax, w, idx, slope, swa_o, o, lse, dm);
  return ga_launch_s<D, DV, G, false, false>(grid, smem, st, q, qp, k, vt, vmax, w, idx, slope, swa_o, o, lse, dm);
}

template <int D, int DV>
static int ga_dispatch_g(int G, dim3 grid, size_t smem, hipStream_t st, const bf16_t* q, bf16_t* qp,
                         const bf16_t* k, const bf16_t* vt, const float* vmax, const bf16_t* w,
                         const int32_t* idx, const float* slope, const bf16_t* swa_o, bf16_t* o, float* lse,
                         bool fine, const GaDims& dm) {
  switch (G) {
    case 1: return ga_launch<D, DV, 1>(grid, smem, st, q, qp, k, vt, vmax, w, idx, slope, swa_o, o, lse, fine, dm);
    case 2: return ga_launch<D, DV, 2>(grid, smem, st, q, qp, k, vt, vmax, w, idx, slope, swa_o, o, lse, fine, dm);
    case 4: return ga_launch<D, DV, 4>(grid, smem, st, q, qp, k, vt, vmax, w, idx, slope, swa_o, o, lse, fine, dm);
    case 8: return ga_launch<D, DV, 8>(grid, smem, st, q, qp, k, vt, vmax, w, idx, slope, swa_o, o, lse, fine, dm);
    case 16: return ga_launch<D, DV, 16>(grid, smem, st, q, qp, k, vt, vmax, w, idx, slope, swa_o, o, lse, fine, dm);
  }
  return -1;
}

static size_t ga_vt_bytes(int B, int H, int nchunk, int Dv) {  // one packed tensor (K or V)
  size_t n = (size_t)B * H * nchunk * Dv * GA_S * sizeof(bf16_t);
  return (n + 255) & ~(size_t)255;
}

static size_t ga_vmax_bytes(int B, int H, int nchunk) {
  return ((size_t)B * H * nchunk * sizeof(float) + 255) & ~(size_t)255;
}

// Tile sizes: the largest T (queries per workgroup, a multiple of q_block and of 8 when it can be)
// such that the fixed-point output tile, the chunk histogram, the pair list and the add counts
// fit in the LDS of a compute unit, with at most GA_MAXP pairs per thread.  The more rows share a
// visit, the fewer bytes of K and V the block pulls per row.  Returns 0 when nothing fits.
// A call too small for that gets more, smaller blocks: one round of the compute units (or two, when it
// would otherwise end in a partly filled second one), down to four queries.  units: (batch, KV head)
// pairs.  (56 blocks of 72 queries -> 250 of 8 at B1 L2000 16/2 heads of 64: 57 -> 22 us; 16 blocks of 64
// -> 256 of 4 at 128 queries on 64K tokens, 32/8 heads of 128: 329 -> 65; 420 of 72 -> 474 of 64 at B3
// L5000 16/2: 150 -> 137; twice as many blocks as compute units were slower again, 31 us in the first.)
#define GA_SMEM_MAX (160 * 1024 - 512)  // dynamic LDS beside the kernel's static arrays
static int ga_pick_T(int L, long units, int G, int Dv, int K, int nchunk, int q_block, size_t* smem_out) {
  // per query: G output rows, K pairs, G add counts, G row scales
  const size_t per_q = (size_t)G * Dv * 4 + (size_t)K * 4 + (size_t)G * 4 + (size_t)G * 4;
  const size_t fixed = (size_t)nchunk * 4;
  if (fixed + per_q > GA_SMEM_MAX) return 0;
  long T = (long)((GA_SMEM_MAX - fixed) / per_q);
  if (T * K > GA_MAXP * GA_THREADS) T = (GA_MAXP * GA_THREADS) / K;
  if (T > L) T = L;
  {
    const long cus = hils_device_cus(), wgs = units * ((L + T - 1) / T);
    const long rounds = wgs <= cus ? 1 : 2;
    if (wgs <= cus || (4 * wgs > 5 * cus && wgs < 2 * cus)) {
      const long per_unit = cus * rounds / units;  // blocks a (batch, KV head) gets
      if (per_unit > 0) {
        long t = (L + per_unit - 1) / per_unit;
        t = t <= 4 ? 4 : (t + 7) & ~7L;
        t = (t + q_block - 1) / q_block * q_block;
        if (t < T) T = t;
      }
    }
  }
  if (T >= 8 && q_block <= 8 && 8 % q_block == 0) T &= ~7L;
  else T -= T % q_block;
  if (T < 1) return 0;
  *smem_out = fixed + (size_t)T * per_q;
  return (int)T;
}

// Workspace the MFMA path needs (the per-chunk transposed copy of V and the per-chunk max|V|),
// 0 if the shape is not covered by it.
size_t hils_ga_workspace_bytes(int B, int L, int Lkv, int HQ, int H, int D, int Dv, int K, int S,
                               int q_block, int WH, float sm_n) {
  if (H <= 0 || HQ % H != 0) return 0;
  const int G = HQ / H;
  const bool ok = S == GA_S && (D == 64 || D == 128) && (Dv == 64 || Dv == 128) &&
                  (G == 1 || G == 2 || G == 4 || G == 8 || G == 16) && q_block >= 1 &&
                  L % q_block == 0 && (WH == HQ || WH == H) && sm_n >= 0.f && L >= 64 && Lkv >= S &&
                  K >= 1 && K <= 256 && (long)L * q_block < (1L << 31);  // hils_udiv by q_block stays exact
  if (!ok) return 0;
  size_t smem;
  const int T = ga_pick_T(L, (long)B * H, G, Dv, K, Lkv / S, q_block, &smem);
  if (T == 0 || T % q_block != 0) return 0;  // a query block holds whole index-sharing groups
  const int nchunk = Lkv / S;
  return ga_vt_bytes(B, H, nchunk, Dv) + ga_vt_bytes(B, H, nchunk, D) + ga_vmax_bytes(B, H, nchunk) +
         (size_t)B * L * HQ * D * sizeof(bf16_t);  // packed V, packed K, per-chunk max|V|, packed Q
}

// Queries of a workgroup for a call of one index row per query, 0 if the MFMA path does not take it.
int hils_ga_block(int B, int L, int Lkv, int HQ, int H, int D, int K) {
  if (hils_ga_workspace_bytes(B, L, Lkv, HQ, H, D, D, K, GA_S, 1, HQ, 0.f) == 0) return 0;
  size_t smem;
  return ga_pick_T(L, (long)B * H, HQ / H, D, K, Lkv / GA_S, 1, &smem);
}

// Returns HILS_OK and sets *handled = 1 when the MFMA path ran.
int hils_sparse_attn_fwd_mfma(const void* q, const void* k, const void* v, const void* weights,
                              const int32_t* indices, const float* slope, const void* swa_o, int merge_col,
                              void* o, float* lse, void* workspace, int workspace_ready, int B, int L,
                              int Lkv, int HQ, int H, int D, int Dv, int K, int NW, int S, float sm_scale,
                              int mask_last, int q_block, int WH, float sm_n, bool fine, void* stream,
                              int* handled) {
  *handled = 0;
  const int G = HQ / H;
  const int nchunk = Lkv / S;
  hipStream_t st = (hipStream_t)stream;
  size_t smem;
  const int T = ga_pick_T(L, (long)B * H, G, Dv, K, nchunk, q_block, &smem);
  if (T == 0 || T % q_block != 0 || H > 65535 || B > 65535) return HILS_OK;
  const int nblk = (L + T - 1) / T;
  const long total = (long)nblk * H * B;
  if (total > (1L << 30)) return HILS_OK;
  bf16_t* vpk = (bf16_t*)workspace;
  bf16_t* kpk = (bf16_t*)((char*)workspace + ga_vt_bytes(B, H, nchunk, Dv));
  float* vmax = (float*)((char*)kpk + ga_vt_bytes(B, H, nchunk, D));
  bf16_t* qpk = (bf16_t*)((char*)vmax + ga_vmax_bytes(B, H, nchunk));
  if (!workspace_ready) pack_kv_launch<false>(k, v, kpk, vpk, nullptr, nullptr, vmax, B, Lkv, H, D, Dv, st);
  GaDims dm{L, Lkv, HQ, H, B, K, NW, T, nblk, nchunk, mask_last, sm_scale, q_block, WH, sm_n, merge_col,
            hils_udiv_magic((uint32_t)K), hils_udiv_magic((uint32_t)q_block)};
  const long per_xcd = (total + 7) / 8;
  dim3 grid((unsigned)(per_xcd * 8));
  int rc = -1;
#define GA_CALL(D_, DV_)                                                                       \
  rc = ga_dispatch_g<D_, DV_>(G, grid, smem, st, (const bf16_t*)q, qpk, kpk, vpk, vmax,        \
                              (const bf16_t*)weights, indices, slope, (const bf16_t*)swa_o, (bf16_t*)o, lse, fine, dm)
  if (D == 64 && Dv == 64) GA_CALL(64, 64);
  else if (D == 128 && Dv == 128) GA_CALL(128, 128);
  else if (D == 64 && Dv == 128) GA_CALL(64, 128);
  else if (D == 128 && Dv == 64) GA_CALL(128, 64);
#undef GA_CALL
  if (rc != HILS_OK) return rc < 0 ? HILS_OK : rc;
  *handled = 1;
  return HILS_OK;
}

// The operands of the backward's dQ kernel.
void hils_bw_pack_launch(const void* k, const void* v, bf16_t* ka, bf16_t* va, bf16_t* kt, float* kmax, float* vmax,
                         int B, int Lkv, int H, int D, int Dv, void* stream) {
  pack_kv_launch<true>(k, v, ka, va, kt, kmax, vmax, B, Lkv, H, D, Dv, (hipStream_t)stream);
}

extern "C" int hils_pack_kv_chunks(const void* k, const void* v, void* workspace, size_t workspace_bytes,
                                   int B, int Lkv, int H, int D, int Dv, void* stream) {
  HILS_REQUIRE(k && v && workspace, "hils_pack_kv_chunks: null pointer");
  HILS_REQUIRE(B > 0 && Lkv >= GA_S && H > 0 && (D == 64 || D == 128) && (Dv == 64 || Dv == 128),
               "hils_pack_kv_chunks: bad sizes (Lkv >= 64, D and Dv in {64, 128})");
  HILS_REQUIRE(H <= 65535 && B <= 65535, "hils_pack_kv_chunks: H/B too large for the grid");
  const int nchunk = Lkv / GA_S;
  {
    const size_t need = ga_vt_bytes(B, H, nchunk, Dv) + ga_vt_bytes(B, H, nchunk, D) + ga_vmax_bytes(B, H, nchunk);
    HILS_REQUIRE(workspace_bytes >= need,
                 "hils_pack_kv_chunks: workspace of %zu bytes is shorter than the %zu bytes the packed K, V and "
                 "per-chunk maxima of this shape take", workspace_bytes, need);
  }
  bf16_t* vpk = (bf16_t*)workspace;
  bf16_t* kpk = (bf16_t*)((char*)workspace + ga_vt_bytes(B, H, nchunk, Dv));
  float* vmax = (float*)((char*)kpk + ga_vt_bytes(B, H, nchunk, D));
  pack_kv_launch<false>(k, v, kpk, vpk, nullptr, nullptr, vmax, B, Lkv, H, D, Dv, (hipStream_t)stream);
  HILS_CHECK_LAUNCH("hils_pack_kv_chunks");
  return HILS_OK;
}

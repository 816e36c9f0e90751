// Exact per-chunk log Z: log_z[b,t,h,c] = log sum_{j in chunk c} exp(sm_scale * <q_t, k_j>)
// over chunks that lie fully before the query's local window.
#include "common.h"
#include "stream_tiles.h"
#include "../../include/hils_amd.h"
#include <type_traits>

#define LZ_THREADS 256

struct LzDims {
  int L, HQ, H, G, D, S, W, N, mask_lmk;
  float sm_scale;
};

// number of fully-remote chunks of query t: chunk c counts iff t >= (c+1)*S + W - 1
__device__ __forceinline__ int lz_limit(const LzDims& dm, int t) {
  int lm = floordiv(t - dm.W + 1, dm.S);
  return lm < 0 ? 0 : (lm > dm.N ? dm.N : lm);
}

// One block per (b, t, hq); wavefront w takes chunks w, w+4, ...; lanes take tokens.
__global__ void __launch_bounds__(LZ_THREADS)
logz_fwd_simple(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
                float* __restrict__ log_z, LzDims dm) {
  extern __shared__ float smem[];
  float* q_s = smem;  // D
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long row = blockIdx.x;  // (b*L + t)*HQ + hq
  const int hq = (int)(row % dm.HQ);
  const long bt = row / dm.HQ;
  const int t = (int)(bt % dm.L);
  const long b = bt / dm.L;
  const int hk = hq / dm.G;
  for (int d = tid; d < dm.D; d += LZ_THREADS) q_s[d] = bf2f(q[row * dm.D + d]);
  __syncthreads();
  const int lim = lz_limit(dm, t);
  float* out = log_z + row * (long)dm.N;
  for (int c = wave; c < dm.N; c += LZ_THREADS / 64) {
    if (c >= lim) {
      if (lane == 0) out[c] = HILS_NEG_INF;
      continue;
    }
    float m = HILS_NEG_INF, l = 0.f;
    for (int s = lane; s < dm.S; s += 64) {
      const int j = c * dm.S + s;
      if (j > t || j >= dm.L) continue;
      if (dm.mask_lmk && ((j + 1) % dm.S) == 0) continue;
      const bf16_t* kr = k + ((b * dm.L + j) * (long)dm.H + hk) * dm.D;
      float a = 0.f;
      for (int d8 = 0; d8 < dm.D / 8; ++d8) {
        float f[8];
        unpack8(*(const uint4*)(kr + d8 * 8), f);
#pragma unroll
        for (int i = 0; i < 8; ++i) a = fmaf(q_s[d8 * 8 + i], f[i], a);
      }
      a *= dm.sm_scale;
      const float mn = fmaxf(m, a);
      l = l * __expf(m - mn) + __expf(a - mn);
      m = mn;
    }
    const float mx = wave_max(m);
    float part = (m > HILS_NEG_INF) ? l * __expf(m - mx) : 0.f;
    part = wave_sum(part);
    if (lane == 0) out[c] = (part > 0.f) ? mx + logf(part) : HILS_NEG_INF;
  }
}

#define LZ_ROWS 32  // score rows per wavefront

// Workgroup order of the matrix-core kernels: one-dimensional grids in which the blocks of a
// (batch, KV head) unit run on one XCD (the hardware hands consecutive workgroup ids to the 8 XCDs in
// turn: id -> (xcd, slot)), so that the keys (or query rows) the unit's workgroups stream are fetched into
// one L2 once instead of into all eight.  A unit count that is no multiple of 8 has its blocks dealt out to
// 2, 4 or 8 XCDs in turn, so that all of them work (two units on two XCDs left three quarters of the chip
// idle).  False for padding ids.
__host__ __device__ __forceinline__ int lz_units_apart(int n_unit) {  // units that run side by side
  return (n_unit & 7) == 0 ? 8 : (n_unit & 3) == 0 ? 4 : (n_unit & 1) == 0 ? 2 : 1;
}
__device__ __forceinline__ bool lz_xcd_unit(int n_blk, int n_unit, int& unit, int& blk) {
  const int g = lz_units_apart(n_unit), m = 8 / g, per = (n_blk + m - 1) / m;
  const int xcd = (int)(blockIdx.x % 8), slot = (int)(blockIdx.x / 8);
  unit = (slot / per) * g + xcd / m;
  blk = (slot % per) * m + xcd % m;
  return blk < n_blk;
}
static dim3 lz_xcd_grid(int n_blk, int n_unit) {
  const int g = lz_units_apart(n_unit), m = 8 / g;
  return dim3((unsigned)(8l * (n_unit / g) * ((n_blk + m - 1) / m)));
}
// ---- streamed tiles of the matrix-core kernels: global memory -> LDS without registers in between -------
// A wavefront's load brings 64 pieces of 16 bytes to consecutive LDS places; which piece a lane fetches is free, so the
// tile's rows lie without padding and piece p of row r at p ^ lz_swz(r): conflict-free (4 cycles a wavefront instruction,
// 8 with rows 16 bytes apart) for the 16-byte row reads of a 32x32 operand and for the transposing reads.
// The loads are inline assembly that the compiler's wait counts do not know: the kernels wait by hand, for all but the
// loads of the last step (vector-memory operations complete in order).
template <int D>
__device__ __forceinline__ int lz_swz(int r) {
  return D == 128 ? (r & 3) << 2 | (r >> 2 & 3) : (r >> 1 & 1) << 2 | (r >> 2 & 3);
}
__device__ __forceinline__ unsigned long long lz_uniform(unsigned long long x) {
  return (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)x) |
         (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(x >> 32)) << 32;
}
__device__ __forceinline__ unsigned lz_lds_addr(const unsigned char* p) {
  return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)p;
}
// (M0, which both statements set, is a register that the compiler never holds a variable in: it warns that naming it cannot
// preserve it.  Named, its own settings of M0 are not taken to last over the statement, which is what is wanted.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// 64 pieces of 16 bytes, lane i's from base + off to lds + 16 i
__device__ __forceinline__ void lz_dma16(unsigned lds, unsigned off, unsigned long long base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
// 64 words, lane i's from addr to lds + 4 i
__device__ __forceinline__ void lz_dma4(unsigned lds, unsigned long long addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds), "v"(addr) : "memory", "m0");
}
#pragma clang diagnostic pop
template <int N>
__device__ __forceinline__ void lz_landed() {  // all but the last N vector-memory operations
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ float lz_halves_sum(float x) {
  const hils_uint2v y = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(y.x) + __uint_as_float(y.y);
}
__device__ __forceinline__ float lz_halves_max(float x) {
  const hils_uint2v y = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(y.x), __uint_as_float(y.y));
}
// Steps 0 .. n-1, four a round: the buffers' numbers are constants, and so the LDS addresses fixed registers
// and immediate offsets.
template <typename F>
__device__ __forceinline__ void lz_walk(int n, F&& step) {
  for (int c = 0; c < n; c += 4) {
    step(c, std::integral_constant<int, 0>{});
    if (c + 1 < n) step(c + 1, std::integral_constant<int, 1>{});
    if (c + 2 < n) step(c + 2, std::integral_constant<int, 2>{});
    if (c + 3 < n) step(c + 3, std::integral_constant<int, 3>{});
  }
}

// Matrix-core forward for 64-token chunks.  A workgroup of four wavefronts owns 128/G consecutive queries of one KV head
// (a wavefront: 32 score rows, query x head of the group) and walks the chunks that are remote for its last query.  A
// wavefront forms the TRANSPOSED scores K Q^T of 32 tokens at a time on 32x32x16 products, so that the 32 tokens of a row
// lie in 16 registers of 2 lanes: the log-sum-exp is in-lane work and one half swap.  The products of the next 32 tokens
// are issued between the exponentials of these (matrix and vector instructions of one wavefront overlap, those of two
// that run in step hardly do), their operands read a stage before.
// Bound by the chip's power: at L 8192, 32/8 heads of 128 it runs at 1.9 to 2.0 of 2.4 GHz, about 1000 cycles for the 32 x 64
// scores of a wavefront against 1170 with 16x16x32 products that waited for their LDS reads and for each other; 325 -> 287 us
// there, 136 -> 107 at 16/2 heads of 64, 75 -> 54 at L 4096 16/16 heads of 64, 26 -> 19 at L 1200 32/8 of 128 (64 rows a
// wavefront, half the LDS reads: 285, 131, 57 and 29 us).  Times at the power limit are the card's: two others took 314 and
// 322 us for the first.
template <int D, int G>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 64 ? 3 : 2, D == 64 ? 3 : 2)))
logz_fwd_mfma(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
              float* __restrict__ log_z, LzDims dm, int n_qt, int n_unit) {
  constexpr int KS = D / 16;
  constexpr int QW = LZ_ROWS / G;       // queries per wavefront
  constexpr int QB = 4 * QW;            // queries per workgroup
  constexpr int NP = D / 32;            // loads of a chunk per wavefront
  constexpr int NB = 4, TB = 64 * D * 2;
  __shared__ __align__(16) unsigned char k_s[NB * TB];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, h = lane >> 5;
  int unit, qt;
  if (!lz_xcd_unit(n_qt, n_unit, unit, qt)) return;
  qt = n_qt - 1 - qt;  // longest rows first
  const int hk = unit % dm.H;
  const long b = unit / dm.H;
  const int t0 = qt * QB + wave * QW;

  bf16x8_t qa[KS];
  const int t = t0 + col / G;
  const bool live = t < dm.L;
  const int lim = live ? lz_limit(dm, t) : 0;
  const long orow = (b * dm.L + (live ? t : dm.L - 1)) * (long)dm.HQ + hk * G + col % G;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qa[ks] = *(const bf16x8_t*)(q + orow * D + h * 8 + ks * 16);
  float* const z_row = log_z + orow * dm.N + h;
  int t_last = qt * QB + QB - 1;
  if (t_last > dm.L - 1) t_last = dm.L - 1;
  const int nc = __builtin_amdgcn_readfirstlane(lz_limit(dm, t_last));  // chunks the workgroup walks
  const float sc2 = dm.sm_scale * HILS_LOG2E;

  const unsigned long long k_unit = lz_uniform((unsigned long long)(k + (b * dm.L * (long)dm.H + hk) * D));
  const unsigned k_step = 64u * dm.H * D * 2u;
  unsigned k_off[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int x = (wave * NP + i) * 64 + lane, row = x / (D / 8), pc = x % (D / 8);
    k_off[i] = (unsigned)(row * (dm.H * D) + (pc ^ lz_swz<D>(row)) * 8) * 2u;
  }
  const unsigned lds0 = __builtin_amdgcn_readfirstlane(lz_lds_addr(k_s) + wave * (NP * 1024));
  auto fetch = [&](int c, int buf) __attribute__((always_inline)) {  // (past the walk: its last chunk again)
    const unsigned long long kc = lz_uniform(k_unit + (unsigned long long)(unsigned)(c < nc ? c : nc - 1) * k_step);
#pragma unroll
    for (int i = 0; i < NP; ++i) lz_dma16(lds0 + buf * TB + i * 1024, k_off[i], kc);
  };
  unsigned r_off[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) r_off[ks] = (unsigned)(col * (D * 2) + ((2 * ks + h) ^ lz_swz<D>(col)) * 16);
  auto read_tile = [&](bf16x8_t (&x)[KS], int buf, int tt) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) x[ks] = *(const bf16x8_t*)(k_s + (r_off[ks] + buf * TB + tt * 32 * (D * 2)));
  };
  auto products = [&](const bf16x8_t (&x)[KS], f32x16_t& st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 16; ++i) st[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[ks], qa[ks], st, 0, 0, 0);
  };
  float keep = 0.f;
  float ref = 0.f;   // reference point of the exponentials: the last chunk's log sum (log2 units)
  bool far = true;   // (uniform) it was not near its predecessor: the next one's maximum is taken at once
  const float last = dm.mask_lmk && h == 1 ? 0.f : 1.f;  // what token 63 (register 15 of the second tile) counts for
  float s[2];
  auto stage = [&](const bf16x8_t (&x)[KS], f32x16_t& nx, const f32x16_t& cu, bool second) __attribute__((always_inline)) {
    products(x, nx);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float e = __builtin_amdgcn_exp2f(fmaf(cu[i], sc2, -ref));
      if (second && i == 15) s[1] = fmaf(e, last, s[1]);
      else s[i & 1] += e;
    }
#pragma unroll
    for (int i = 0; i < KS; ++i) {  // a product, the additions and fused ones of 16 / KS exponentials, those
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 32 / KS, 0);
      __builtin_amdgcn_sched_group_barrier(0x400, 16 / KS, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto about_max = [&](const f32x16_t& y0, const f32x16_t& y1, float& m) __attribute__((always_inline)) {
    const float x63 = last == 0.f ? HILS_NEG_INF : y1[15];
    m = fmaxf(y0[15], x63);
#pragma unroll
    for (int i = 0; i < 15; ++i) m = fmaxf(fmaxf(m, y0[i]), y1[i]);
    m = lz_halves_max(m) * sc2;  // in log2 units, as the sum below
    float p0 = 0.f, p1 = __builtin_amdgcn_exp2f(fmaf(x63, sc2, -m));
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      p0 += __builtin_amdgcn_exp2f(fmaf(y0[i], sc2, -m));
      if (i < 15) p1 += __builtin_amdgcn_exp2f(fmaf(y1[i], sc2, -m));
    }
    return lz_halves_sum(p0 + p1);
  };
  bf16x8_t a0[KS], a1[KS];
  f32x16_t xa, xb;  // scores of this chunk's first tile; second tile
  auto step = [&](int c, auto bc) __attribute__((always_inline)) {
    constexpr int B0 = decltype(bc)::value, B1 = (B0 + 1) % NB, B3 = (B0 + 3) % NB;
    lz_landed<NP>();  // chunk c + 1
    lds_barrier();    // ... of all wavefronts; chunk c - 1 has been read
    fetch(c + 3, B3);
    // The reference point need not be the maximum, only near it: the exponents of the terms that count and the log of
    // the sum are rounded at the size of their distance from it.  The previous chunk's log sum serves while the
    // sums of the whole wavefront stay within [1/8, 8] of it, which scores of a standard deviation of 1 do (the error
    // against 64 bits is then a tenth below the maximum's; within 2^60 it was up to 1.2 times it with peaked
    // scores); else the maximum is taken, at once where the last chunk's sum was not near its predecessor's, or going
    // through the chunk again.  The scale is applied inside the exponent's fused multiply-add.
    float m = ref, sum;
    read_tile(a0, B1, 0);
    if (!far) {
      s[0] = s[1] = 0.f;
      __builtin_amdgcn_sched_barrier(0);
      stage(a1, xb, xa, false);
      read_tile(a1, B1, 1);
      __builtin_amdgcn_sched_barrier(0);
      stage(a0, xa, xb, true);
      sum = lz_halves_sum(s[0] + s[1]);
      far = __any(!(sum > 0.125f && sum < 8.f));
      if (far) {
        bf16x8_t x[KS];
        f32x16_t y0, y1;
        read_tile(x, B0, 0);
        products(x, y0);
        read_tile(x, B0, 1);
        products(x, y1);
        sum = about_max(y0, y1, m);
      }
    } else {
      products(a1, xb);
      read_tile(a1, B1, 1);
      sum = about_max(xa, xb, m);
      products(a0, xa);
    }
    const float lse2 = m + __builtin_amdgcn_logf(sum);
    if (far) far = __any(!(fabsf(lse2 - ref) < 1.5f));  // (well inside: a chunk gone through twice costs 1.7 times)
    ref = lse2;
    const float val = (c < lim) ? lse2 * HILS_LN2 : HILS_NEG_INF;
    if (h == (c & 1)) keep = val;
    if ((c & 1) || c == nc - 1) {
      if (live && (c & ~1) + h <= c) z_row[c & ~1] = keep;
    }
  };
  if (nc > 0) {
    fetch(0, 0);
    fetch(1, 1);
    lz_landed<NP>();
    lds_barrier();
    fetch(2, 2);
    read_tile(a0, 0, 0);
    read_tile(a1, 0, 1);
    products(a0, xa);
    lz_walk(nc, step);
    lz_landed<0>();
  }
  // chunks past the workgroup's walk are not remote for any of its rows
  for (int r = 0; r < LZ_ROWS; ++r) {
    const int t = t0 + r / G, g = r % G;
    if (t >= dm.L) break;
    float* out = log_z + ((b * dm.L + t) * (long)dm.HQ + hk * G + g) * dm.N;
    for (int c = nc + lane; c < dm.N; c += 64) out[c] = HILS_NEG_INF;
  }
}

// ---- matrix-core backward -------------------------------------------------------------------
// Both gradients are a pair of products around the same element-wise step
//   dS[row, tok] = d_log_z[row, c(tok)] * exp(s[row, tok] - log_z[row, c(tok)]) * sm_scale
//   dQ = dS K,   dK = dS^T Q.
// One side of the product is OWNED by a wavefront (32 rows, held in registers as matrix operands,
// with the fp32 gradient accumulators), the other side STREAMS through LDS in 64-row tiles, stored
// row-major: the operand of the score product is a row read, that of the gradient product
// (whose contraction runs over the streamed rows) comes through the transposing LDS load.  With a second, transposed
// copy in LDS a tile took 16 lane permutations, 8 more stores and two barriers; L 8192, 32/8 heads of 128: dQ
// 715 -> 530 us, dK 840 -> 635 us.
// The scores are computed with the owned side as matrix columns, so their accumulator registers are already an operand of
// the gradient product.
// dQ: a wavefront owns 32 score rows (query x head), the chunks' keys stream 32 tokens at a time: the scores of the next
// 32, the exponentials of these and the gradient product of the last ones are independent, and one wavefront's vector
// instructions run beside its matrix ones.  32x32x16 products; four buffers, loaded without registers between, the keys three
// chunks ahead and the rows' log_z and d_log_z two.  Bound by the chip's power: L 8192, 32/8 heads of 128 in 2720 cycles a chunk and pair of
// workgroups instead of 4010, but at 1.55 GHz instead of 2.1, 522 -> 471 us (1.16 PFLOP/s; a large plain product 1.39);
// 180 -> 150 us at 16/2 heads of 64, 79 -> 61 at L 4096 16/16 of 64, 29 -> 22 at L 1200 32/8 of 128.  The same for dK, whose factors
// differ by register instead of by lane, spilled and was slower.  (Two other cards: 495 and 528 us.)
template <int D, int G>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
logz_bwd_dq_mfma(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
                 const float* __restrict__ log_z, const float* __restrict__ d_log_z,
                 bf16_t* __restrict__ dq, LzDims dm, int n_qt, int n_unit) {
  typedef short lz_s4 __attribute__((ext_vector_type(4)));
  typedef short lz_s8 __attribute__((ext_vector_type(8)));
  typedef unsigned lz_u4 __attribute__((ext_vector_type(4)));
  constexpr int KS = D / 16, DT = D / 32;
  constexpr int QW = LZ_ROWS / G, QB = 4 * QW;
  constexpr int NP = D / 32;  // loads of a chunk per wavefront
  constexpr int NB = 4, TB = 64 * D * 2;
  __shared__ __align__(16) unsigned char k_s[NB * TB + 4 * NB * 256];  // keys; a wavefront's log_z and d_log_z of a chunk
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, h = lane >> 5;
  int unit, qt;
  if (!lz_xcd_unit(n_qt, n_unit, unit, qt)) return;
  qt = n_qt - 1 - qt;
  const int hk = unit % dm.H;
  const long b = unit / dm.H;
  const int t = qt * QB + wave * QW + col / G;
  const bool live = t < dm.L;
  const int lim = live ? lz_limit(dm, t) : 0;
  const long orow = ((b * dm.L + (live ? t : dm.L - 1)) * (long)dm.HQ + hk * G + col % G);
  bf16x8_t qa[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qa[ks] = *(const bf16x8_t*)(q + orow * D + h * 8 + ks * 16);
  int t_last = qt * QB + QB - 1;
  if (t_last > dm.L - 1) t_last = dm.L - 1;
  const int nc = __builtin_amdgcn_readfirstlane(lz_limit(dm, t_last));
  const float sc2 = dm.sm_scale * HILS_LOG2E;

  const unsigned long long k_unit = lz_uniform((unsigned long long)(k + (b * dm.L * (long)dm.H + hk) * D));
  const unsigned k_step = 64u * dm.H * D * 2u;
  unsigned k_off[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int x = (wave * NP + i) * 64 + lane, row = x / (D / 8), pc = x % (D / 8);
    k_off[i] = (unsigned)(row * (dm.H * D) + (pc ^ lz_swz<D>(row)) * 8) * 2u;
  }
  const unsigned lds0 = __builtin_amdgcn_readfirstlane(lz_lds_addr(k_s) + wave * (NP * 1024));
  const unsigned z_lds = __builtin_amdgcn_readfirstlane(lz_lds_addr(k_s) + NB * TB + wave * (NB * 256));
  // lanes 0..31 bring log_z of the wavefront's rows, the others d_log_z
  const unsigned long long z_lane = (unsigned long long)((h ? d_log_z : log_z) + orow * dm.N);
  auto fetch = [&](int c, int buf) __attribute__((always_inline)) {  // (past the walk: its last chunk again)
    const unsigned long long kc = lz_uniform(k_unit + (unsigned long long)(unsigned)(c < nc ? c : nc - 1) * k_step);
#pragma unroll
    for (int i = 0; i < NP; ++i) lz_dma16(lds0 + buf * TB + i * 1024, k_off[i], kc);
  };
  auto fetch_z = [&](int c, int buf) __attribute__((always_inline)) {
    lz_dma4(z_lds + buf * 256, z_lane + (unsigned)(c < nc ? c : nc - 1) * 4u);
  };
  // LDS addresses: rows of a 32-token tile (operand of the scores), columns of 16 tokens (of the gradient)
  unsigned r_off[KS], c_off[DT];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) r_off[ks] = (unsigned)(col * (D * 2) + ((2 * ks + h) ^ lz_swz<D>(col)) * 16);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    const int l = lane & 15, row = 4 * h + (l >> 2), pc = dt * 4 + (lane >> 4 & 1) * 2 + (l >> 1 & 1);
    c_off[dt] = (unsigned)(row * (D * 2) + (pc ^ lz_swz<D>(row)) * 16 + (l & 1) * 8);
  }
  f32x16_t acc[DT], sa, sb;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;
  bf16x8_t ra[KS], ca[2][DT], pp[2];
  auto read_row = [&](int ks, int buf, int tt) __attribute__((always_inline)) {
    ra[ks] = *(const bf16x8_t*)(k_s + (r_off[ks] + buf * TB + tt * 32 * (D * 2)));
  };
  auto read_col = [&](int s, int dt, int buf, int tt) __attribute__((always_inline)) {
    const int imm = buf * TB + (tt * 32 + s * 16) * (D * 2);
    unsigned down;  // the same piece eight rows further down: the swizzle's bit 1 (worked out here: four registers less)
    asm volatile("v_xor_b32 %0, 32, %1" : "=v"(down) : "v"(c_off[dt]));
    const lz_s4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lz_s4*)(k_s + (c_off[dt] + imm)));
    const lz_s4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lz_s4*)(k_s + (down + (imm + 8 * (D * 2)))));
    ca[s][dt] = __builtin_bit_cast(bf16x8_t, (lz_s8)__builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  float off = 0.f, coef = 0.f;
  // One stage: scores of the next tile (nx), exponentials of this one's (cu), gradient product of the last one's (pp, ca).
  // The next stage's operands are read behind the last use of these: rows of tile rtt of rbuf, columns of this tile.
  auto stage = [&](f32x16_t& nx, const f32x16_t& cu, int rbuf, int rtt, int cbuf, int ctt) __attribute__((always_inline)) {
    float p[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) nx[i] = 0.f;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      nx = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ra[u], qa[u], nx, 0, 0, 0);
      read_row(u, rbuf, rtt);
      const int s = u / DT, dt = u % DT;
      acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ca[s][dt], pp[s], acc[dt], 0, 0, 0);
      read_col(s, dt, cbuf, ctt);
#pragma unroll
      for (int i = u * 16 / KS; i < (u + 1) * 16 / KS; ++i) p[i] = __builtin_amdgcn_exp2f(fmaf(cu[i], sc2, -off)) * coef;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      lz_u4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = pack_bf2(p[s * 8 + 2 * e], p[s * 8 + 2 * e + 1]);
      pp[s] = __builtin_bit_cast(bf16x8_t, x);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // (step c asks for the keys of chunk c + 3 and the row values of c + 2)
  auto step = [&](int c, auto bc) __attribute__((always_inline)) {
    constexpr int B0 = decltype(bc)::value, B1 = (B0 + 1) % NB, B2 = (B0 + 2) % NB, B3 = (B0 + 3) % NB;
    lz_landed<NP + 1>();  // the keys of chunk c + 1, the row values of c
    lds_barrier();        // ... of all wavefronts; chunk c - 1 has been read
    const float* zs = (const float*)(k_s + (NB * TB + wave * (NB * 256) + B0 * 256 + col * 4));
    const float lz = zs[0], dz = zs[32];
    const bool ok = c < lim && lz > -1e30f;
    off = ok ? lz * HILS_LOG2E : INFINITY;  // (no probability but 0, however large the score)
    coef = ok ? dz * dm.sm_scale : 0.f;
    fetch(c + 3, B3);
    fetch_z(c + 2, B2);
    __builtin_amdgcn_sched_barrier(0);
    stage(sb, sa, B1, 0, B0, 0);
    stage(sa, sb, B1, 1, B0, 1);
  };
  if (nc > 0) {
    fetch(0, 0);
    fetch_z(0, 0);
    fetch(1, 1);
    fetch_z(1, 1);
    lz_landed<NP + 1>();
    lds_barrier();
    fetch(2, 2);
    // the first tile's scores; the gradient product before it is one with zeros
#pragma unroll
    for (int u = 0; u < KS; ++u) read_row(u, 0, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i) sa[i] = 0.f;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      sa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ra[u], qa[u], sa, 0, 0, 0);
      read_row(u, 0, 1);
      read_col(u / DT, u % DT, 0, 0);
    }
    pp[0] = pp[1] = __builtin_bit_cast(bf16x8_t, (lz_s8)(0));
    lz_walk(nc, step);
#pragma unroll
    for (int u = 0; u < KS; ++u)  // of the last tile
      acc[u % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ca[u / DT][u % DT], pp[u / DT], acc[u % DT], 0, 0, 0);
    lz_landed<0>();
  }
  if (!live) return;
  bf16_t* out = dq + orow * D + 4 * h;  // a lane holds four neighbouring features of its row
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint2 x;
      x.x = pack_bf2(acc[dt][4 * e], acc[dt][4 * e + 1]);
      x.y = pack_bf2(acc[dt][4 * e + 2], acc[dt][4 * e + 3]);
      *(uint2*)(out + dt * 32 + e * 8) = x;
    }
}

// dK: a workgroup owns two chunks (wavefront: 32 tokens of one chunk), the score rows of the
// queries behind them stream in tiles of 64 rows (64/G queries x G heads).  The first chunks have the whole
// sequence behind them, the last ones nothing: walks are cut into segments of about equal length whose fp32
// sums logz_bwd_dk_sum adds up.  With one workgroup per pair of chunks the kernel ran as long as the first
// pair's walk: L 8192, 32/8 heads of 128: 1010 us, in segments 880 us; forward and both gradients at L 3532,
// 16/2 heads of 64: 707 us, in segments and with the units dealt out to all XCDs 202 us.
struct LzSeg {
  int target;   // tiles of a segment, about
  int max_seg;  // segments of the longest walk (1: no walk is cut)
};
__host__ __device__ __forceinline__ int lz_tile0(int pair, int W, int QT) {  // first tile behind a pair's first chunk
  const int t = (2 * pair + 1) * 64 + W - 1;
  return t < 0 ? 0 : t / QT;
}
__host__ __device__ __forceinline__ int lz_nseg(int len, const LzSeg& sg) {
  int n = len > 0 ? (len + sg.target / 2) / sg.target : 1;
  return n < 1 ? 1 : (n > sg.max_seg ? sg.max_seg : n);
}
template <int D, int G>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 64 ? 3 : 2, D == 64 ? 3 : 2)))
logz_bwd_dk_mfma(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
                 const float* __restrict__ log_z, const float* __restrict__ d_log_z,
                 bf16_t* __restrict__ dk, LzDims dm, int n_pair, int n_unit, LzSeg sg, float* __restrict__ part) {
  constexpr int KS = D / 32, DT = D / 16;
  constexpr int QT = 64 / G;  // queries per streamed tile
  constexpr int PITCH = D * 2 + 32;
  constexpr int NP = D / 32;  // 16-byte pieces of a tile per thread
  __shared__ __align__(16) unsigned char q_s[2][64 * PITCH];
  __shared__ __align__(16) float off_s[2][2][64];
  __shared__ __align__(16) float coef_s[2][2][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, j = lane >> 4;
  // Workgroup order.  The workgroups of one (batch, KV head) stream the same query rows, each from the
  // first query behind its chunks to the last one: they walk the tiles from the END, so that all of
  // them are on the same tile at the same time, and the one-dimensional grid puts them on one XCD
  // (the hardware hands consecutive workgroup ids to the 8 XCDs in turn: id -> (xcd, slot)), whose L2
  // then serves all but the first reader of a tile.  Walking forward from different starting points
  // in the hardware's order, every read of a tile missed (L2 hit rate 2 %, the kernel waiting on
  // HBM latency at one wavefront per SIMD).  The chunk pairs of a unit come longest walk first; of the
  // segments the last ones (which only long walks have) start first, so that the short walks fill the end.
  int unit, pair;
  if (!lz_xcd_unit(n_pair * sg.max_seg, n_unit, unit, pair)) return;
  const int seg_i = sg.max_seg - 1 - pair / n_pair;
  pair %= n_pair;
  const int c0 = 2 * pair, ch = wave >> 1;
  const int hk = unit % dm.H;
  const long b = unit / dm.H;
  const int tok0 = (c0 + ch) * 64 + (wave & 1) * 32;  // first owned token

  bf16x8_t ka[2][KS];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    int tok = tok0 + tt * 16 + col;
    if (tok > dm.L - 1) tok = dm.L - 1;  // such tokens get no gradient: every coefficient is 0
    const bf16_t* kp = k + ((b * dm.L + tok) * (long)dm.H + hk) * D + j * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) ka[tt][ks] = *(const bf16x8_t*)(kp + ks * 32);
  }
  // first query with chunk c0 fully behind its window, rounded down to a tile
  int tile0 = lz_tile0(pair, dm.W, QT);
  int n_tiles = (dm.L + QT - 1) / QT;
  const int n_seg = lz_nseg(n_tiles - tile0, sg);
  if (seg_i >= n_seg) return;
  if (n_seg > 1) {  // segment 0 has the last tiles
    const int len = n_tiles - tile0, hi = n_tiles;
    n_tiles = hi - (int)((long)len * seg_i / n_seg);
    tile0 = hi - (int)((long)len * (seg_i + 1) / n_seg);
  }
  const float sc2 = dm.sm_scale * HILS_LOG2E;

  // staging: a uniform base per tile and fixed lane offsets; only the sequence's last tile may reach past its end,
  // and its rows there read the last query again (their coefficients are 0)
  typedef unsigned lz_u32x4 __attribute__((ext_vector_type(4)));
  lz_u32x4 qr[NP];
  float zo = 0.f, zc = 0.f;  // raw log_z and d_log_z of this thread's (row, chunk); zin: inside the limits
  bool zin = false;
  const long q_row = (long)dm.HQ * D, z_row = (long)dm.HQ * dm.N;  // of one query
  const bf16_t* const q_unit = q + b * dm.L * q_row + hk * G * D;
  const float* const z_unit = log_z + b * dm.L * z_row + (long)hk * G * dm.N;
  const float* const dz_unit = d_log_z + b * dm.L * z_row + (long)hk * G * dm.N;
  const int z_r = tid & 63, z_c = c0 + (tid >> 6 & 1);  // row and chunk of this thread's coefficient (the first 128)
  const int z_cc = z_c < dm.N ? z_c : dm.N - 1;
  const int z_t0 = z_c < dm.N ? (z_c + 1) * 64 + dm.W - 1 : 0x7fffffff;  // first query with the chunk behind its window
  auto fetch = [&](int tile) __attribute__((always_inline)) {
    const int last = dm.L - 1 - tile * QT;  // last query of the sequence, counted from the tile's first
    const bf16_t* qc = q_unit + (long)tile * QT * q_row;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int row = (tid + 256 * i) / (D / 8);
      const int t = row / G < last ? row / G : last;
      qr[i] = *(const lz_u32x4*)(qc + (unsigned)((t * dm.HQ + row % G) * D + (tid + 256 * i) % (D / 8) * 8));
    }
    if (tid < 128) {
      // raw values: what a row outside the limits gets is decided in stash(), so that nothing
      // here waits for a load (which would also wait for the query rows issued before it)
      const int tr = z_r / G, t = tr < last ? tr : last;
      const unsigned zi = (unsigned)((t * dm.HQ + z_r % G) * dm.N + z_cc);
      zo = (z_unit + (long)tile * QT * z_row)[zi];
      zc = (dz_unit + (long)tile * QT * z_row)[zi];
      zin = tr <= last && tile * QT + tr >= z_t0;
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NP; ++i)
      *(lz_u32x4*)(&q_s[buf][(tid + 256 * i) / (D / 8) * PITCH + (tid + 256 * i) % (D / 8) * 16]) = qr[i];
    if (tid < 128) {
      const bool ok = zin && zo > -1e30f;
      off_s[buf][tid >> 6][tid & 63] = ok ? zo * HILS_LOG2E : INFINITY;  // (no probability but 0, however large the score)
      coef_s[buf][tid >> 6][tid & 63] = ok ? zc * dm.sm_scale : 0.f;
    }
  };
  f32x4_t acc[2][DT];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[tt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (tile0 < n_tiles) {
    fetch(n_tiles - 1);
    stash(0);
  }
  __syncthreads();
  for (int tile = n_tiles - 1, buf = 0; tile >= tile0; --tile, buf ^= 1) {
    fetch(tile > tile0 ? tile - 1 : tile);
    __builtin_amdgcn_sched_barrier(0);
    const unsigned char* qb = q_s[buf];
    float p[2][4][4];  // [owned token tile][streamed row tile][row 4j+i]
    {
      f32x4_t st[2][4];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) st[tt][rr] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int rr = 0; rr < 4; ++rr)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const bf16x8_t a = *(const bf16x8_t*)(qb + (rr * 16 + col) * PITCH + ks * 64 + j * 16);
#pragma unroll
          for (int tt = 0; tt < 2; ++tt)
            st[tt][rr] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, ka[tt][ks], st[tt][rr], 0, 0, 0);
        }
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const float4 o4 = *(const float4*)&off_s[buf][ch][rr * 16 + 4 * j];
        const float4 c4 = *(const float4*)&coef_s[buf][ch][rr * 16 + 4 * j];
        const float o[4] = {o4.x, o4.y, o4.z, o4.w}, cf[4] = {c4.x, c4.y, c4.z, c4.w};
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            p[tt][rr][i] = __builtin_amdgcn_exp2f(st[tt][rr][i] * sc2 - o[i]) * cf[i];
      }
    }
    lzm_grad_product_rows<D, 2, PITCH, true>(qb, p, acc, col, j);
    stash(buf ^ 1);
    __syncthreads();
  }
  // (a lane holds a feature of four tokens.  With four features of a token, and 16-byte stores, the whole kernel was 1 to 7 %
  // slower at 54 of 60 lengths and head shapes: L2048 32/8 heads of 128 67.9 us against 64.0, L8192 582 against 573)
  if (n_seg > 1) {
    float* out = part + (((long)unit * n_pair + pair) * sg.max_seg + seg_i) * (128 * D);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) out[(wave * 32 + tt * 16 + 4 * j + i) * D + dt * 16 + col] = acc[tt][dt][i];
    return;
  }
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tok = tok0 + tt * 16 + 4 * j + i;
      if (tok >= dm.L) continue;
      bf16_t* out = dk + ((b * dm.L + tok) * (long)dm.H + hk) * D + col;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) out[dt * 16] = f2bf(acc[tt][dt][i]);
    }
}

// the segments of the cut walks, in order; four features per thread
__global__ void __launch_bounds__(256)
logz_bwd_dk_sum(const float* __restrict__ part, bf16_t* __restrict__ dk, LzDims dm, int n_pair, LzSeg sg) {
  const int pair = blockIdx.x % n_pair, unit = blockIdx.x / n_pair, QT = 64 / dm.G, D = dm.D;
  const int n_seg = lz_nseg((dm.L + QT - 1) / QT - lz_tile0(pair, dm.W, QT), sg);
  if (n_seg == 1) return;
  const int hk = unit % dm.H;
  const long b = unit / dm.H;
  const f32x4_t* src = (const f32x4_t*)(part + ((long)unit * n_pair + pair) * sg.max_seg * (128 * D));
  const int n = 128 * D / 4;
  for (int i = blockIdx.y * 256 + threadIdx.x; i < n; i += gridDim.y * 256) {
    const int t = i / (D / 4), f = (i - t * (D / 4)) * 4, tok = pair * 128 + t;
    if (tok >= dm.L) break;
    f32x4_t x = src[i];
    for (int s = 1; s < n_seg; ++s) {
      const f32x4_t y = src[(long)s * n + i];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] += y[e];
    }
    uint2 pk;
    pk.x = pack_bf2(x[0], x[1]);
    pk.y = pack_bf2(x[2], x[3]);
    *(uint2*)(dk + ((b * dm.L + tok) * (long)dm.H + hk) * D + f) = pk;
  }
}

// dq[b,t,hq,:] = sum_c sum_j dlz[c] * exp(s_j - lz[c]) * scale * k_j
__global__ void __launch_bounds__(LZ_THREADS)
logz_bwd_dq_simple(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
                   const float* __restrict__ log_z, const float* __restrict__ d_log_z,
                   bf16_t* __restrict__ dq, LzDims dm) {
  extern __shared__ float smem[];
  float* q_s = smem;          // D
  float* ds = q_s + dm.D;     // S
  const int tid = threadIdx.x;
  const long row = blockIdx.x;
  const int hq = (int)(row % dm.HQ);
  const long bt = row / dm.HQ;
  const int t = (int)(bt % dm.L);
  const long b = bt / dm.L;
  const int hk = hq / dm.G;
  for (int d = tid; d < dm.D; d += LZ_THREADS) q_s[d] = bf2f(q[row * dm.D + d]);
  const int lim = lz_limit(dm, t);
  float acc = 0.f;  // thread d (< D) owns one output column
  for (int c = 0; c < lim; ++c) {
    const float lz = log_z[row * (long)dm.N + c];
    const float dlz = d_log_z[row * (long)dm.N + c];
    __syncthreads();
    for (int s = tid; s < dm.S; s += LZ_THREADS) {
      const int j = c * dm.S + s;
      float val = 0.f;
      if (j <= t && j < dm.L && lz > -1e30f) {
        const bf16_t* kr = k + ((b * dm.L + j) * (long)dm.H + hk) * dm.D;
        float a = 0.f;
        for (int d8 = 0; d8 < dm.D / 8; ++d8) {
          float f[8];
          unpack8(*(const uint4*)(kr + d8 * 8), f);
#pragma unroll
          for (int i = 0; i < 8; ++i) a = fmaf(q_s[d8 * 8 + i], f[i], a);
        }
        val = dlz * __expf(a * dm.sm_scale - lz) * dm.sm_scale;
      }
      ds[s] = val;
    }
    __syncthreads();
    for (int d = tid; d < dm.D; d += LZ_THREADS) {
      float a = 0.f;
      for (int s = 0; s < dm.S; ++s) {
        const int j = c * dm.S + s;
        if (j < dm.L) a = fmaf(ds[s], bf2f(k[((b * dm.L + j) * (long)dm.H + hk) * dm.D + d]), a);
      }
      acc += a;  // D <= LZ_THREADS: one column per thread
    }
  }
  if (tid < dm.D) dq[row * dm.D + tid] = f2bf(acc);
}

// dk[b, c*S+s, hk, :] = sum_{g} sum_{t} dlz[t,hq,c] * exp(s - lz) * scale * q[t,hq,:]
// One block per (b, c, hk); queries are streamed in tiles of LZ_TT.
#define LZ_TT 8
#define LZ_MAX_ACC 32
__global__ void __launch_bounds__(LZ_THREADS)
logz_bwd_dk_simple(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
                   const float* __restrict__ log_z, const float* __restrict__ d_log_z,
                   bf16_t* __restrict__ dk, LzDims dm) {
  extern __shared__ float smem[];
  const int G = dm.G, S = dm.S, D = dm.D, DP = dm.D + 1;
  float* k_s = smem;                          // S*DP
  float* q_s = k_s + (size_t)S * DP;          // TT*G*D
  float* ds = q_s + (size_t)LZ_TT * G * D;    // TT*G*S
  const int tid = threadIdx.x;
  const int c = blockIdx.x, hk = blockIdx.y;
  const long b = blockIdx.z;
  for (int i = tid; i < S * D; i += LZ_THREADS) {
    const int s = i / D, d = i - s * D;
    const int j = c * S + s;
    k_s[s * DP + d] = (j < dm.L) ? bf2f(k[((b * dm.L + j) * (long)dm.H + hk) * D + d]) : 0.f;
  }
  float acc[LZ_MAX_ACC];
#pragma unroll
  for (int i = 0; i < LZ_MAX_ACC; ++i) acc[i] = 0.f;
  int t_first = (c + 1) * S + dm.W - 1;
  if (t_first < 0) t_first = 0;
  for (int t0 = t_first; t0 < dm.L; t0 += LZ_TT) {
    __syncthreads();
    for (int i = tid; i < LZ_TT * G * D; i += LZ_THREADS) {
      const int tt = i / (G * D), r = i - tt * (G * D);
      const int t = t0 + tt;
      q_s[i] = (t < dm.L) ? bf2f(q[((b * dm.L + t) * (long)dm.HQ + hk * G) * D + r]) : 0.f;
    }
    __syncthreads();
    for (int i = tid; i < LZ_TT * G * S; i += LZ_THREADS) {
      const int tt = i / (G * S), r = i - tt * (G * S);
      const int g = r / S, s = r - g * S;
      const int t = t0 + tt, j = c * S + s;
      float val = 0.f;
      if (t < dm.L && j <= t && j < dm.L) {
        const long zrow = ((b * dm.L + t) * (long)dm.HQ + hk * G + g) * dm.N + c;
        const float lz = log_z[zrow];
        if (lz > -1e30f) {
          const float* qr = q_s + (tt * G + g) * D;
          float a = 0.f;
          for (int d = 0; d < D; ++d) a = fmaf(qr[d], k_s[s * DP + d], a);
          val = d_log_z[zrow] * __expf(a * dm.sm_scale - lz) * dm.sm_scale;
        }
      }
      ds[i] = val;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < LZ_MAX_ACC; ++e) {
      const int oi = tid + e * LZ_THREADS;
      if (oi < S * D) {
        const int s = oi / D, d = oi - s * D;
        float a = acc[e];
        for (int r = 0; r < LZ_TT * G; ++r) a = fmaf(ds[r * S + s], q_s[r * D + d], a);
        acc[e] = a;
      }
    }
  }
#pragma unroll
  for (int e = 0; e < LZ_MAX_ACC; ++e) {
    const int oi = tid + e * LZ_THREADS;
    if (oi < S * D) {
      const int s = oi / D, d = oi - s * D;
      const int j = c * S + s;
      if (j < dm.L) dk[((b * dm.L + j) * (long)dm.H + hk) * D + d] = f2bf(acc[e]);
    }
  }
}

// shapes of the matrix-core kernels: 64-token chunks, head dim 64/128, group size dividing 16, and a window that is not
// negative: with one a query's walk takes in chunks that end behind it, of which it sees a part, and the ragged last chunk,
// whose rows the kernels would read past the end of the keys
static bool lz_mfma_covers(int G, int D, int S, int H, int B, int W) {
  return S == 64 && W >= 0 && (D == 64 || D == 128) && (G == 1 || G == 2 || G == 4 || G == 8 || G == 16) &&
         H <= 65535 && B <= 65535;
}
// ... the forward and dQ also need keys at a multiple of 16 bytes, which their direct loads to LDS want (loads to registers
// take any address: the general kernels and dK)
static bool lz_direct_loads(const void* k) { return (uintptr_t)k % 16 == 0; }
// expands LZ_LAUNCH(D, G) for the covered (D, G)
#define LZ_DISPATCH_G(DD, G_)                                                                  \
  switch (G_) {                                                                                \
    case 1: LZ_LAUNCH(DD, 1); break;                                                           \
    case 2: LZ_LAUNCH(DD, 2); break;                                                           \
    case 4: LZ_LAUNCH(DD, 4); break;                                                           \
    case 8: LZ_LAUNCH(DD, 8); break;                                                           \
    default: LZ_LAUNCH(DD, 16); break;                                                         \
  }
#define LZ_DISPATCH(D_, G_)                                                                    \
  if ((D_) == 64) { LZ_DISPATCH_G(64, G_) } else { LZ_DISPATCH_G(128, G_) }

static int lz_check(const char* name, int B, int L, int HQ, int H, int D, int S) {
  HILS_REQUIRE(B > 0 && L > 0 && HQ > 0 && H > 0 && D > 0 && S > 0, "%s: sizes must be positive", name);
  HILS_REQUIRE(HQ % H == 0, "%s: HQ (%d) must be a multiple of H (%d)", name, HQ, H);
  HILS_REQUIRE(D % 8 == 0, "%s: D (%d) must be a multiple of 8", name, D);
  HILS_REQUIRE((long)B * L * HQ <= 2147483647L, "%s: grid too large", name);
  return HILS_OK;
}

extern "C" int hils_chunk_logz_fwd(const void* q, const void* k, float* log_z, int B, int L, int HQ,
                                   int H, int D, int S, int window, float sm_scale, int mask_lmk,
                                   void* stream) {
  HILS_REQUIRE(q && k && log_z, "hils_chunk_logz_fwd: null pointer");
  if (int rc = lz_check("hils_chunk_logz_fwd", B, L, HQ, H, D, S)) return rc;
  LzDims dm{L, HQ, H, HQ / H, D, S, window, (L + S - 1) / S, mask_lmk, sm_scale};
  const int G = HQ / H;
  if (lz_mfma_covers(G, D, S, H, B, window) && lz_direct_loads(k)) {
    const int QB = 4 * LZ_ROWS / G;
    const int n_qt = (L + QB - 1) / QB;
    HILS_REQUIRE(((long)B * H + 8) * (n_qt + 8) < (1L << 31), "hils_chunk_logz_fwd: B * H * L too large for the grid");
    const dim3 grid = lz_xcd_grid(n_qt, B * H);
#define LZ_LAUNCH(DD, GG)                                                                      \
  hipLaunchKernelGGL((logz_fwd_mfma<DD, GG>), grid, dim3(256), 0, (hipStream_t)stream,         \
                     (const bf16_t*)q, (const bf16_t*)k, log_z, dm, n_qt, B * H)
    LZ_DISPATCH(D, G);
#undef LZ_LAUNCH
    HILS_CHECK_LAUNCH("hils_chunk_logz_fwd");
    return HILS_OK;
  }
  hipLaunchKernelGGL(logz_fwd_simple, dim3((unsigned)((long)B * L * HQ)), dim3(LZ_THREADS),
                     D * sizeof(float), (hipStream_t)stream, (const bf16_t*)q, (const bf16_t*)k,
                     log_z, dm);
  HILS_CHECK_LAUNCH("hils_chunk_logz_fwd");
  return HILS_OK;
}

extern "C" int hils_chunk_logz_bwd_dq(const void* q, const void* k, const float* log_z,
                                      const float* d_log_z, void* dq, int B, int L, int HQ, int H,
                                      int D, int S, int window, float sm_scale, void* stream) {
  HILS_REQUIRE(q && k && log_z && d_log_z && dq, "hils_chunk_logz_bwd_dq: null pointer");
  if (int rc = lz_check("hils_chunk_logz_bwd_dq", B, L, HQ, H, D, S)) return rc;
  HILS_REQUIRE(D <= LZ_THREADS, "hils_chunk_logz_bwd_dq: D (%d) must be <= %d", D, LZ_THREADS);
  LzDims dm{L, HQ, H, HQ / H, D, S, window, (L + S - 1) / S, 0, sm_scale};
  if (lz_mfma_covers(HQ / H, D, S, H, B, window) && lz_direct_loads(k)) {
    const int G = HQ / H;
    const int QB = 4 * LZ_ROWS / G;
    const int n_qt = (L + QB - 1) / QB;
    HILS_REQUIRE(((long)B * H + 8) * (n_qt + 8) < (1L << 31), "hils_chunk_logz_bwd_dq: B * H * L too large for the grid");
    const dim3 grid = lz_xcd_grid(n_qt, B * H);
#define LZ_LAUNCH(DD, GG)                                                                      \
  hipLaunchKernelGGL((logz_bwd_dq_mfma<DD, GG>), grid, dim3(256), 0, (hipStream_t)stream,      \
                     (const bf16_t*)q, (const bf16_t*)k, log_z, d_log_z, (bf16_t*)dq, dm, n_qt, B * H)
    LZ_DISPATCH(D, G);
#undef LZ_LAUNCH
    HILS_CHECK_LAUNCH("hils_chunk_logz_bwd_dq");
    return HILS_OK;
  }
  hipLaunchKernelGGL(logz_bwd_dq_simple, dim3((unsigned)((long)B * L * HQ)), dim3(LZ_THREADS),
                     (D + S) * sizeof(float), (hipStream_t)stream, (const bf16_t*)q,
                     (const bf16_t*)k, log_z, d_log_z, (bf16_t*)dq, dm);
  HILS_CHECK_LAUNCH("hils_chunk_logz_bwd_dq");
  return HILS_OK;
}

// Segments of the dK walks.  Equal shares fill the chip the better the more of them there are, but each leaves a partial
// result of as many bytes as four tiles, and a block's segments are summed one after the other: eight items per compute
// unit (two or three run at once) in segments of 40 tiles and more, five in segments of 24 and more, else three, and none
// shorter than eight tiles.  Whole backward, us, for three / five / eight items (in brackets, the tiles of a segment): L8192
// 32/8 heads of 128 [170, 102, 64] 1204 / 1175 / 1153, L8192 16/2 of 64 [85, 51, 32] 454 / 407 and 396 with 40, L5000 32/4 of
// 128 [65, 39, 24] 468 / 460 / 490, L4096 32/8 of 128 [42, 25, 16] 347 / 336, L4096 16/2 of 64 [21, 12, 8] 147 / 156 / 167,
// B2 L2048 32/8 of 128 [21, 12, 8] 179 / 185 / 197; the other way only L8192 4/4 of 64 [21, 12, 8], 174 / 167.
static LzSeg lz_segments(int B, int L, int G, int H, int N, int W) {
  const int n_pair = (N + 1) / 2, QT = 64 / G, n_tiles = (L + QT - 1) / QT;
  long total = 0;
  for (int p = 0; p < n_pair; ++p) {
    const int len = n_tiles - lz_tile0(p, W, QT);
    if (len <= 0) break;
    total += len;
  }
  const int longest = n_tiles - lz_tile0(0, W, QT);
  auto tiles = [&](long items, long most) -> long {  // of a segment with that many items per compute unit
    const long t = total * B * H / (items * hils_device_cus());
    return t < most ? t : most;
  };
  const long three = tiles(3, 24), five = tiles(5, 40), eight = tiles(8, 1 << 30);
  long target = three > five ? three : five;
  target = target > eight ? target : eight;
  if (target < 8) target = 8;
  LzSeg sg{(int)(target < (1 << 30) ? target : (1 << 30)), 1 << 30};
  sg.max_seg = lz_nseg(longest, sg);
  return sg;
}
extern "C" size_t hils_chunk_logz_bwd_dk_workspace(int B, int L, int HQ, int H, int D, int S, int window) {
  if (B <= 0 || L <= 0 || H <= 0 || HQ <= 0 || HQ % H != 0 || !lz_mfma_covers(HQ / H, D, S, H, B, window)) return 0;
  const int N = (L + S - 1) / S;
  const LzSeg sg = lz_segments(B, L, HQ / H, H, N, window);
  return sg.max_seg == 1 ? 0 : (size_t)B * H * ((N + 1) / 2) * sg.max_seg * 128 * D * sizeof(float);
}

extern "C" int hils_chunk_logz_bwd_dk_ws(const void* q, const void* k, const float* log_z,
                                         const float* d_log_z, void* dk, int B, int L, int HQ, int H,
                                         int D, int S, int window, float sm_scale, void* workspace,
                                         size_t workspace_bytes, void* stream) {
  HILS_REQUIRE(q && k && log_z && d_log_z && dk, "hils_chunk_logz_bwd_dk: null pointer");
  if (int rc = lz_check("hils_chunk_logz_bwd_dk", B, L, HQ, H, D, S)) return rc;
  const int G = HQ / H;
  HILS_REQUIRE(S * D <= LZ_MAX_ACC * LZ_THREADS, "hils_chunk_logz_bwd_dk: S*D (%d) too large", S * D);
  LzDims dm{L, HQ, H, G, D, S, window, (L + S - 1) / S, 0, sm_scale};
  if (lz_mfma_covers(G, D, S, H, B, window)) {
    const int n_pair = (dm.N + 1) / 2;
    HILS_REQUIRE(((long)B * H + 8) * (n_pair + 8) * 8 < (1L << 31), "hils_chunk_logz_bwd_dk: B * H * N too large for the grid");
    const int n_unit = B * H;
    const LzSeg sg = workspace ? lz_segments(B, L, G, H, dm.N, window) : LzSeg{1 << 30, 1};
    HILS_REQUIRE(sg.max_seg == 1 || workspace_bytes >= (size_t)n_unit * n_pair * sg.max_seg * 128 * D * sizeof(float),
                 "hils_chunk_logz_bwd_dk: the workspace is too short (%zu bytes)", workspace_bytes);
    const dim3 grid = lz_xcd_grid(n_pair * sg.max_seg, n_unit);
#define LZ_LAUNCH(DD, GG)                                                                      \
  hipLaunchKernelGGL((logz_bwd_dk_mfma<DD, GG>), grid, dim3(256), 0, (hipStream_t)stream,      \
                     (const bf16_t*)q, (const bf16_t*)k, log_z, d_log_z, (bf16_t*)dk, dm, n_pair, n_unit, sg, \
                     (float*)workspace)
    LZ_DISPATCH(D, G);
#undef LZ_LAUNCH
    if (sg.max_seg > 1)
      hipLaunchKernelGGL(logz_bwd_dk_sum, dim3((unsigned)(n_pair * n_unit), 4), dim3(256), 0, (hipStream_t)stream,
                         (const float*)workspace, (bf16_t*)dk, dm, n_pair, sg);
    HILS_CHECK_LAUNCH("hils_chunk_logz_bwd_dk");
    return HILS_OK;
  }
  size_t smem = ((size_t)S * (D + 1) + (size_t)LZ_TT * G * D + (size_t)LZ_TT * G * S) * sizeof(float);
  HILS_REQUIRE(smem <= 160 * 1024, "hils_chunk_logz_bwd_dk: tile does not fit in LDS");
  HILS_REQUIRE(H <= 65535 && B <= 65535, "hils_chunk_logz_bwd_dk: H/B too large for the grid");
  if (smem > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)logz_bwd_dk_simple,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  hipLaunchKernelGGL(logz_bwd_dk_simple, dim3(dm.N, H, B), dim3(LZ_THREADS), smem,
                     (hipStream_t)stream, (const bf16_t*)q, (const bf16_t*)k, log_z, d_log_z,
                     (bf16_t*)dk, dm);
  HILS_CHECK_LAUNCH("hils_chunk_logz_bwd_dk");
  return HILS_OK;
}

extern "C" int hils_chunk_logz_bwd_dk(const void* q, const void* k, const float* log_z,
                                      const float* d_log_z, void* dk, int B, int L, int HQ, int H,
                                      int D, int S, int window, float sm_scale, void* stream) {
  return hils_chunk_logz_bwd_dk_ws(q, k, log_z, d_log_z, dk, B, L, HQ, H, D, S, window, sm_scale, nullptr, 0, stream);
}

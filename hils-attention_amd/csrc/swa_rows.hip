// Sliding-window attention for few query rows (a decode step, a short slice on a cache).
//
// The tile kernel (swa.hip) gives a workgroup 128 or 256 score rows and walks the window tile by tile:
// with a single query per sequence most of those rows are padding and the walk over a window of 512 is a
// serial chain of phases (13 us for one sequence of heads of 64, 18 us for 64 (sequence, KV head) pairs of heads of 128).
// Here a workgroup owns 16 score rows (16/G queries times the G heads of a KV head: the 16 columns of the
// matrix instructions) and its eight wavefronts share the WINDOW: units of 32 tokens go round-robin, the
// next unit's K and V loads are in flight while one is worked on, and the eight partial results
// (running maximum, sum, output) meet once in LDS.  The chain is two or three units long.
//
// S^T = K q^T takes the K rows straight from memory as A operands (a lane reads 16 bytes of its token's
// row); V is staged row-major in the wavefront's own LDS area and read by the transposing LDS load as the
// A operand of O^T += V^T P, in the token order in which the S^T accumulators hold P.  Rows are matrix
// columns in both products, so maxima, sums and the rescaling of the accumulators stay in their lanes.
//
// With few rows a compute unit's share of the memory system bounds it: all of a row's keys and values are asked for at
// once, 128 KB (heads of 64, window 512) arrive in about 3.5 us.  What a unit of 32 tokens computes comes on top, three
// of them in series, so it must not branch: 0.4 us a unit, where masks tested score by score took 1.0 (the kernel in a
// row of launches, 1 / 64 / 256 workgroups: heads of 64 6.2 / 6.8 / 7.5 -> 5.6 / 5.9 / 6.4 us, of 128 10.2 / 11.4 /
// 14.3 -> 9.1 / 10.1 / 13.3).  Loads through buffer descriptors with the next unit asked for between its scores and its
// softmax were slower (8.0 against 7.4 us at 64 workgroups): the loads past the end take their turn in the queue too.
#include "stream_tiles.h"
#include "swa_dims.h"

#define SR_WAVES 8
#define SR_UNIT 32  // tokens a wavefront works on at a time

template <int D, int DVF, int VS>
__global__ void __launch_bounds__(SR_WAVES * 64) __attribute__((amdgpu_waves_per_eu(2)))
swa_fwd_rows(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
             bf16_t* __restrict__ o, float* __restrict__ lse, SwaDims dm, int g_bits) {
  constexpr int DV = DVF / VS;  // the value features of this workgroup, of DVF
  constexpr int KS = D / 32, MT = DV / 16;
  constexpr int VL = DV / 8, TPI = 64 / VL, VI = SR_UNIT / TPI;  // lanes per V row, rows per load, loads per unit
  constexpr int VP = 2 * DV + 16;                                // bytes of a staged V row
  constexpr int OP = DV + 4;                                     // floats of a parked output row
  constexpr int AREA = SR_UNIT * VP > 16 * OP * 4 ? SR_UNIT * VP : 16 * OP * 4;
  typedef unsigned sr_u4 __attribute__((ext_vector_type(4)));
  typedef short sr_s4 __attribute__((ext_vector_type(4)));
  typedef short sr_s8 __attribute__((ext_vector_type(8)));
  __shared__ __align__(16) unsigned char area_s[SR_WAVES * AREA];
  __shared__ float m_s[SR_WAVES][16], l_s[SR_WAVES][16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, j = lane >> 4;
  const int G = 1 << g_bits, QB = 16 >> g_bits;  // (no division: one is tens of instructions before the first load)
  const int tq0 = blockIdx.x * QB;
  const int hk = VS > 1 ? blockIdx.y % dm.H : blockIdx.y, part = VS > 1 ? blockIdx.y / dm.H : 0;
  const long b = blockIdx.z;
  const int q_off = dm.kv_start + dm.Lk - dm.Lq;  // absolute position of query 0

  // this lane's row and the key positions it sees, [vlo, vlo + vspan] (a start no position reaches: none)
  const int t = tq0 + (col >> g_bits), g = col & (G - 1);
  const bool live = t < dm.Lq;
  const int tc = live ? t : dm.Lq - 1;
  bf16x8_t qb[KS];
  {
    const bf16_t* qp = q + ((b * dm.Lq + tc) * (long)dm.HQ + hk * G + g) * D + j * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qb[ks] = *(const bf16x8_t*)(qp + ks * 32);
  }
  auto win_start = [&](int tt) -> int {  // first absolute position query tt sees
    const int left = q_off + tt - dm.window + 1;
    return !dm.expand ? left : dm.chunk_pow2 ? left & -dm.chunk : floordiv(left, dm.chunk) * dm.chunk;
  };
  int vlo;
  unsigned vspan;
  {
    const int c0 = win_start(tc), hi = q_off + tc;
    const bool some = live && hi >= c0;
    vlo = some ? c0 : 0x7fffffff;
    vspan = some ? (unsigned)(hi - c0) : 0u;
  }
  // key range of the workgroup (raw indices into k / v), in units
  int lo = win_start(tq0) - dm.kv_start;
  lo = lo < 0 ? 0 : lo;
  int tq1 = tq0 + QB - 1;
  tq1 = tq1 < dm.Lq ? tq1 : dm.Lq - 1;
  int hi = q_off + tq1 - dm.kv_start + 1;
  hi = hi < dm.Lk ? hi : dm.Lk;
  const int n_units = hi > lo ? (hi - lo + SR_UNIT - 1) / SR_UNIT : 0;
  const float c2 = dm.sm_scale * HILS_LOG2E;

  const bf16_t* kb = k + b * dm.k_batch + (long)hk * D + j * 8;
  const bf16_t* vb = v + b * dm.v_batch + (long)hk * DVF + part * DV + (lane % VL) * 8;
  auto issue = [&](sr_u4 (&kd)[2][KS], sr_u4 (&vd)[VI], int u) __attribute__((always_inline)) {
    const int t0 = lo + u * SR_UNIT;  // tokens past the end read the last row: their scores are masked
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      int tok = t0 + tt * 16 + col;
      tok = tok < dm.Lk ? tok : dm.Lk - 1;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kd[tt][ks] = *(const sr_u4*)(kb + (long)tok * dm.H * D + ks * 32);
    }
#pragma unroll
    for (int i = 0; i < VI; ++i) {
      int tok = t0 + i * TPI + lane / VL;
      tok = tok < dm.Lk ? tok : dm.Lk - 1;
      vd[i] = *(const sr_u4*)(vb + (long)tok * dm.H * DVF);
    }
  };

  unsigned char* area = area_s + wave * AREA;
  unsigned char* const w_addr = area + (lane / VL) * VP + (lane % VL) * 16;
  const unsigned char* const t_addr = area + (4 * j + (col >> 2)) * VP + (col & 3) * 8;
  f32x4_t O[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) O[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = HILS_NEG_INF, l_run = 0.f;  // of this lane's row over the units seen (l_run: this lane's tokens)

  auto unit = [&](const sr_u4 (&kd)[2][KS], const sr_u4 (&vd)[VI], int u) __attribute__((always_inline)) {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < VI; ++i) *(sr_u4*)(w_addr + i * TPI * VP) = vd[i];
    __builtin_amdgcn_wave_barrier();
    f32x4_t S[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      S[tt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        S[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kd[tt][ks]), qb[ks], S[tt], 0, 0, 0);
    }
    const int tok_raw0 = lo + u * SR_UNIT + 4 * j;
    const unsigned base = (unsigned)(dm.kv_start + tok_raw0 - vlo);
    // (positions end at the last key's, so the end of the keys needs no test of its own; the options are decided once
    // a unit: tested per element they made some twenty branches of it, 1.0 us against 0.5)
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[tt][i] = base + (unsigned)(tt * 16 + i) <= vspan ? S[tt][i] : HILS_NEG_INF;
    if (dm.mask_lmk) {
      const int ta = dm.kv_start + tok_raw0 + 1;
      if (dm.chunk_pow2) {
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
          for (int i = 0; i < 4; ++i) S[tt][i] = ((ta + tt * 16 + i) & (dm.chunk - 1)) ? S[tt][i] : HILS_NEG_INF;
      } else {
#pragma unroll 1
        for (int e = 0; e < 8; ++e) {  // (rolled: the divisions would be most of the kernel's code)
          const int i = e & 3;
          const bool lm = (ta + (e >> 2) * 16 + i) % dm.chunk == 0;
#pragma unroll
          for (int x = 0; x < 8; ++x) S[x >> 2][x & 3] = lm && x == e ? HILS_NEG_INF : S[x >> 2][x & 3];
        }
      }
    }
    float mx = HILS_NEG_INF;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, S[tt][i]);
    mx = rows_max(mx);
    const float m_new = fmaxf(m_run, mx);
    const bool any = m_new > HILS_NEG_INF;
    const float mc = any ? m_new * c2 : 0.f;
    const float corr = any ? __builtin_amdgcn_exp2f(fmaf(m_run, c2, -mc)) : 1.f;  // exp2(-inf) = 0: nothing yet
    m_run = m_new;
    float sum = 0.f;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = __builtin_amdgcn_exp2f(fmaf(S[tt][i], c2, -mc));
        S[tt][i] = e;
        sum += e;
      }
    l_run = l_run * corr + sum;
    sr_u4 pk;
    pk.x = pack_bf2(S[0][0], S[0][1]);
    pk.y = pack_bf2(S[0][2], S[0][3]);
    pk.z = pack_bf2(S[1][0], S[1][1]);
    pk.w = pack_bf2(S[1][2], S[1][3]);
    const bf16x8_t pb = __builtin_bit_cast(bf16x8_t, pk);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const sr_s4 a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) sr_s4*)(t_addr + mt * 32));
      const sr_s4 a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) sr_s4*)(t_addr + mt * 32 + 16 * VP));
      const sr_s8 a = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
      for (int i = 0; i < 4; ++i) O[mt][i] *= corr;
      O[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), pb, O[mt], 0, 0, 0);
    }
  };
  {
    // two units' loads in flight; an index past the end reads the last unit again and is not worked on
    sr_u4 ka[2][KS], va[VI], kc[2][KS], vc[VI];
    const int last = n_units - 1;
    if (wave < n_units) {
      issue(ka, va, wave);
      for (int u = wave; u < n_units; u += 2 * SR_WAVES) {
        const int u1 = u + SR_WAVES, u2 = u + 2 * SR_WAVES;
        issue(kc, vc, u1 < last ? u1 : last);
        unit(ka, va, u);
        if (u1 >= n_units) break;
        issue(ka, va, u2 < last ? u2 : last);
        unit(kc, vc, u1);
      }
    }
  }
  // park the partial results: accumulator register i of tile mt in lane (row = col, j) is feature mt*16 + 4j + i
  __builtin_amdgcn_wave_barrier();
  float* o_s = (float*)area;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) *(f32x4_t*)&o_s[col * OP + mt * 16 + 4 * j] = O[mt];
  const float l_row = rows_sum(l_run);
  if (j == 0) {
    m_s[wave][col] = m_run;
    l_s[wave][col] = l_row;
  }
  __syncthreads();
  // 16 rows x DV/4 pieces of four features over the workgroup
  for (int p = tid; p < 16 * (DV / 4); p += SR_WAVES * 64) {
    const int row = p / (DV / 4), d4 = p % (DV / 4);
    const int tr = tq0 + (row >> g_bits);
    if (tr >= dm.Lq) continue;
    float M = HILS_NEG_INF;
#pragma unroll
    for (int w = 0; w < SR_WAVES; ++w) M = fmaxf(M, m_s[w][row]);
    float L = 0.f;
    f32x4_t x = {0.f, 0.f, 0.f, 0.f};
    // (no maximum: nothing was seen, and the sums are zero, or scores that are not numbers, which the sums keep)
#pragma unroll
    for (int w = 0; w < SR_WAVES; ++w) {
      const float f = M > HILS_NEG_INF ? __builtin_amdgcn_exp2f((m_s[w][row] - M) * c2) : 1.f;
      const f32x4_t ow = *(const f32x4_t*)((const float*)(area_s + w * AREA) + row * OP + d4 * 4);
      L = fmaf(f, l_s[w][row], L);
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = fmaf(f, ow[i], x[i]);
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    const long rix = (b * dm.Lq + tr) * (long)dm.HQ + hk * G + (row & (G - 1));
    uint2 pk;
    pk.x = pack_bf2(x[0] * inv, x[1] * inv);
    pk.y = pack_bf2(x[2] * inv, x[3] * inv);
    *(uint2*)(o + rix * DVF + part * DV + d4 * 4) = pk;
    if (d4 == 0 && part == 0) lse[rix] = L > 0.f ? (M * c2 + __builtin_amdgcn_logf(L)) * HILS_LN2 : HILS_NEG_INF;
  }
}

// The tile kernel gives a workgroup 128 or 256 score rows of a KV head, the row kernel 16.  With one or two row blocks
// a (sequence, KV head) the tile kernel's workgroups are mostly padding and walk the window in series; with more,
// every row block reads the window again.  Row / tile kernel in us, 256, 512, 1024, 2048 workgroups of the row kernel:
//   one block:   heads of 64, window 512  6.8/14  13/38  25/73  67/149;  window 64  5.6/5.5  5.7/5.8  7.3/9.3  13/15
//                heads of 128, 512  13/21  25/52  47/102  112/224;  256  9/12  17/30  31/57  71/125;
//                128  5.6/7.7  11/10  20/22  38/38;  64  5.8/5.8  7.6/7.1  15/13  28/25
//                keys of 64 and values of 128, 512  24/51 (640 workgroups), 256  27/52 (1280); the reverse 27/51 and 30/51
//   two blocks:  heads of 64, 512  7.8/15  15/17  26/41  49/79;  256  5.4/11  9/11  17/25  31/49;  128  5.5/8.5  7/9  13/10  23/21
//   eight:       heads of 64 (16 queries of eight heads), 512  -  15/15  27/16  48/18;  64  -  5.6/6.7  10/7  18/7
//   four:        heads of 128 (16 queries of four heads), 512  15/21  27/23  52/25;  64  5.6/8.2  11/8  21/9
// The line is not the times' alone.  Both round probabilities to bf16 and sum in fp32, but the row kernel takes them about
// each wavefront's own maximum, whose probability is exactly 1, the tile kernel about a reference point that lags behind the
// maximum: from 64 bits, relative, window 512, row / tile kernel 2.06e-3 / 2.28e-3 (32/8 heads of 128, 160 to 256
// queries; 16/2 of 64, 900 queries: 2.05 / 2.27; about the maximum itself the tile kernel has 2.16), window 64 2.02 / 2.08,
// 1.66 of each the output's own rounding.  So calls of up to 512 workgroups, and up to 1024 with narrow heads and a
// long window, stay with the row kernel also where the tile kernel would be ahead (20 / 18 us and 19 / 13 us of the
// two above).
bool hils_swa_rows_better(int B, int D, int Dv, const SwaDims& dm) {
  if (B > 65535 || dm.H > 65535) return false;  // (dimensions of the row kernel's grid)
  const int QB = 16 / (dm.HQ / dm.H);
  const long n_rb = (dm.Lq + QB - 1) / QB, wgs = n_rb * dm.H * B;
  const bool narrow = D <= 64 && Dv <= 64, wide_window = dm.window >= 256;
  if (wgs <= (narrow && wide_window ? 1024 : 512)) return true;
  return wide_window ? n_rb <= (narrow ? 2 : 1) : narrow && n_rb == 1;
}

int hils_swa_fwd_rows(int B, hipStream_t st, const void* q, const void* k, const void* v, void* o, float* lse, int D,
                      int Dv, const SwaDims& dm) {
  const int G = dm.HQ / dm.H;
  const int n_rb = (dm.Lq + 16 / G - 1) / (16 / G), g_bits = __builtin_ctz(G);
  // While both fit the chip at once, two workgroups a row block, each with all keys and half of the value features: a
  // compute unit's share of the memory system is the bound, and nothing has to be added up (one / two, window 512, us:
  // heads of 64 5.5/5.3 with one row block, 6.0/5.8 with 128, 6.0/9.2 with 192; of 128 9.2/8.6, 10.0/9.3, 10.6/16.6;
  // window 64: 3.6/3.5 and 4.5/4.2 with 128.  Four quarters: 8.8 against 9.2 on 64 blocks of heads of 128, else no faster).
  const bool halves = 2l * n_rb * dm.H * B <= hils_device_cus();
  const dim3 grid(n_rb, dm.H * (halves ? 2 : 1), B), wg(SR_WAVES * 64);
#define SR_CALL(D_, V_, S_)                                                                                 \
  hipLaunchKernelGGL((swa_fwd_rows<D_, V_, S_>), grid, wg, 0, st, (const bf16_t*)q, (const bf16_t*)k,        \
                     (const bf16_t*)v, (bf16_t*)o, lse, dm, g_bits)
#define SR_CALL_S(D_, V_) do { if (halves) SR_CALL(D_, V_, 2); else SR_CALL(D_, V_, 1); } while (0)
  if (D == 64 && Dv == 64) SR_CALL_S(64, 64);
  else if (D == 128 && Dv == 128) SR_CALL_S(128, 128);
  else if (D == 64) SR_CALL_S(64, 128);
  else SR_CALL_S(128, 64);
#undef SR_CALL_S
#undef SR_CALL
  return HILS_OK;
}

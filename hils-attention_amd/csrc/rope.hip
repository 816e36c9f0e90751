// Rotary position embedding in the "rotate half" convention: the two halves of a head vector are
// the real and imaginary parts, out1 = x1*c - x2*s, out2 = x2*c' + x1*s'.  fp32 arithmetic on bf16
// inputs, one rounding to bf16 at the end.  Pure HBM streaming: one thread per 16-byte piece of
// the low half, which also loads the matching piece of the high half.
#include "common.h"
#include "../../include/hils_amd.h"

// cos/sin rows hold D values per position; lo_only: both halves use the first D/2 of them
template <bool TAB_F32>
__global__ void __launch_bounds__(256)
rope_kernel(const bf16_t* __restrict__ x, const void* __restrict__ cos_t, const void* __restrict__ sin_t,
            bf16_t* __restrict__ out, long total, int L, int H, int D, long tab_batch_stride, int lo_only,
            float sin_sign) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;  // piece of 8 elements of the low half
  if (i >= total) return;
  const int pph = D / 16;  // pieces per half
  const int pc = (int)(i % pph);
  const long row = i / pph;  // (b*L + l)*H + h
  const long bl = row / H;
  const long l = bl % L, b = bl / L;
  const long xo = row * D + pc * 8;
  const uint4 lo4 = *(const uint4*)(x + xo);
  const uint4 hi4 = *(const uint4*)(x + xo + D / 2);
  float x1[8], x2[8], c1[8], s1[8], c2[8], s2[8];
  unpack8(lo4, x1);
  unpack8(hi4, x2);
  const long to = b * tab_batch_stride + l * D + pc * 8;
  const long th = lo_only ? to : to + D / 2;
  if (TAB_F32) {
    const float* ct = (const float*)cos_t;
    const float* st = (const float*)sin_t;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      c1[e] = ct[to + e]; s1[e] = st[to + e];
      c2[e] = ct[th + e]; s2[e] = st[th + e];
    }
  } else {
    unpack8(*(const uint4*)((const bf16_t*)cos_t + to), c1);
    unpack8(*(const uint4*)((const bf16_t*)sin_t + to), s1);
    unpack8(*(const uint4*)((const bf16_t*)cos_t + th), c2);
    unpack8(*(const uint4*)((const bf16_t*)sin_t + th), s2);
  }
  float o1[8], o2[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    o1[e] = x1[e] * c1[e] - x2[e] * (s1[e] * sin_sign);
    o2[e] = x2[e] * c2[e] + x1[e] * (s2[e] * sin_sign);
  }
  uint4 w1, w2;
  w1.x = pack_bf2(o1[0], o1[1]); w1.y = pack_bf2(o1[2], o1[3]); w1.z = pack_bf2(o1[4], o1[5]); w1.w = pack_bf2(o1[6], o1[7]);
  w2.x = pack_bf2(o2[0], o2[1]); w2.y = pack_bf2(o2[2], o2[3]); w2.z = pack_bf2(o2[4], o2[5]); w2.w = pack_bf2(o2[6], o2[7]);
  *(uint4*)(out + xo) = w1;
  *(uint4*)(out + xo + D / 2) = w2;
}

extern "C" int hils_rope(const void* x, const void* cos_t, const void* sin_t, void* out, int B, int L,
                         int H, int D, int table_per_batch, int table_f32, int lo_only,
                         float sin_sign, void* stream) {
  HILS_REQUIRE(x && cos_t && sin_t && out, "hils_rope: null pointer");
  HILS_REQUIRE(B > 0 && L > 0 && H > 0 && D > 0, "hils_rope: sizes must be positive");
  HILS_REQUIRE(D % 16 == 0, "hils_rope: D (%d) must be a multiple of 16", D);
  const long total = (long)B * L * H * (D / 16);
  const long nblk = (total + 255) / 256;
  HILS_REQUIRE(nblk <= 2147483647L, "hils_rope: grid too large");
  const long tbs = table_per_batch ? (long)L * D : 0;
  if (table_f32)
    hipLaunchKernelGGL(rope_kernel<true>, dim3((unsigned)nblk), dim3(256), 0, (hipStream_t)stream,
                       (const bf16_t*)x, cos_t, sin_t, (bf16_t*)out, total, L, H, D, tbs, lo_only, sin_sign);
  else
    hipLaunchKernelGGL(rope_kernel<false>, dim3((unsigned)nblk), dim3(256), 0, (hipStream_t)stream,
                       (const bf16_t*)x, cos_t, sin_t, (bf16_t*)out, total, L, H, D, tbs, lo_only, sin_sign);
  HILS_CHECK_LAUNCH("hils_rope");
  return HILS_OK;
}

// ---------------------------------------------------------------------------
// Key (or query) preparation in one pass over the projected tensor: per-head RMS norm, rotary
// embedding, and the mean over each chunk (the chunk keys) - the layer's sequence
//   k = k_norm(k);  k = k*cos + rotate_half(k)*sin;  lmk = k.view(B,N,S,H,D).mean(2)
// which otherwise reads and writes the (B,L,H,D) tensor once per step.  Roundings follow that
// sequence on bf16 tensors: the normalised value is rounded to bf16 before the weight multiplies it,
// each product and the sum of the rotation are rounded to bf16, and the mean is taken over the
// rounded outputs (fp32 sum, one rounding).
//
// Bound by HBM: the tensor in and out (forward), x, the gradient and dx (backward).  A workgroup owns
// the S tokens of a (batch, chunk) for HG neighbouring heads, HG the largest power of two that divides H
// and still leaves a wavefront's 64 lanes (D/8 lanes per (token, head) row) whole tokens: every
// load and store of a wavefront is one contiguous 1 KiB run, the tables are read once per token and not
// once per head, and a lane keeps one head and one piece of its vector, so the chunk mean (and the norm
// weight's gradient) accumulate in registers and meet once per workgroup.  The wavefronts share out the
// tokens, four steps of loads in flight each.  The rows' reductions and the exchange between the halves of
// a head vector stay inside 8, 16 or 32 lanes and run as DPP moves (no LDS traffic).
// ---------------------------------------------------------------------------
__device__ __forceinline__ float np_round_bf16(float x) { return bf2f(f2bf(x)); }
// a vector rounded to bf16 in pairs (three instructions for two values)
__device__ __forceinline__ void np_round8(float (&f)[8]) {
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const uint32_t u = pack_bf2(f[e], f[e + 1]);
    f[e] = __uint_as_float(u << 16);
    f[e + 1] = __uint_as_float(u & 0xffff0000u);
  }
}

struct NpDims {
  int B, L, H, S, hg, hg_log2, nchunk_all, nchunk_full;
  long tab_batch_stride;
  float eps;
};

constexpr int kNpBatch = 4;  // steps whose loads are in flight together

// The mirrored lane of the eight (one move that folds into its use; the lane with bit 2 flipped takes two and copies).
__device__ __forceinline__ float np_mirror8(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xf, 0xf, true));  // row_half_mirror
}
// Piece of the head vector that a row's lane holds, and the value of the lane with the other half's: with eight lanes
// the upper four hold their pieces in reverse, so that the mirrored lane has the partner.
template <int LPR>
__device__ __forceinline__ int np_piece(int lane) {
  const int p = lane % LPR;
  return LPR == 8 && p >= 4 ? 11 - p : p;
}
template <int LPR>
__device__ __forceinline__ float np_other(float v) {
  if (LPR == 8) return np_mirror8(v);
  return lane_xor<LPR / 2>(v);
}

// sum over the LPR lanes of a row
template <int LPR>
__device__ __forceinline__ float np_row_sum(float v) {
  v += lane_xor<1>(v);
  v += lane_xor<2>(v);
  v += np_mirror8(v);  // (four lanes alike by now)
  if (LPR > 8) v += lane_xor<8>(v);
  if (LPR > 16) v += lane_xor<16>(v);
  return v;
}

template <int LPR>  // lanes per token row = D / 8
__global__ void __launch_bounds__(1024)
norm_rope_pool_fwd_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                          const bf16_t* __restrict__ cos_t, const bf16_t* __restrict__ sin_t,
                          bf16_t* __restrict__ out, bf16_t* __restrict__ lmk, NpDims dm) {
  constexpr int D = LPR * 8, RPI = 64 / LPR;  // (token, head) rows per wavefront and step
  extern __shared__ float np_red[];           // [wavefront][HG * LPR][8], chunk sums
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int hgroups = dm.H >> dm.hg_log2, tps = RPI >> dm.hg_log2;  // tokens per step
  const int bn = blockIdx.x / hgroups, hg0 = (blockIdx.x % hgroups) << dm.hg_log2;
  const int b = bn / dm.nchunk_all, n = bn % dm.nchunk_all;
  const int p = np_piece<LPR>(lane), r = lane / LPR;
  const int h = hg0 + (r & (dm.hg - 1)), tt = r >> dm.hg_log2;
  const long row0 = (long)b * dm.L;
  float wv[8];
  if (w) unpack8(*(const uint4*)(w + p * 8), wv);
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  const int steps = (dm.S + tps - 1) / tps;
  for (int i0 = wave; i0 < steps; i0 += kNpBatch * nw) {
    uint4 xv[kNpBatch], cv[kNpBatch], sv[kNpBatch];
#pragma unroll
    for (int u = 0; u < kNpBatch; ++u) {
      const int tok = (i0 + u * nw) * tps + tt;
      const int t = n * dm.S + tok;
      const bool ok = tok < dm.S && t < dm.L;
      const long tc = ok ? t : 0;
      xv[u] = *(const uint4*)(x + ((row0 + tc) * dm.H + h) * (long)D + p * 8);
      if (cos_t) {
        const long to = b * dm.tab_batch_stride + tc * D + p * 8;
        cv[u] = *(const uint4*)(cos_t + to);
        sv[u] = *(const uint4*)(sin_t + to);
      }
    }
#pragma unroll
    for (int u = 0; u < kNpBatch; ++u) {
      const int tok = (i0 + u * nw) * tps + tt;
      const int t = n * dm.S + tok;
      const bool ok = tok < dm.S && t < dm.L;
      float f[8];
      unpack8(xv[u], f);
      if (w) {
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(f[e], f[e], ss);
        const float rr = rsqrtf(np_row_sum<LPR>(ss) * (1.f / D) + dm.eps);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] *= rr;
        np_round8(f);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] *= wv[e];
        if (cos_t) np_round8(f);  // (else the packed output is that rounding)
      }
      if (cos_t) {
        float c[8], s[8];
        unpack8(cv[u], c);
        const uint32_t flip = p < LPR / 2 ? 0x80008000u : 0u;  // rotate_half: (-x_hi, x_lo)
        unpack8(make_uint4(sv[u].x ^ flip, sv[u].y ^ flip, sv[u].z ^ flip, sv[u].w ^ flip), s);
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] *= np_other<LPR>(f[e]);
#pragma unroll
        for (int e = 0; e < 8; ++e) c[e] *= f[e];
        np_round8(c);
        np_round8(s);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = c[e] + s[e];
      }
      if (ok) {
        uint4 o;
        o.x = pack_bf2(f[0], f[1]); o.y = pack_bf2(f[2], f[3]); o.z = pack_bf2(f[4], f[5]); o.w = pack_bf2(f[6], f[7]);
        *(uint4*)(out + ((row0 + t) * dm.H + h) * (long)D + p * 8) = o;
        if (lmk) {  // of the rounded outputs
          unpack8(o, f);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[e] += f[e];
        }
      }
    }
  }
  if (lmk && n < dm.nchunk_full) {
    for (int o2 = dm.hg * LPR; o2 < 64; o2 <<= 1)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], o2, 64);
    const int cols = dm.hg * LPR;
    if (lane < cols) {
#pragma unroll
      for (int e = 0; e < 8; ++e) np_red[((wave * cols) + lane) * 8 + e] = acc[e];
    }
    lds_barrier();
    if ((int)threadIdx.x < cols) {
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = 0.f;
      for (int k = 0; k < nw; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += np_red[((k * cols) + lane) * 8 + e];
      const float inv = 1.f / (float)dm.S;
      uint4 o;
      o.x = pack_bf2(acc[0] * inv, acc[1] * inv); o.y = pack_bf2(acc[2] * inv, acc[3] * inv);
      o.z = pack_bf2(acc[4] * inv, acc[5] * inv); o.w = pack_bf2(acc[6] * inv, acc[7] * inv);
      *(uint4*)(lmk + (((long)b * dm.nchunk_full + n) * dm.H + h) * (long)D + p * 8) = o;
    }
  }
}

// Backward of the pass above.  g = d_out + d_lmk / S (either may be absent); through the rotation:
// gz = g*cos + rotate_half^T(g*sin); through the weight: d_w += gz * y, gy = gz * w; through the
// norm (y = x r, r = (mean x^2 + eps)^-1/2): dx = r (gy - y mean(gy y)).  The D sums of d_w leave a
// workgroup as one row of `part` (norm_rope_pool_dw_kernel adds the rows), or, without that scratch, as one
// atomic per feature.  With an atomic per wavefront and feature, every wavefront of the chip on the same D
// words, the adds took thirty times as long as the pass (B8 L8192 H16 D64: 3.18 ms).
template <int LPR>
__global__ void __launch_bounds__(1024)
norm_rope_pool_bwd_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                          const bf16_t* __restrict__ cos_t, const bf16_t* __restrict__ sin_t,
                          const bf16_t* __restrict__ g_out, const bf16_t* __restrict__ g_lmk,
                          bf16_t* __restrict__ dx, float* __restrict__ dw, float* __restrict__ part, NpDims dm) {
  constexpr int D = LPR * 8, RPI = 64 / LPR;
  extern __shared__ float np_red[];  // [wavefront][D]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int hgroups = dm.H >> dm.hg_log2, tps = RPI >> dm.hg_log2;
  const int bn = blockIdx.x / hgroups, hg0 = (blockIdx.x % hgroups) << dm.hg_log2;
  const int b = bn / dm.nchunk_all, n = bn % dm.nchunk_all;
  const int p = np_piece<LPR>(lane), r = lane / LPR;
  const int h = hg0 + (r & (dm.hg - 1)), tt = r >> dm.hg_log2;
  const long row0 = (long)b * dm.L;
  float wv[8], gl[8], wacc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) { wv[e] = 1.f; gl[e] = 0.f; wacc[e] = 0.f; }
  if (w) unpack8(*(const uint4*)(w + p * 8), wv);
  if (g_lmk && n < dm.nchunk_full) {
    unpack8(*(const uint4*)(g_lmk + (((long)b * dm.nchunk_full + n) * dm.H + h) * (long)D + p * 8), gl);
    const float inv = 1.f / (float)dm.S;
#pragma unroll
    for (int e = 0; e < 8; ++e) gl[e] *= inv;
  }
  const int steps = (dm.S + tps - 1) / tps;
  for (int i0 = wave; i0 < steps; i0 += kNpBatch * nw) {
    uint4 xv[kNpBatch], gv[kNpBatch], cv[kNpBatch], sv[kNpBatch];
#pragma unroll
    for (int u = 0; u < kNpBatch; ++u) {
      const int tok = (i0 + u * nw) * tps + tt;
      const int t = n * dm.S + tok;
      const long tc = tok < dm.S && t < dm.L ? t : 0;
      const long xo = ((row0 + tc) * dm.H + h) * (long)D + p * 8;
      xv[u] = *(const uint4*)(x + xo);
      gv[u] = g_out ? *(const uint4*)(g_out + xo) : make_uint4(0u, 0u, 0u, 0u);
      if (cos_t) {
        const long to = b * dm.tab_batch_stride + tc * D + p * 8;
        cv[u] = *(const uint4*)(cos_t + to);
        sv[u] = *(const uint4*)(sin_t + to);
      }
    }
#pragma unroll
    for (int u = 0; u < kNpBatch; ++u) {
      const int tok = (i0 + u * nw) * tps + tt;
      const int t = n * dm.S + tok;
      const bool ok = tok < dm.S && t < dm.L;
      float f[8], g[8];
      unpack8(xv[u], f);
      unpack8(gv[u], g);
#pragma unroll
      for (int e = 0; e < 8; ++e) g[e] = ok ? g[e] + gl[e] : 0.f;
      if (cos_t) {
        float c[8], s[8];
        unpack8(cv[u], c);
        unpack8(sv[u], s);
        const float sign = p < LPR / 2 ? 1.f : -1.f;  // transpose of rotate_half: (u_hi, -u_lo)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float other = np_other<LPR>(g[e] * s[e]);
          g[e] = fmaf(g[e], c[e], sign * other);
        }
      }
      if (w) {
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(f[e], f[e], ss);
        const float rr = rsqrtf(np_row_sum<LPR>(ss) * (1.f / D) + dm.eps);
        float dot = 0.f, y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          y[e] = f[e] * rr;
          wacc[e] = fmaf(g[e], np_round_bf16(y[e]), wacc[e]);
          g[e] *= wv[e];
          dot = fmaf(g[e], y[e], dot);
        }
        dot = np_row_sum<LPR>(dot) * (1.f / D);
#pragma unroll
        for (int e = 0; e < 8; ++e) g[e] = rr * (g[e] - y[e] * dot);
      }
      if (ok) {
        uint4 o;
        o.x = pack_bf2(g[0], g[1]); o.y = pack_bf2(g[2], g[3]); o.z = pack_bf2(g[4], g[5]); o.w = pack_bf2(g[6], g[7]);
        *(uint4*)(dx + ((row0 + t) * dm.H + h) * (long)D + p * 8) = o;
      }
    }
  }
  if (w && (dw || part)) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int o2 = LPR; o2 < 64; o2 <<= 1) wacc[e] += __shfl_xor(wacc[e], o2, 64);
    if (lane < LPR) {
#pragma unroll
      for (int e = 0; e < 8; ++e) np_red[wave * D + p * 8 + e] = wacc[e];
    }
    lds_barrier();
    for (int c = threadIdx.x; c < D; c += blockDim.x) {
      float v = 0.f;
      for (int k = 0; k < nw; ++k) v += np_red[k * D + c];
      if (part) part[(long)blockIdx.x * D + c] = v;
      else if (v != 0.f) unsafeAtomicAdd(dw + c, v);
    }
  }
}

// Adds the rows of `part`: a workgroup takes 16 features (64 bytes of a row) and 256 rows at a time, in a fixed
// order.  256 KiB to 4 MiB that the pass above has just left in the L2: about 5 us.
__global__ void __launch_bounds__(1024)
norm_rope_pool_dw_kernel(const float* __restrict__ part, void* __restrict__ dw, int dw_bf16, int rows, int D) {
  __shared__ float red[256][17];
  const int c = (threadIdx.x & 3) * 4, rg = threadIdx.x >> 2;
  const float* src = part + blockIdx.x * 16 + c;
  f32x4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = rg; k < rows; k += 256) a += *(const f32x4_t*)(src + (long)k * D);
#pragma unroll
  for (int e = 0; e < 4; ++e) red[rg][c + e] = a[e];
  __syncthreads();
  const int f = threadIdx.x & 15, q = threadIdx.x >> 4;  // 64 threads per feature, four rows each
  float v = red[q][f] + red[q + 64][f] + red[q + 128][f] + red[q + 192][f];
  __syncthreads();
  red[q][f] = v;
  __syncthreads();
  if (threadIdx.x < 16) {
    v = 0.f;
    for (int k = 0; k < 64; ++k) v += red[k][f];
    if (dw_bf16) ((bf16_t*)dw)[blockIdx.x * 16 + f] = f2bf(v);
    else ((float*)dw)[blockIdx.x * 16 + f] = v;
  }
}

static int np_check(const char* who, const void* x, const void* cos_t, const void* sin_t, int B, int L, int H,
                    int D, int S) {
  HILS_REQUIRE(x, "%s: null pointer", who);
  HILS_REQUIRE((cos_t == nullptr) == (sin_t == nullptr), "%s: cos and sin come together", who);
  HILS_REQUIRE(B > 0 && L > 0 && H > 0 && S > 0, "%s: sizes must be positive", who);
  HILS_REQUIRE(D == 64 || D == 128 || D == 256, "%s: head dim %d not supported (64, 128 or 256)", who, D);
  HILS_REQUIRE((long)B * ((L + S - 1) / S) * H <= 2147483647L && (long)L + S <= 2147483647L, "%s: grid too large", who);
  return HILS_OK;
}

// heads per workgroup: the largest power of two that divides H and leaves a wavefront whole tokens
static int np_heads(int H, int D) {
  int hg = 1;
  while (hg * 2 <= 512 / D && H % (hg * 2) == 0) hg *= 2;
  return hg;
}

static long np_blocks(int B, int L, int H, int D, int S) { return (long)B * ((L + S - 1) / S) * (H / np_heads(H, D)); }

// Tokens of a workgroup that forms no chunk mean: 64, fewer while the grid leaves compute units idle (a step is 200 to
// 250 vector instructions of a wavefront: with a chunk per workgroup a short sequence kept 64 of 256 compute units busy,
// 16 wavefronts each; B2 L1024 16 and 2 heads of 64, forward 9.4 -> 6.3 us, backward 12.5 -> 8.0), down to one step per
// wavefront.
static int np_tokens(int B, int L, int H, int D, long least_blocks) {
  const int tps = 512 / D / np_heads(H, D);
  int tok = 64;
  while (tok >= 8 * tps && np_blocks(B, L, H, D, tok) < least_blocks) tok /= 2;
  return tok;
}

// Launch shape: 4 wavefronts per workgroup; with a chunk mean up to 16 while the grid has fewer than 16 wavefronts per
// compute unit and every wavefront still has a token (short sequences: the pass is a chain of a wavefront's loads).
static NpDims np_dims(int B, int L, int H, int D, int S, bool pool, int table_per_batch, float eps, int* threads) {
  NpDims dm{B, L, H, S, np_heads(H, D), 0, (L + S - 1) / S, L / S, table_per_batch ? (long)L * D : 0, eps};
  while ((1 << dm.hg_log2) < dm.hg) ++dm.hg_log2;
  const int tps = 512 / D / dm.hg, steps = (S + tps - 1) / tps;
  int nw = 4;
  while (pool && nw < 16 && nw * 2 <= steps && np_blocks(B, L, H, D, S) * nw < 16L * hils_device_cus()) nw *= 2;
  *threads = nw * 64;
  return dm;
}

extern "C" int hils_norm_rope_pool_fwd(const void* x, const void* norm_weight, const void* cos_t,
                                       const void* sin_t, void* out, void* lmk, int B, int L, int H, int D,
                                       int S, int table_per_batch, float eps, void* stream) {
  if (int rc = np_check("hils_norm_rope_pool_fwd", x, cos_t, sin_t, B, L, H, D, S)) return rc;
  HILS_REQUIRE(out, "hils_norm_rope_pool_fwd: null output");
  int threads;
  if (!lmk) S = np_tokens(B, L, H, D, 4L * hils_device_cus());
  const NpDims dm = np_dims(B, L, H, D, S, lmk != nullptr, table_per_batch, eps, &threads);
  const dim3 grid((unsigned)np_blocks(B, L, H, D, S));
  const size_t lds = lmk ? (size_t)(threads / 64) * dm.hg * D * sizeof(float) : 0;
#define NP_FWD(LPR_)                                                                                      \
  hipLaunchKernelGGL(norm_rope_pool_fwd_kernel<LPR_>, grid, dim3(threads), lds, (hipStream_t)stream,      \
                     (const bf16_t*)x, (const bf16_t*)norm_weight, (const bf16_t*)cos_t, (const bf16_t*)sin_t, \
                     (bf16_t*)out, (bf16_t*)lmk, dm)
  if (D == 64) NP_FWD(8); else if (D == 128) NP_FWD(16); else NP_FWD(32);
#undef NP_FWD
  HILS_CHECK_LAUNCH("hils_norm_rope_pool_fwd");
  return HILS_OK;
}

// One block per compute unit of the chip: every block is a row of d_weight's sum.  (Not of the device as it is partitioned:
// the workspace and the order of the sum go by the shape alone.)
static int np_bwd_tokens(int B, int L, int H, int D) { return np_tokens(B, L, H, D, 256); }

static int np_bwd(const char* who, const void* x, const void* norm_weight, const void* cos_t, const void* sin_t,
                  const void* d_out, const void* d_lmk, void* dx, float* d_weight, float* part, int B, int L, int H,
                  int D, int S, int table_per_batch, float eps, void* stream) {
  if (int rc = np_check(who, x, cos_t, sin_t, B, L, H, D, S)) return rc;
  HILS_REQUIRE(dx && (d_out || d_lmk), "%s: null pointer", who);
  int threads;
  const NpDims dm = np_dims(B, L, H, D, S, d_lmk != nullptr, table_per_batch, eps, &threads);
  const dim3 grid((unsigned)np_blocks(B, L, H, D, S));
  const size_t lds = norm_weight ? (size_t)(threads / 64) * D * sizeof(float) : 0;
#define NP_BWD(LPR_)                                                                                      \
  hipLaunchKernelGGL(norm_rope_pool_bwd_kernel<LPR_>, grid, dim3(threads), lds, (hipStream_t)stream,      \
                     (const bf16_t*)x, (const bf16_t*)norm_weight, (const bf16_t*)cos_t, (const bf16_t*)sin_t, \
                     (const bf16_t*)d_out, (const bf16_t*)d_lmk, (bf16_t*)dx, d_weight, part, dm)
  if (D == 64) NP_BWD(8); else if (D == 128) NP_BWD(16); else NP_BWD(32);
#undef NP_BWD
  HILS_CHECK_LAUNCH(who);
  return HILS_OK;
}

extern "C" int hils_norm_rope_pool_bwd(const void* x, const void* norm_weight, const void* cos_t,
                                       const void* sin_t, const void* d_out, const void* d_lmk, void* dx,
                                       float* d_weight, int B, int L, int H, int D, int S,
                                       int table_per_batch, float eps, void* stream) {
  HILS_REQUIRE(!norm_weight || d_weight, "hils_norm_rope_pool_bwd: the norm weight needs d_weight");
  if (!d_lmk && B > 0 && L > 0 && H > 0 && S > 0 && (D == 64 || D == 128 || D == 256)) S = np_bwd_tokens(B, L, H, D);
  return np_bwd("hils_norm_rope_pool_bwd", x, norm_weight, cos_t, sin_t, d_out, d_lmk, dx, d_weight, nullptr, B, L,
                H, D, S, table_per_batch, eps, stream);
}

extern "C" size_t hils_norm_rope_pool_bwd_workspace(int B, int L, int H, int D, int S) {
  if (B <= 0 || L <= 0 || H <= 0 || S <= 0 || (D != 64 && D != 128 && D != 256)) return 0;
  const long pooled = np_blocks(B, L, H, D, S), plain = np_blocks(B, L, H, D, np_bwd_tokens(B, L, H, D));
  return (size_t)(pooled > plain ? pooled : plain) * D * sizeof(float);
}

extern "C" int hils_norm_rope_pool_bwd_ws(const void* x, const void* norm_weight, const void* cos_t,
                                          const void* sin_t, const void* d_out, const void* d_lmk, void* dx,
                                          void* d_weight, int d_weight_bf16, void* workspace, size_t workspace_bytes,
                                          int B, int L, int H, int D, int S, int table_per_batch, float eps,
                                          void* stream) {
  const char* who = "hils_norm_rope_pool_bwd_ws";
  HILS_REQUIRE(norm_weight && d_weight && workspace, "%s: null pointer", who);
  HILS_REQUIRE(workspace_bytes >= hils_norm_rope_pool_bwd_workspace(B, L, H, D, S), "%s: workspace too small", who);
  if (!d_lmk && B > 0 && L > 0 && H > 0 && S > 0 && (D == 64 || D == 128 || D == 256)) S = np_bwd_tokens(B, L, H, D);
  if (int rc = np_bwd(who, x, norm_weight, cos_t, sin_t, d_out, d_lmk, dx, nullptr, (float*)workspace, B, L, H, D, S,
                      table_per_batch, eps, stream))
    return rc;
  hipLaunchKernelGGL(norm_rope_pool_dw_kernel, dim3(D / 16), dim3(1024), 0, (hipStream_t)stream,
                     (const float*)workspace, d_weight, d_weight_bf16, (int)np_blocks(B, L, H, D, S), D);
  HILS_CHECK_LAUNCH(who);
  return HILS_OK;
}

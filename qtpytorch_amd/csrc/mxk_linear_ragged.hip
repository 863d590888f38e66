// MFMA weight-only linear for gfx950 over weights whose blocks do not line up
// with 128-column tiles: N (mx_linear, [K][N]) or K ([N][K]: mx_dynamic_linear
// and the input gradients) no multiple of 128, or blocks other than 128.
//
//   y[m,n] = sum_k x[m,k] * c(k,n) * s[flat(k,n) / block],
//   flat = k N + n ([K][N], WT false) or n K + k ([N][K], WT true)
//
// A scale then covers neither a whole tile column nor a whole tile row, so it
// cannot go into the x operand or the epilogue as in mxk_linear_mfma.hip: the
// weight itself, c * s, goes in as an f16 pair hi + lo (22 significant bits)
// beside x's hi + lo, three v_mfma_f32_16x16x32_f16 per product (hi hi,
// lo hi, hi lo; the dropped lo lo term is 2^-22 of a product), fp32
// accumulation.  16-bit x has no lo part (mxk_linear_mfma.h): two.
//
// Work split.  A workgroup of 4 waves owns 128 columns; a wave takes RT row
// tiles of 16 rows and every WK-th step of 32 k (WM x WK = 4).  Lane (j, g)
// decodes codes of rows k 8g .. +7 and columns 8j .. +7, which are the B
// fragments it feeds to its own MFMAs (column tile t, MFMA column j is column
// 8j + t): no LDS and no barrier inside the loop.  8 consecutive codes of a
// row ([K][N]) or column ([N][K]) start anywhere in a dword: they come as
// whole aligned dwords and are brought together with v_alignbit.  With blocks
// of a power of two from 8 on a group of 8 codes meets at most one block boundary: two
// scales and a position.  Waves that split K meet in LDS in a fixed order, K
// splits across workgroups in a second kernel.
//
// What bounds it: few rows, the decode (about 480 VALU per 32 x 128 step of a
// wave) and the number of column tiles against CUs; many rows, decode and MFMA
// in equal parts (a wave decodes its weights for 64 rows).  16 x 4096 x 50257
// int8: 1149 us on the scalar kernel, here 96.8 (the profiler gives the product
// 98 and the prepass 6 us, each by itself); VALU instructions take 55% of the
// SIMDs' time, 73% where a CU holds two of the 393 tiles, MFMAs 9%.  1.2e-6 off
// the 64-bit product there, 3.0e-7 here.
//
// Range.  Both operands are scaled by powers of two to just below f16's largest
// values: rows of x by 2^ex[m], to [2^14, 2^15); the weight by 2^es, one per
// column ([N][K]) or per group of columns ([K][N]: of 8 for blocks below 128, of
// 32 from there on, whose columns share three blocks in four), that keeps the
// largest |c s| at most 2^15.  Scales that are not finite are left out of es:
// they spoil their own columns alone.  An f16 pair keeps 2^-25, so a value keeps
// 2^-38 of the largest of its row or columns.  With rows at [1, 2) x kept 2^-25
// of it, and outputs whose terms are of x large where the weight is small were
// off by 4e-3 (4e-7 here); with one es per 128 columns a column lost bits beside
// others 2^16 times larger.  Products are at most 2^30, their sums below 2^55.
//
// Infinities and NaN.  Only they, in x or in the scales, bring out a NaN here (inf -
// inf in a split, 0 * inf).  A NaN in a row of x is a NaN in all of its outputs.
// Any other one is summed again in fp32, over the terms that are not finite, so
// that infinities come out as the scalar kernel gives them: the wave looks for
// such terms 64 k at a time, and a lane sums its 4 rows x 8 columns of a row tile
// side by side until all are NaN.  64 x 2048 x 1001 int8, 83 us (scalar kernel
// 368): with a NaN 79 us, with infinities in every third row 555 (each output
// by one lane over all of K: 3.3 and 52 ms).  Where K is split, the second kernel
// finds them, one lane per output, and that lane sums all of K: 20 x 16384 x 1001
// 74 us, with infinities 1.7 ms (scalar kernel 3.9).
#include "mxk_linear_mfma.h"

#include <algorithm>
#include <type_traits>

namespace mxk {

namespace {

constexpr int RG_WAVES = 4;
constexpr int RG_CHUNKS = 8;  // parts of K that the largest scale of a group of columns is found in

struct RgArgs {
  const void* x;       // the caller's x (recomputed outputs)
  const _Float16* xh;  // hi and lo of x * 2^ex, tiled (lm_xoff)
  const _Float16* xl;
  const int* ex;       // [M]
  const float* smax;   // largest finite |scale|: [RG_CHUNKS][groups of 2^gsh columns of all tiles] or, WT, [N]
  const uint8_t* w;
  const float* scales;
  const float* bias;
  float* out;
  float* part;         // [S][M][N], or null
  int64_t K, Kp, N;
  uint32_t wbytes, sbytes, block, sh;  // block = 2^sh
  int M, x_type, wm, steps, sps, S;
  int tiles, per_xcd, mtiles;  // column tiles, those of one XCD, row groups
  int gsh;                     // ([K][N]) groups of 2^gsh columns share an exponent
};

// Largest |c s| 2^es is at most 2^15: s 2^es below 2^(15 - bits of the largest |c|)
__host__ __device__ constexpr int rg_scale_top(int fmt) {
  return fmt == LM_I8 ? 8 : fmt == LM_I4 ? 12 : fmt == LM_I2 ? 14 : fmt == LM_I1 ? 15 : fmt == LM_F8 ? 14 : 26;
}

// The exponent that brings the scales of column n to their range (0 for a zero maximum)
template <int FMT, bool WT>
__device__ __forceinline__ int rg_exponent(const RgArgs& a, int64_t n) {
  float mx = a.smax[WT ? n : n >> a.gsh];
  if constexpr (!WT) {
#pragma unroll
    for (int c = 1; c < RG_CHUNKS; ++c) mx = fmaxf(mx, a.smax[c * ((128 * a.tiles) >> a.gsh) + (n >> a.gsh)]);
  }
  const int be = (int)((__float_as_uint(mx) >> 23) & 0xFFu);
  return mx == 0.0f ? 0 : rg_scale_top(FMT) + 126 - (be == 0 ? 1 : be);
}

// The bits of |s|, 0 for infinities and NaN
__device__ __forceinline__ uint32_t rg_finite(float s) {
  const uint32_t b = mag_bits(s);
  return b < 0x7F800000u ? b : 0u;
}

// The packed codes of a lane's 8 x 8 block as loaded, and its scales
template <int BITS>
struct RgRaw {
  uint32_t d[8][BITS == 8 ? 3 : 2];
  uint32_t s[8][2];
};

// Byte b of w as a signed code, in float
__device__ __forceinline__ uint32_t rg_i8(uint32_t w, int b) { return __float_as_uint((float)(int8_t)(w >> (8 * b))); }

// Pair q (codes 2q, 2q + 1) of 8 codes that lie one after another in w0 (8-bit codes: w0, w1)
template <int FMT>
__device__ __forceinline__ uint32_t rg_pair_along(uint32_t w0, uint32_t w1, int q) {
  constexpr int BITS = lm_bits(FMT);
  if constexpr (BITS == 8) {
    const uint32_t w = q < 2 ? w0 : w1;
    return lm_pair<FMT>(__builtin_amdgcn_perm(w, w, lm_sel_f<FMT>(2 * (q & 1), 2 * (q & 1) + 1)));
  } else if constexpr (BITS == 4) {
    return lm_pair<FMT>(__builtin_amdgcn_perm(w0 >> 4, w0, lm_sel(q, q)));
  } else if constexpr (BITS == 2) {
    return lm_pair<FMT>(__builtin_amdgcn_perm(w0 >> 2, w0, lm_sel(q >> 1, q >> 1)) >> (4 * (q & 1)));
  } else {
    return lm_pair<FMT>(__builtin_amdgcn_perm(w0 >> 1, w0, lm_sel(0, 0)) >> (2 * q));
  }
}

// The weight c * s at flat index `flat` and the element (m, k) of x, in fp32
template <int FMT>
__device__ __forceinline__ float rg_weight(const RgArgs& a, uint32_t flat) {
  constexpr int BITS = lm_bits(FMT);
  const uint32_t bit = (flat & 7u) * BITS;  // (flat * BITS may not fit 32 bits)
  const uint32_t code = ((uint32_t)a.w[(flat >> 3) * BITS + (bit >> 3)] >> (bit & 7u)) & ((1u << BITS) - 1u);
  const uint32_t pair = lm_pair<FMT>(FMT == LM_F8 ? code << 8 : code);
  return (float)__builtin_bit_cast(h2v, pair)[0] * lm_post(FMT) * a.scales[flat >> a.sh];
}
__device__ __forceinline__ float rg_x(const RgArgs& a, int64_t m, int64_t k) {
  const int64_t at = m * a.K + k;
  return a.x_type == MXK_IN_F32   ? ((const float*)a.x)[at]
         : a.x_type == MXK_IN_F16 ? ElemT<__half>::cvt(((const __half*)a.x)[at])
                                  : ElemT<hip_bfloat16>::cvt(((const hip_bfloat16*)a.x)[at]);
}

// The places k0 .. k0 + 63 whose terms may not be finite in the row tile at mt
// (rows that hold a NaN aside) and the column tile at n0, as a mask; the wave's
// 64 lanes together
template <bool WT>
__device__ __forceinline__ uint64_t rg_odd(const RgArgs& a, int64_t mt, uint32_t n0, int64_t k0, int lane) {
  const int64_t kl = min(k0 + lane, a.K - 1);
  bool odd = false, all = false;
  auto rows = [&](const auto* x, uint32_t emask) {
#pragma unroll 4
    for (int r = 0; r < 16; ++r) {
      const int64_t m = min(mt + r, (int64_t)a.M - 1);
      const uint32_t b = x[m * a.K + kl];
      odd = odd || (a.ex[m] != LM_NAN_ROW && (b & emask) == emask);
    }
  };
  if (a.x_type == MXK_IN_F32) rows((const uint32_t*)a.x, 0x7F800000u);
  else rows((const uint16_t*)a.x, a.x_type == MXK_IN_F16 ? 0x7C00u : 0x7F80u);
  auto scales = [&](int64_t f0, int64_t f1) {
    bool hit = false;
    for (uint32_t q = (uint32_t)f0 >> a.sh; q <= (uint32_t)f1 >> a.sh; ++q)
      hit = hit || mag_bits(a.scales[q]) >= 0x7F800000u;
    return hit;
  };
  if constexpr (WT) {
    for (int64_t n = (int64_t)n0 + lane; n < min((int64_t)n0 + 128, a.N); n += 64)
      all = all || scales(n * a.K + k0, n * a.K + min(k0 + 63, a.K - 1));
  } else {
    odd = odd || scales(kl * a.N + n0, kl * a.N + min((int64_t)n0 + 127, a.N - 1));
  }
  const uint64_t in = a.K - k0 >= 64 ? ~0ull : (1ull << (a.K - k0)) - 1;
  return (__ballot(all) != 0 ? ~0ull : __ballot(odd)) & in;
}

// The outputs of the row tile at mt and the column tile at n0 that came out as NaN
// without one in their row, summed again by the wave that wrote them.  A
// function of its own, which reads the kernel's arguments (args: where they lie)
// itself: inlined, what it needs of them stayed in registers across the product's
// loop and 18 to 34 more of the loop's own spilled (64-row tiles of fp32 x: 48 x
// 4096 x 1000 int8 37.6 -> 44.6 us).
template <int FMT, bool WT>
__device__ __attribute__((noinline)) void rg_rescue(const RgArgs* args, int64_t mt, uint32_t n0, int lane) {
  const RgArgs& a = *args;
  const int64_t m = mt + 4 * (lane >> 4);
  const uint32_t nl = n0 + 8u * (lane & 15);
  uint32_t todo = 0u;  // bit 8 q + t: the output of row m + q and column nl + t (which this lane wrote)
  for (int e = 0; e < 32; ++e) {
    const int64_t mr = m + (e >> 3), n = (int64_t)nl + (e & 7);
    if (mr >= a.M || n >= a.N || a.ex[mr] == LM_NAN_ROW) continue;
    const float v = a.out[mr * a.N + n];
    todo |= (v != v ? 1u : 0u) << e;
  }
  if (__ballot(todo != 0u) == 0) return;
  float y[4][8];
#pragma unroll
  for (int e = 0; e < 32; ++e) y[e >> 3][e & 7] = 0.0f;
  bool open = true;
#pragma unroll 1
  for (int64_t k0 = 0; k0 < a.K && open; k0 += 64) {
    uint64_t odd = rg_odd<WT>(a, mt, n0, k0, lane);
    while (odd != 0 && open) {
      const int64_t k = k0 + __builtin_ctzll(odd);
      odd &= odd - 1;
      float xv[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) xv[q] = rg_x(a, min(m + q, (int64_t)a.M - 1), k);
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const int64_t n = min((int64_t)nl + t, a.N - 1);
        const float w = rg_weight<FMT>(a, (uint32_t)(WT ? n * a.K + k : k * a.N + n));
#pragma unroll
        for (int q = 0; q < 4; ++q) y[q][t] = __builtin_fmaf(xv[q], w, y[q][t]);
        if (t & 1) asm volatile("" ::: "memory");  // (addresses of two columns at a time, not of eight: no stack)
      }
      uint32_t nan = 0u;
#pragma unroll
      for (int e = 0; e < 32; ++e) nan |= (y[e >> 3][e & 7] != y[e >> 3][e & 7] ? 1u : 0u) << e;
      open = __ballot((todo & ~nan) != 0u) != 0;
    }
  }
#pragma unroll
  for (int e = 0; e < 32; ++e) {
    const int64_t n = (int64_t)nl + (e & 7);
    if ((todo >> e) & 1u) a.out[(m + (e >> 3)) * a.N + n] = y[e >> 3][e & 7] + (a.bias ? a.bias[n] : 0.0f);
  }
}

// the finished output from its sum in the scaled units
template <int FMT>
__device__ __forceinline__ float rg_finish(float v, int e) {
  const float y = __builtin_ldexpf(v, e);
  return lm_post(FMT) != 1.0f ? y * lm_post(FMT) : y;
}

template <int FMT, bool WT, int RT, bool XLO, bool STR>
__global__ __launch_bounds__(RG_WAVES * 64, 2) void k_linear_ragged(RgArgs a) {
  constexpr int BITS = lm_bits(FMT);
  constexpr int ND = BITS == 8 ? 3 : 2;
  __shared__ __attribute__((aligned(16))) f4v red[2 * RT * 8 * 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int WM = a.wm, WK = RG_WAVES / WM;
  const int wmi = wave % WM, wk = wave / WM;
  const int j = lane & 15, g = lane >> 4;
  // Neighbouring column tiles run on one XCD (workgroup b on XCD b % 8): a
  // tile's row of codes starts anywhere in a 128-byte line, so every row shares
  // its first and last line with the tiles beside it, and only one L2 then
  // fetches them.  Row groups of a tile, which read the same codes, follow one
  // another.
  const int xi = (int)(blockIdx.x >> 3);
  const int tile = (int)(blockIdx.x & 7) * a.per_xcd + (xi / a.mtiles) % a.per_xcd;
  const int z = xi / (a.mtiles * a.per_xcd);
  if (tile >= a.tiles) return;
  const int64_t m0 = ((int64_t)(xi % a.mtiles) * WM + wmi) * (16 * RT);
  const uint32_t n0 = tile * 128u, nl = n0 + 8u * j;
  const int s0 = z * a.sps, s1 = min(s0 + a.sps, a.steps);
  const uint32_t ldw = (uint32_t)(WT ? a.K : a.N);
  const int64_t rows16 = lm_rows16((int64_t)a.M - m0);
  const uint32_t xbytes = rows16 > 0 ? (uint32_t)((rows16 < 16 * RT ? rows16 : 16 * RT) * a.Kp * 2) : 0u;
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(a.w, a.wbytes), rs = make_rsrc(a.scales, a.sbytes);
  const __amdgpu_buffer_rsrc_t rh = make_rsrc(a.xh + m0 * a.Kp, xbytes);
  const __amdgpu_buffer_rsrc_t rl = make_rsrc(XLO ? a.xl + m0 * a.Kp : a.xh, XLO ? xbytes : 0u);

  int esv[8];
#pragma unroll
  for (int t = 0; t < 8; ++t)
    esv[t] = rg_exponent<FMT, WT>(a, WT ? min((int64_t)nl + t, a.N - 1) : (int64_t)nl);

  // Flat index of group 0 of a step (group i: row 8g + i, or column 8j + i).  The
  // last step takes the last 32 rows of K, x being zero where the step before has
  // them too (lm_prep_row): past K it would read the next column ([N][K]) or the
  // padding, whose scales may be past f16's range under this column's exponent or not
  // finite, and x's zero times infinity is NaN.  (Zeros in place of these scales, in
  // that step alone, cut the loop in two blocks and spilled: 300 x 2050 x 4098 int8, fp32
  // x, 144 us, so 82; without either 125.)
  auto flat0 = [&](int step) -> uint32_t {
    const uint32_t k = (uint32_t)min(32 * step, (int)a.K - 32) + 8u * g;
    return WT ? nl * ldw + k : k * ldw + nl;
  };
  // Loads are issued whether or not the step exists (`dead` offsets lie past
  // every buffer and read zeros), so that the wait counts stay exact.
  auto load_raw = [&](RgRaw<BITS>& r, int step, bool live, const int i0 = 0, const int i1 = 8) __attribute__((always_inline)) {
    const uint32_t dead = live ? 0u : LM_OOB;
    uint32_t f = flat0(step);
    f += i0 * ldw;
#pragma unroll
    for (int i = i0; i < i1; ++i) {
      const uint32_t off = (BITS == 8 ? f & ~3u : BITS == 4 ? (f >> 3) * 4u : BITS == 2 ? (f >> 4) * 4u : (f >> 5) * 4u) |
                           dead;
      if constexpr (ND == 3) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b96(rw, (int)off, 0, 0);
        r.d[i][0] = v[0];
        r.d[i][1] = v[1];
        r.d[i][2] = v[2];
      } else {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(rw, (int)off, 0, 0);
        r.d[i][0] = v[0];
        r.d[i][1] = v[1];
      }
      const uint32_t q = ((f >> a.sh) * 4u) | dead;
      if constexpr (STR) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(rs, (int)q, 0, 0);
        r.s[i][0] = v[0];
        r.s[i][1] = v[1];
      } else {
        r.s[i][0] = buf_load_b32(rs, q, 0u);
      }
      f += ldw;
    }
  };
  struct XA {
    u4v h[RT], l[XLO ? RT : 1];
  };
  auto load_x = [&](XA& x, int step, bool live) {
    const uint32_t dead = live ? 0u : LM_OOB;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const uint32_t at = (uint32_t)(lm_xoff(16 * i + j, 32 * (int64_t)step + 8 * g, a.Kp) * 2) | dead;
      x.h[i] = buf_load_b128(rh, at, 0u);
      if constexpr (XLO) x.l[i] = buf_load_b128(rl, at, 0u);
    }
  };

  f4v acc[RT][8];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[i][t] = f4v{0.f, 0.f, 0.f, 0.f};

  // Per step: the codes and scales loaded one step ahead are brought together
  // (after which the next step's can be requested into the same registers),
  // then each column tile is decoded and fed to its MFMAs in turn; the
  // scheduling barriers keep the tiles apart (one tile's fragments live).
  struct Step {
    KnCodes<BITS> c;
    float sa[8], sb[8];
    uint32_t pre[2];  // bit 8 (i % 4) + u of word i / 4: code u of group i lies before its block boundary
  };
  auto take = [&](Step& p, const RgRaw<BITS>& r, int step) {
    uint32_t f = flat0(step);
    if constexpr (STR) p.pre[0] = p.pre[1] = 0u;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t sh = BITS == 8 ? (f & 3u) * 8u : BITS == 4 ? (f & 7u) * 4u : BITS == 2 ? (f & 15u) * 2u : f & 31u;
      const uint32_t w = __builtin_amdgcn_alignbit(r.d[i][1], r.d[i][0], sh);
      if constexpr (BITS == 8) {
        p.c.w[2 * i] = w;
        p.c.w[2 * i + 1] = __builtin_amdgcn_alignbit(r.d[i][ND - 1], r.d[i][1], sh);
      } else {
        p.c.w[i] = BITS == 4 ? w : w & ((1u << (8 * BITS)) - 1u);
      }
      const int e = WT ? esv[i] : esv[0];
      p.sa[i] = __builtin_ldexpf(__uint_as_float(r.s[i][0]), e);
      if constexpr (STR) {
        p.sb[i] = __builtin_ldexpf(__uint_as_float(r.s[i][1]), e);
        p.pre[i >> 2] |= ((1u << min(a.block - (f & (a.block - 1u)), 8u)) - 1u) << (8 * (i & 3));
      }
      f += ldw;
    }
  };
  auto tiles = [&](const Step& p, const XA& x, const int t0, const int t1) __attribute__((always_inline)) {
    auto scale = [&](int i, const int u) __attribute__((always_inline)) -> float {  // of code u of group i
      if constexpr (!STR) return p.sa[i];
      // a mask by v_bfe_i32 and v_bfi: a compare and a select through VCC wait on each other
      uint32_t m;
      asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(m) : "v"(p.pre[i >> 2]), "s"(8 * (i & 3) + u));
      return __uint_as_float((__float_as_uint(p.sa[i]) & m) | (__float_as_uint(p.sb[i]) & ~m));
    };
#pragma unroll
    for (int t = t0; t < t1; ++t) {
      u4v bh, bl;
      u4v d = {0u, 0u, 0u, 0u};
      if constexpr (!WT && FMT != LM_I8) d = kn_frag<FMT>(p.c, t);
#pragma unroll
      for (int q = 0; q < 4; q += 2) {
        // codes 2q .. 2q + 3 of column t: rows ([K][N]) or places along the group ([N][K])
        uint32_t c[4], h0, h1, l0, l1;
        float s[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) s[u] = WT ? scale(t, 2 * q + u) : scale(2 * q + u, t);
        if constexpr (FMT == LM_I8) {
          // one convert a code, against a permute, an xor and half a packed subtraction
#pragma unroll
          for (int u = 0; u < 4; ++u)
            c[u] = WT ? rg_i8(p.c.w[2 * t + (q >> 1)], u) : rg_i8(p.c.w[2 * (2 * q + u) + (t >> 2)], t & 3);
          lm_split4<true>(c, s, h0, h1, l0, l1);
        } else {
          if constexpr (WT) {
            c[0] = rg_pair_along<FMT>(p.c.w[BITS == 8 ? 2 * t : t], p.c.w[BITS == 8 ? 2 * t + 1 : t], q);
            c[2] = rg_pair_along<FMT>(p.c.w[BITS == 8 ? 2 * t : t], p.c.w[BITS == 8 ? 2 * t + 1 : t], q + 1);
          } else {
            c[0] = d[q];
            c[2] = d[q + 1];
          }
          c[1] = c[3] = 0u;
          lm_split4<false>(c, s, h0, h1, l0, l1);
        }
        bh[q] = h0;
        bh[q + 1] = h1;
        bl[q] = l0;
        bl[q + 1] = l1;
      }
      lm_settle(bh, bl);
      const h8v h = __builtin_bit_cast(h8v, bh), l = __builtin_bit_cast(h8v, bl);
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const h8v xh = __builtin_bit_cast(h8v, x.h[i]);
        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, h, acc[i][t], 0, 0, 0);
        if constexpr (XLO)
          acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8v, x.l[i]), h, acc[i][t], 0, 0, 0);
        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, l, acc[i][t], 0, 0, 0);
      }
      if (t & 1) __builtin_amdgcn_sched_barrier(0);
    }
  };

  // This wave's steps s0 + wk, + WK, ...: codes DR steps ahead (few rows: the
  // loads in flight bound it), x one or DR steps ahead while the registers
  // allow it (64-row tiles: requested when the last MFMA of the step has read
  // it).  64-row tiles of [N][K] weights: column tile t needs the codes of group t
  // alone, so the second half of the next step's waits until the first half of the
  // tiles is done, which spares the registers to hold them (int8, fp32 x, 48 x 4096 x
  // 1000 37.3 us, else 39.1; 300 x 2050 x 4098 82, else 103).
  {
    constexpr bool HALF = WT && RT == 4;
    constexpr int DR = RT == 1 ? 2 : 1, DX = RT < 4 ? 2 : 1, U = DX;
    RgRaw<BITS> r[DR];
    XA x[DX];
    int st = s0 + wk;
#pragma unroll
    for (int d = 0; d < DR; ++d) {
      load_raw(r[d], st + d * WK, st + d * WK < s1);
      load_x(x[d], st + d * WK, st + d * WK < s1);
    }
    for (; st < s1; st += U * WK) {
#pragma unroll
      for (int p = 0; p < U; ++p) {
        const int cur = st + p * WK, nx = cur + DR * WK;  // a step past s1 computes on zeros
        Step sp;
        take(sp, r[p % DR], cur);
        load_raw(r[p % DR], nx, nx < s1, 0, HALF ? 4 : 8);
        if constexpr (DX == 2 && DR == 1) load_x(x[p ^ 1], nx, nx < s1);
        __builtin_amdgcn_sched_barrier(0);
        tiles(sp, x[p], 0, 4);
        if constexpr (HALF) {
          load_raw(r[p % DR], nx, nx < s1, 4, 8);
          __builtin_amdgcn_sched_barrier(0);
        }
        tiles(sp, x[p], 4, 8);
        if constexpr (DX == DR) load_x(x[p], nx, nx < s1);
      }
    }
  }

  // waves that split K: halves meet in LDS in a fixed order
  for (int half = WK >> 1; half >= 1; half >>= 1) {
    f4v* slot = red + (size_t)((wk & (half - 1)) * WM + wmi) * (RT * 8 * 64);
    __syncthreads();
    if (wk >= half && wk < 2 * half) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int t = 0; t < 8; ++t) slot[(i * 8 + t) * 64 + lane] = acc[i][t];
    }
    __syncthreads();
    if (wk < half) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const f4v v = slot[(i * 8 + t) * 64 + lane];
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[i][t][q] += v[q];
        }
    }
  }
  if (wk > 0) return;
  bool bad = false;
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t m = m0 + 16 * i + 4 * g + q;
      if (m >= a.M) continue;
      const int exm = a.part ? 0 : a.ex[m];
      float* dst = a.part ? a.part + ((int64_t)z * a.M + m) * a.N + nl : a.out + m * a.N + nl;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        if ((int64_t)nl + t >= a.N) continue;
        const float v = acc[i][t][q];
        bad = bad || (v != v && exm != LM_NAN_ROW);
        dst[t] = a.part ? v : rg_finish<FMT>(v, -(exm + esv[t])) + (a.bias ? a.bias[nl + t] : 0.0f);
      }
    }
  if (a.part || __ballot(bad) == 0) return;
#pragma unroll 1
  for (int i = 0; i < RT; ++i)
    rg_rescue<FMT, WT>((const RgArgs*)__builtin_amdgcn_kernarg_segment_ptr(), m0 + 16 * i, n0, lane);
}

// outputs from the K splits' partials, summed in split order
template <int FMT, bool WT>
__global__ __launch_bounds__(256) void k_linear_ragged_reduce(RgArgs a) {
  const int64_t total = (int64_t)a.M * a.N;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    float v = a.part[i];
    for (int z = 1; z < a.S; ++z) v += a.part[z * total + i];
    const int64_t m = i / a.N, n = i - m * a.N;
    float y = rg_finish<FMT>(v, -(a.ex[m] + rg_exponent<FMT, WT>(a, n)));
    if (v != v && a.ex[m] != LM_NAN_ROW) {
      y = 0.0f;
#pragma unroll 8
      for (int64_t k = 0; k < a.K; ++k)
        y = __builtin_fmaf(rg_x(a, m, k), rg_weight<FMT>(a, (uint32_t)(WT ? n * a.K + k : k * a.N + n)), y);
    }
    a.out[i] = a.bias ? y + a.bias[n] : y;
  }
}

// Workgroups 0 .. M - 1: a row of x each (lm_prep_row); the others the largest
// finite |scale|: of four columns each ([N][K], one wave per column), or ([K][N]) of
// the groups of columns of a run of column tiles over one of RG_CHUNKS parts of K.
// Blocks of 128 and more: 8 tiles, a row of them by 8 threads side by side, since
// their scales lie together (one tile per workgroup: 15 us at 4096 x 50257, so 5; few
// tiles as well: 5.2 at 4096 x 4098, so 4.4); at most two blocks meet a row of a
// tile, and the groups of 32 are kept in registers.  Smaller blocks: one tile, 16
// threads to a row, a thread to each group of 8.  Its loads depend on nothing, 16 at a
// time; a loop over a row's blocks with a maximum in LDS for each waited on every one
// (16 x 4096 x 1000 int8, blocks of 64: call 37.4 -> 21.5 us; the pass with 2 and 4 tiles
// per workgroup 6.1 and 9.6 us, so 4.4; at 4096 x 50257 15.2 and 18.6, so 14.2).
template <typename T, bool VEC, bool WT, bool LO>
__global__ __launch_bounds__(256) void k_linear_ragged_prep(const T* __restrict__ x, RgArgs a, _Float16* __restrict__ xh,
                                                            _Float16* __restrict__ xl, int* __restrict__ ex,
                                                            float* __restrict__ smax) {
  __shared__ float sm[4];
  const int tid = threadIdx.x, lane = tid & 63;
  if ((int64_t)blockIdx.x < a.M) {
    lm_prep_row<T, true, LM_X_TOP, VEC, LO>(x, lm_prep_m(blockIdx.x, a.M), a.K, a.Kp, a.Kp - 32, nullptr, xh, xl, ex, sm);
    return;
  }
  const int64_t b = (int64_t)blockIdx.x - a.M;
  if constexpr (WT) {
    const int64_t n = 4 * b + (tid >> 6);
    if (n >= a.N) return;
    float mx = 0.0f;
    const uint32_t q0 = (uint32_t)((n * a.K) >> a.sh), q1 = (uint32_t)((n * a.K + a.K - 1) >> a.sh);
    for (uint32_t q = q0 + lane; q <= q1; q += 64) mx = fmaxf(mx, __uint_as_float(rg_finite(a.scales[q])));
    mx = group_max<64>(mx);
    if (lane == 0) smax[n] = mx;
  } else {
    __shared__ uint32_t gm[128];  // [wave][tile][4 groups of 32], or [16 groups of 8]
    const uint32_t ch = (uint32_t)(b % RG_CHUNKS);
    const uint32_t N = (uint32_t)a.N, K = (uint32_t)a.K, tiles = (uint32_t)a.tiles, per = (K + RG_CHUNKS - 1) / RG_CHUNKS;
    const uint32_t k1 = min(K, (ch + 1) * per);
    if (a.gsh == 5) {
      const uint32_t tile0 = (uint32_t)(b / RG_CHUNKS) * 8u, tile = tile0 + (tid & 7), n0 = 128u * tile, cl = min(128u, N - n0) - 1u;  // (cl: its last column)
      uint32_t m[4] = {0u, 0u, 0u, 0u};
      if (tile < tiles) {
        // the loads of 8 rows at a time (past the last row: that row again)
        for (uint32_t k = ch * per + (tid >> 3); k < k1; k += 256) {
          uint32_t c[8];
          float s0[8], s1[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const uint32_t f = min(k + 32u * u, k1 - 1u) * N + n0, q = f >> a.sh;
            c[u] = ((q + 1u) << a.sh) - f;  // the second block's column
            s0[u] = a.scales[q];
            s1[u] = a.scales[(f + cl) >> a.sh];
          }
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const uint32_t v0 = rg_finite(s0[u]), v1 = rg_finite(s1[u]);
#pragma unroll
            for (uint32_t w = 0; w < 4; ++w) m[w] = max(m[w], max(32u * w < c[u] ? v0 : 0u, 32u * w + 32u > c[u] ? v1 : 0u));
          }
        }
      }
#pragma unroll
      for (int w = 0; w < 4; ++w) {
#pragma unroll
        for (int o = 8; o < 64; o <<= 1) m[w] = max(m[w], (uint32_t)__shfl_xor((int)m[w], o));
        if (lane < 8) gm[(tid >> 6) * 32 + 4 * lane + w] = m[w];
      }
      __syncthreads();
      if (tid < 32 && tile0 + tid / 4 < tiles)
        smax[ch * 4u * tiles + 4u * tile0 + tid] =
            __uint_as_float(max(max(gm[tid], gm[32 + tid]), max(gm[64 + tid], gm[96 + tid])));
    } else {
      // a thread: one group (at most two blocks meet its 8 columns) in every 16th row
      const uint32_t tile = (uint32_t)(b / RG_CHUNKS), gi = (uint32_t)tid & 15u, n = 128u * tile + 8u * gi;
      uint32_t m = 0u;
      if (n < N) {
        const uint32_t cl = min(7u, N - 1u - n);
        for (uint32_t k = ch * per + (tid >> 4); k < k1; k += 128) {
          float s0[8], s1[8];
#pragma unroll
          for (uint32_t u = 0; u < 8; ++u) {
            const uint32_t f = min(k + 16u * u, k1 - 1u) * N + n;
            s0[u] = a.scales[f >> a.sh];
            s1[u] = a.scales[(f + cl) >> a.sh];
          }
#pragma unroll
          for (int u = 0; u < 8; ++u) m = max(m, max(rg_finite(s0[u]), rg_finite(s1[u])));
        }
      }
#pragma unroll
      for (int o = 16; o < 64; o <<= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o));
      if (lane < 16) gm[(tid >> 6) * 16 + lane] = m;
      __syncthreads();
      if (tid < 16)
        smax[ch * 16u * tiles + 16u * tile + tid] =
            __uint_as_float(max(max(gm[tid], gm[16 + tid]), max(gm[32 + tid], gm[48 + tid])));
    }
  }
}

// ---------------------------------------------------------------- plan and launch
struct RgPlan {
  int rt = 1, wm = 1, S = 1, sps = 1, steps = 0;
  int64_t Kp = 0;
  size_t off_ex = 0, off_es = 0, off_x = 0, off_p = 0, bytes = 0;
};

// Shapes the kernel takes: one step of K at least, flat indices and every buffer
// below 2^31, blocks of a power of two from 8 on
bool rg_shape_ok(int64_t M, int64_t K, int64_t N, int bits, int64_t block) {
  const int64_t lim = int64_t(1) << 31;
  if (bits != 1 && bits != 2 && bits != 4 && bits != 8) return false;
  if (M < 1 || K < 32 || N < 1 || block < 8 || (block & (block - 1)) != 0 || block >= lim || K >= lim / 64 || N >= lim / 64) return false;
  if ((K + 64) * (N + 128) >= lim || M >= lim || 64 * (K + 32) * 2 >= lim) return false;
  return 8 * ceil_div(ceil_div(N, 128), 8) * ceil_div(M, 16) * 16 < lim;
}

// Rows: RT tiles of 16 per wave (few rows: fewer, they only cost MFMAs; from
// 33 rows on 4, the most the registers hold), waves side by side along M while
// there are rows for them.  K splits over workgroups, with at least 8 steps of
// 32 k left to a wave, to the number of splits with the least work on the
// fullest CU, a split (its partials and its start) counting as much as two
// steps and any split as much as eight (the second launch).
RgPlan rg_plan(int64_t M, int64_t K, int64_t N) {
  RgPlan p;
  p.steps = (int)ceil_div(K, 32);
  p.Kp = (int64_t)p.steps * 32;
  p.rt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  p.wm = M <= 64 ? 1 : M <= 128 ? 2 : 4;
  const int64_t groups = ceil_div(N, 128) * ceil_div(M, 16 * p.rt * p.wm);
  const int64_t most = std::max<int64_t>(1, p.steps / (8 * (RG_WAVES / p.wm)));
  int64_t best = -1;
  for (int64_t S = 1; S <= std::min<int64_t>(most, 16); ++S) {
    const int64_t cost = ceil_div(groups * S, num_cus()) * (ceil_div(p.steps, S * (RG_WAVES / p.wm)) + 2) + (S > 1 ? 8 : 0);
    if (best < 0 || cost < best) {
      best = cost;
      p.S = (int)S;
    }
  }
  p.sps = (int)ceil_div(p.steps, p.S);
  p.S = (int)ceil_div(p.steps, p.sps);
  size_t o = LM_WS_BASE;
  p.off_ex = o;
  o += lm_round((size_t)M * 4);
  p.off_es = o;
  o += lm_round((size_t)ceil_div(N, 128) * 128 * 4);  // N, or RG_CHUNKS times at most 16 groups per tile
  p.off_x = o;
  o += lm_round((size_t)lm_rows16(M) * (size_t)p.Kp * 4);
  p.off_p = o;
  if (p.S > 1) o += lm_round((size_t)p.S * (size_t)M * (size_t)N * 4);
  p.bytes = o;
  return p;
}

template <int FMT, bool WT, bool STR>
void rg_launch(const RgPlan& p, const RgArgs& a, bool xlo, hipStream_t st) {
  const dim3 grid((unsigned)(8 * (int64_t)a.per_xcd * a.mtiles * p.S));
  const dim3 blk(RG_WAVES * 64);
  if (p.rt == 1) hipLaunchKernelGGL((k_linear_ragged<FMT, WT, 1, true, STR>), grid, blk, 0, st, a);
  else if (p.rt == 2) hipLaunchKernelGGL((k_linear_ragged<FMT, WT, 2, true, STR>), grid, blk, 0, st, a);
  else if (xlo) hipLaunchKernelGGL((k_linear_ragged<FMT, WT, 4, true, STR>), grid, blk, 0, st, a);
  else hipLaunchKernelGGL((k_linear_ragged<FMT, WT, 4, false, STR>), grid, blk, 0, st, a);
  if (p.S > 1) {
    const int64_t wgs = std::min<int64_t>(ceil_div((int64_t)a.M * a.N, 256), 16 * (int64_t)num_cus());
    hipLaunchKernelGGL((k_linear_ragged_reduce<FMT, WT>), dim3((unsigned)wgs), dim3(256), 0, st, a);
  }
}

template <int FMT, bool WT>
void rg_launch_s(const RgPlan& p, const RgArgs& a, bool xlo, bool straddle, hipStream_t st) {
  // 1- and 2-bit weights: the general form only
  if constexpr (lm_bits(FMT) >= 4) {
    if (!straddle) return rg_launch<FMT, WT, false>(p, a, xlo, st);
  }
  rg_launch<FMT, WT, true>(p, a, xlo, st);
}

// workgroups of the prepass that find the largest scales
int64_t rg_max_groups(bool nk, const RgArgs& a) {
  return nk ? ceil_div(a.N, 4) : RG_CHUNKS * ceil_div(a.tiles, a.gsh == 5 ? 8 : 1);
}

template <bool WT, typename T>
void rg_prep(const RgPlan& p, const RgArgs& a, _Float16* xh, _Float16* xl, int* ex, float* smax, hipStream_t st) {
  const dim3 grid((unsigned)(a.M + rg_max_groups(WT, a)));
  const T* x = (const T*)a.x;
  const bool vec = aligned16(x) && (a.K * (int64_t)sizeof(T)) % 16 == 0;
  // only the 64-row tiles have a form without lo
  if constexpr (sizeof(T) == 2) {
    if (p.rt == 4) {
      if (vec) hipLaunchKernelGGL((k_linear_ragged_prep<T, true, WT, false>), grid, dim3(256), 0, st, x, a, xh, xl, ex, smax);
      else hipLaunchKernelGGL((k_linear_ragged_prep<T, false, WT, false>), grid, dim3(256), 0, st, x, a, xh, xl, ex, smax);
      return;
    }
  }
  if (vec) hipLaunchKernelGGL((k_linear_ragged_prep<T, true, WT, true>), grid, dim3(256), 0, st, x, a, xh, xl, ex, smax);
  else hipLaunchKernelGGL((k_linear_ragged_prep<T, false, WT, true>), grid, dim3(256), 0, st, x, a, xh, xl, ex, smax);
}

template <bool WT>
int rg_run(const void* x, int x_type, int64_t M, int64_t K, const void* w, int64_t w_nbytes, const float* scales,
           int64_t nscales, int64_t N, int kind, int bits, int block, const float* bias, float* out, void* workspace,
           size_t workspace_nbytes, hipStream_t st) {
  const int fmt = lm_format(kind, bits);
  if (fmt == 0 || !rg_shape_ok(M, K, N, bits, block)) return MXK_EUNSUPPORTED;
  if (x_type != MXK_IN_F32 && x_type != MXK_IN_F16 && x_type != MXK_IN_BF16) return MXK_EUNSUPPORTED;
  const RgPlan p = rg_plan(M, K, N);
  // whole aligned dwords of codes are loaded; without a workspace the scalar kernel runs
  if (!workspace || workspace_nbytes < p.bytes || (reinterpret_cast<uintptr_t>(w) & 3u) != 0 || w_nbytes % 4 != 0 ||
      w_nbytes >= (int64_t(1) << 31))
    return MXK_EUNSUPPORTED;
  uint8_t* ws = reinterpret_cast<uint8_t*>(workspace);
  _Float16* xh = reinterpret_cast<_Float16*>(ws + p.off_x);
  _Float16* xl = xh + (size_t)lm_rows16(M) * (size_t)p.Kp;
  int* ex = reinterpret_cast<int*>(ws + p.off_ex);
  float* smax = reinterpret_cast<float*>(ws + p.off_es);
  int l = 0;
  while ((int64_t(1) << l) < block) ++l;
  RgArgs a;
  a.x = x;
  a.xh = xh;
  a.xl = xl;
  a.ex = ex;
  a.smax = smax;
  a.w = reinterpret_cast<const uint8_t*>(w);
  a.scales = scales;
  a.bias = bias;
  a.out = out;
  a.part = p.S > 1 ? reinterpret_cast<float*>(ws + p.off_p) : nullptr;
  a.K = K;
  a.Kp = p.Kp;
  a.N = N;
  a.wbytes = (uint32_t)w_nbytes;
  a.sbytes = (uint32_t)(nscales * 4);
  a.block = (uint32_t)block;
  a.sh = (uint32_t)l;
  a.M = (int)M;
  a.x_type = x_type;
  a.wm = p.wm;
  a.steps = p.steps;
  a.sps = p.sps;
  a.S = p.S;
  a.tiles = (int)ceil_div(N, 128);
  a.gsh = l >= 7 ? 5 : 3;
  a.per_xcd = (int)ceil_div(a.tiles, 8);
  a.mtiles = (int)ceil_div(M, 16 * p.rt * p.wm);
  if (x_type == MXK_IN_F32) rg_prep<WT, float>(p, a, xh, xl, ex, smax, st);
  else if (x_type == MXK_IN_F16) rg_prep<WT, __half>(p, a, xh, xl, ex, smax, st);
  else rg_prep<WT, hip_bfloat16>(p, a, xh, xl, ex, smax, st);
  const bool xlo = x_type == MXK_IN_F32;
  const bool straddle = (WT ? K : N) % 8 != 0;
  switch (fmt) {
    case LM_I1: rg_launch_s<LM_I1, WT>(p, a, xlo, straddle, st); break;
    case LM_I2: rg_launch_s<LM_I2, WT>(p, a, xlo, straddle, st); break;
    case LM_I4: rg_launch_s<LM_I4, WT>(p, a, xlo, straddle, st); break;
    case LM_I8: rg_launch_s<LM_I8, WT>(p, a, xlo, straddle, st); break;
    case LM_F4: rg_launch_s<LM_F4, WT>(p, a, xlo, straddle, st); break;
    case LM_F8: rg_launch_s<LM_F8, WT>(p, a, xlo, straddle, st); break;
  }
  return check_launch(WT ? "linear_wq_nt(ragged)" : "linear_wq(ragged)");
}

}  // namespace

// ---------------------------------------------------------------- internal entry points
size_t linear_ragged_workspace(int64_t M, int64_t K, int64_t N, int bits, int64_t block) {
  return rg_shape_ok(M, K, N, bits, block) ? rg_plan(M, K, N).bytes : 0;
}

int linear_ragged_kn(const void* x, int x_type, int64_t M, int64_t K, const void* w, int64_t w_nbytes,
                     const float* scales, int64_t nscales, int64_t N, int kind, int bits, int block,
                     const float* bias, float* out, void* workspace, size_t workspace_nbytes, hipStream_t st) {
  return rg_run<false>(x, x_type, M, K, w, w_nbytes, scales, nscales, N, kind, bits, block, bias, out, workspace,
                       workspace_nbytes, st);
}

int linear_ragged_nk(const void* x, int x_type, int64_t M, int64_t K, const void* w, int64_t w_nbytes,
                     const float* scales, int64_t nscales, int64_t N, int kind, int bits, int block,
                     const float* bias, float* out, void* workspace, size_t workspace_nbytes, hipStream_t st) {
  return rg_run<true>(x, x_type, M, K, w, w_nbytes, scales, nscales, N, kind, bits, block, bias, out, workspace,
                      workspace_nbytes, st);
}

}  // namespace mxk

// What the two MFMA weight-only linears share (mxk_linear_mfma.hip and
// mxk_linear_ragged.hip): weight formats and their f16 B operands, the hi + lo
// split, the tiled layout of the scaled x and the pass that writes it.
#pragma once
#include "mxk_internal.h"

#include <algorithm>

namespace mxk {

namespace {

typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));

constexpr uint32_t LM_OOB = 0x80000000u;       // past every buffer: loads return zeros
constexpr size_t LM_WS_BASE = 65536;           // workspace bytes left to the decode kernels' counters

// Integer codes as f16 pairs of c 2^-E (E 0 or 14): all values are exact and
// normal, and E only changes constants.  The f16 2^(10 - E) with code bits in its
// low bits is (1024 + code) 2^-E.
template <int E>
__device__ __forceinline__ uint32_t lm_ipair(uint32_t d, uint32_t flip, float bias) {
  const uint32_t e = d ^ (((0x6400u - ((uint32_t)E << 10)) | flip) * 0x00010001u);
  const _Float16 b = (_Float16)((1024.0f + bias) / (float)(1 << E));
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2v, e) - h2v{b, b});
}
// Two int4 codes at bits 0-3 and 16-19 of d (other bits ignored): c ^ 8 is c + 8
template <int E = 0>
__device__ __forceinline__ uint32_t lm_i4pair(uint32_t d) {
  return lm_ipair<E>(d & 0x000F000Fu, 8u, 8.0f);
}
// Two int8 codes at bits 0-7 and 16-23 of d (bits 8-15, 24-31 zero)
template <int E = 0>
__device__ __forceinline__ uint32_t lm_i8pair(uint32_t d) {
  return lm_ipair<E>(d, 0x80u, 128.0f);
}
// Two int2 codes at bits 0-1 and 16-17 of d (other bits ignored)
template <int E = 0>
__device__ __forceinline__ uint32_t lm_i2pair(uint32_t d) {
  return lm_ipair<E>(d & 0x00030003u, 2u, 2.0f);
}
// Two int1 codes at bits 0 and 16 of d (other bits ignored): code 0 is
// +1 and code 1 is -1 (the reference's 1-bit grid), so the code is the f16
// sign bit of 2^-E.
template <int E = 0>
__device__ __forceinline__ uint32_t lm_i1pair(uint32_t d) {
  return ((d & 0x00010001u) << 15) | ((0x3C00u - ((uint32_t)E << 10)) * 0x00010001u);
}
// Weight formats: the code width in the low 4 bits, 16 for float grids
enum : int { LM_I1 = 1, LM_I2 = 2, LM_I4 = 4, LM_I8 = 8, LM_F4 = 16 + 4, LM_F8 = 16 + 8 };
__host__ __device__ constexpr int lm_bits(int fmt) { return fmt & 15; }
// The factor the outputs take for B fragments that hold v * 2^-P instead of
// the grid value v / vmax: RN(1/6) * 2^14, RN(1/480) * 2^8, or 1 for integer
// codes.
__host__ __device__ constexpr float lm_post(int fmt) {
  return fmt == LM_F4 ? (1.0f / 6.0f) * 16384.0f : fmt == LM_F8 ? (1.0f / 480.0f) * 256.0f : 1.0f;
}
inline int lm_format(int kind, int bits) {
  if (kind == MXK_KIND_INT) return bits == 1 ? LM_I1 : bits == 2 ? LM_I2 : bits == 4 ? LM_I4 : bits == 8 ? LM_I8 : 0;
  if (kind == MXK_KIND_FLOAT) return bits == 4 ? LM_F4 : bits == 8 ? LM_F8 : 0;
  return 0;
}
// Two codes of a format (layout of its width) as an f16 B-operand pair (integer
// codes: times 2^-E)
template <int FMT, int E = 0>
__device__ __forceinline__ uint32_t lm_pair(uint32_t d) {
  if constexpr (FMT == LM_I4) return lm_i4pair<E>(d);
  else if constexpr (FMT == LM_I8) return lm_i8pair<E>(d);
  else if constexpr (FMT == LM_I2) return lm_i2pair<E>(d);
  else if constexpr (FMT == LM_I1) return lm_i1pair<E>(d);
  else return fp_code_pair_f16<lm_bits(FMT)>(d);
}

// v_perm_b32 selector: byte a of s1 into byte 0, byte b of s0 into byte 2, zeros in bytes 1 and 3
__host__ __device__ constexpr uint32_t lm_sel(int a, int b) {
  return (uint32_t)a | 0x0C00u | ((uint32_t)(4 + b) << 16) | 0x0C000000u;
}
// the same bytes into bytes 1 and 3 (FP8 codes at the top of each half), zeros in bytes 0 and 2
__host__ __device__ constexpr uint32_t lm_selh(int a, int b) {
  return 0x0Cu | ((uint32_t)a << 8) | 0x0C0000u | ((uint32_t)(4 + b) << 24);
}
// the byte-pair selector a format's pair decoder takes
template <int FMT>
__host__ __device__ constexpr uint32_t lm_sel_f(int a, int b) {
  return FMT == LM_F8 ? lm_selh(a, b) : lm_sel(a, b);
}

// p = c * s as f16 hi + lo for four elements: hi = RN16(c s), lo = RN16(c s -
// hi), each one v_fma_mix (fp32 product, f16 result), so |c s - hi - lo| <= 2^-22
// |c s| (less for values whose lo is subnormal: at most 2^-25 absolute).  c is
// four floats (F32) or two f16 pairs, in c[0] and c[2].  One asm statement: an
// instruction that writes the high half of a register may not be followed at once
// by one that reads it, and the compiler, which may move single asm statements
// about, does not see that they do.  Here another one always lies between, and
// the last two write low halves.  (The two wait states before an MFMA: lm_settle.)
template <bool F32>
__device__ __forceinline__ void lm_split4(const uint32_t (&c)[4], const float (&s)[4], uint32_t& h0, uint32_t& h1,
                                          uint32_t& l0, uint32_t& l1) {
  if constexpr (F32) {
    asm("v_fma_mixlo_f16 %0, %4, %8, 0 op_sel_hi:[0,0,0]\n\t"
        "v_fma_mixlo_f16 %1, %6, %10, 0 op_sel_hi:[0,0,0]\n\t"
        "v_fma_mixhi_f16 %0, %5, %9, 0 op_sel_hi:[0,0,0]\n\t"
        "v_fma_mixhi_f16 %1, %7, %11, 0 op_sel_hi:[0,0,0]\n\t"
        "v_fma_mixhi_f16 %2, %5, %9, -%0 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %3, %7, %11, -%1 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %2, %4, %8, -%0 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %3, %6, %10, -%1 op_sel_hi:[0,0,1]"
        : "=&v"(h0), "=&v"(h1), "=&v"(l0), "=&v"(l1)
        : "v"(c[0]), "v"(c[1]), "v"(c[2]), "v"(c[3]), "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(s[3]));
  } else {
    asm("v_fma_mixlo_f16 %0, %4, %6, 0 op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixlo_f16 %1, %5, %8, 0 op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixhi_f16 %0, %4, %7, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixhi_f16 %1, %5, %9, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixhi_f16 %2, %4, %7, -%0 op_sel:[1,0,1] op_sel_hi:[1,0,1]\n\t"
        "v_fma_mixhi_f16 %3, %5, %9, -%1 op_sel:[1,0,1] op_sel_hi:[1,0,1]\n\t"
        "v_fma_mixlo_f16 %2, %4, %6, -%0 op_sel_hi:[1,0,1]\n\t"
        "v_fma_mixlo_f16 %3, %5, %8, -%1 op_sel_hi:[1,0,1]"
        : "=&v"(h0), "=&v"(h1), "=&v"(l0), "=&v"(l1)
        : "v"(c[0]), "v"(c[2]), "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(s[3]));
  }
}

// Two wait states between the asm instructions that wrote a and b and the
// MFMAs that read them: an MFMA may read a register two states after a VALU
// wrote it, and the compiler, which sees no VALU instruction in an asm
// statement, leaves them out (wrong operands were seen without them).
__device__ __forceinline__ void lm_settle(u4v& a, u4v& b) { asm volatile("s_nop 1" : "+v"(a), "+v"(b)); }
// the same for whatever was written before this point
__device__ __forceinline__ void lm_settle() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 1");
  __builtin_amdgcn_sched_barrier(0);
}

// s_barrier after this wave's LDS stores are done; global loads still in
// flight (prefetches) stay in flight.
__device__ __forceinline__ void lm_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The codes of rows 8 r8 .. +7 and columns 8 c8 .. +7 of a [K][N] weight,
// one row per word (8-bit codes: two)
template <int BITS>
struct KnCodes {
  uint32_t w[BITS == 8 ? 16 : 8];
};

// the B fragment of column tile t (column 8 c8 + t) from the thread's block
template <int FMT>
__device__ __forceinline__ u4v kn_frag(const KnCodes<lm_bits(FMT)>& c, int t) {
  constexpr int BITS = lm_bits(FMT);
  u4v f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if constexpr (BITS == 1) {
      // rows 2q and 2q+1 (8 bits each) 16 bits apart: column 8 c8 + t at bits t, 16 + t
      const uint32_t d = c.w[2 * q] | (c.w[2 * q + 1] << 16);
      f[q] = lm_pair<FMT>(d >> t);
    } else if constexpr (BITS == 2) {
      // rows 2q and 2q+1 (16 bits each) side by side: column 8 c8 + t at bits 2t, 2t + 1
      const uint32_t d = c.w[2 * q] | (c.w[2 * q + 1] << 16);
      f[q] = lm_pair<FMT>(d >> (2 * t));
    } else if constexpr (BITS == 4) {
      // byte t/2 of rows 2q and 2q+1: the low nibbles are column 8 c8 + t for even t
      const uint32_t d = __builtin_amdgcn_perm(c.w[2 * q + 1], c.w[2 * q], lm_sel(t >> 1, t >> 1));
      f[q] = lm_pair<FMT>((t & 1) ? d >> 4 : d);
    } else {
      const int h = t >> 2, u = t & 3;
      f[q] = lm_pair<FMT>(
          __builtin_amdgcn_perm(c.w[2 * (2 * q + 1) + h], c.w[2 * (2 * q) + h], lm_sel_f<FMT>(u, u)));
    }
  }
  return f;
}

// x' (and its f16 hi / lo) in HBM as tiles of 16 rows x 8 columns of K,
// tile (m / 16, k / 8) at element ((m / 16) * Kp/8 + k / 8) * 128 and
// element (m % 16) * 8 + k % 8 inside it, so that the 64 lanes of an A
// operand load (rows j of a row tile, columns 8 g .. 8 g + 7 of a k step)
// read one contiguous 2 KiB (fp32) or 1 KiB (f16): with x' row-major the 16
// rows of one load are Kp elements apart and land on one memory channel.
__host__ __device__ __forceinline__ int64_t lm_xoff(int64_t m, int64_t k, int64_t Kp) {
  return ((m >> 4) * (Kp >> 3) + (k >> 3)) * 128 + (m & 15) * 8 + (k & 7);
}
// rows of x' the tiled layout holds (whole row tiles)
__host__ __device__ __forceinline__ int64_t lm_rows16(int64_t M) { return (M + 15) & ~(int64_t)15; }

// ---------------------------------------------------------------- prepasses
// Rows of x in f16 pairs have their largest value in [2^14, 2^15): the pair then
// keeps 2^-39 of it (at [1, 2): 2^-25).  The products stay far below fp32's limit.
constexpr int LM_X_TOP = 14;

// ex[m] of a row that holds a NaN: all its outputs are NaN, whatever they are scaled by
constexpr int LM_NAN_ROW = 1 << 20;

// Row m of x: ex[m] such that its largest |x| times 2^ex lies in [2^TOP,
// 2^(TOP + 1)) (0 for a zero row), and x * 2^ex on Kp columns, those from Kz on
// moved to the end and zeros before them (Kz = K: zeros at the end), as
// fp32 (SPLIT false) or as f16 hi + lo (SPLIT true: hi = RN16(v), lo = RN16(v -
// hi), v - hi exact in fp32; a value keeps 2^-25, so 2^(-25 - TOP) of its row's
// largest).  VEC: 16-byte rows (K * sizeof(T) % 16 == 0, x
// 16-byte aligned); rows of up to 2048 16-byte chunks stay in registers
// between the maximum and the scaled copy, longer ones are read twice.
// LO false (16-bit x only) leaves lo out: an fp16 or bf16 value times a
// power of two is its own hi, down to values below half of f16's smallest
// subnormal, whose lo rounds to zero.
template <typename T, bool SPLIT, bool LO>
__device__ __forceinline__ void lm_put(float* __restrict__ xs, _Float16* __restrict__ xh, _Float16* __restrict__ xl,
                                       int64_t at, float v) {
  if constexpr (SPLIT) {
    const _Float16 h = (_Float16)v;
    xh[at] = h;
    if constexpr (LO) xl[at] = (_Float16)(v - (float)h);
  } else {
    xs[at] = v;
  }
}

// The row that workgroup b of the row pass takes: the 16 rows of a row tile go to
// one XCD (workgroup b runs on XCD b % 8), since every 128-byte line of the
// tiled layout holds 16 bytes of each of 8 of them: with row b on XCD b % 8,
// eight L2s wrote pieces of each line (2048 x 4096 bf16: 31 -> 11.5 us with no lo
// to write either; fp32 x to fp32 22 -> 15.5 us).
__device__ __forceinline__ int64_t lm_prep_m(int64_t b, int64_t M) {
  return b < (M & ~(int64_t)127) ? (b & ~(int64_t)127) + (b & 7) * 16 + ((b >> 3) & 15) : b;
}

// Row m by one workgroup of 256 threads (red: 4 floats of LDS)
template <typename T, bool SPLIT, int TOP, bool VEC, bool LO = true>
__device__ __forceinline__ void lm_prep_row(const T* __restrict__ x, int64_t m, int64_t K, int64_t Kp, int64_t Kz,
                                            float* __restrict__ xs, _Float16* __restrict__ xh,
                                            _Float16* __restrict__ xl, int* __restrict__ ex, float* red) {
  static_assert(LO || (SPLIT && sizeof(T) == 2), "fp32 x needs lo");
  constexpr int E = 16 / (int)sizeof(T), NCH = 8;
  const int tid = threadIdx.x;
  const T* row = x + m * K;
  const int64_t nch = K / E;
  const bool cached = VEC && nch <= (int64_t)NCH * 256;
  u4v c[NCH];
  auto elems = [&](const u4v& w, float (&v)[E]) {
    const T* t = reinterpret_cast<const T*>(&w);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = ElemT<T>::cvt(t[e]);
  };
  uint32_t mx = 0u;
  if (cached) {
#pragma unroll
    for (int q = 0; q < NCH; ++q) {
      const int64_t ch = tid + 256 * q;
      c[q] = ch < nch ? *reinterpret_cast<const u4v*>(row + ch * E) : u4v{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int q = 0; q < NCH; ++q) {
      float v[E];
      elems(c[q], v);
#pragma unroll
      for (int e = 0; e < E; ++e) mx = max(mx, mag_bits(v[e]));
    }
  } else {
    for (int64_t k = tid; k < K; k += 256) mx = max(mx, mag_bits(ElemT<T>::cvt(row[k])));
  }
  mx = group_max_u<64>(mx);
  if ((tid & 63) == 0) red[tid >> 6] = __uint_as_float(mx);
  __syncthreads();
  mx = max(max(__float_as_uint(red[0]), __float_as_uint(red[1])), max(__float_as_uint(red[2]), __float_as_uint(red[3])));
  const int be = (int)(mx >> 23);
  const int e = (be == 0xFF || mx == 0u) ? 0 : 127 + TOP - (be == 0 ? 1 : be);
  if (tid == 0) ex[m] = mx > 0x7F800000u ? LM_NAN_ROW : e;
  if (cached) {
#pragma unroll
    for (int q = 0; q < NCH; ++q) {
      const int64_t ch = tid + 256 * q;
      if (ch >= nch) break;
      float v[E];
      elems(c[q], v);
#pragma unroll
      for (int u = 0; u < E; ++u) v[u] = __builtin_ldexpf(v[u], e);
      // E <= 8 values within one 8-column group (Kp - K is a multiple of E, as K and Kp are)
      const int64_t at = lm_xoff(m, ch * E + (ch * E >= Kz ? Kp - K : 0), Kp);
      if constexpr (SPLIT) {
        _Float16 h[E], l[E];
#pragma unroll
        for (int u = 0; u < E; ++u) {
          h[u] = (_Float16)v[u];
          l[u] = (_Float16)(v[u] - (float)h[u]);
        }
        if constexpr (E == 4) {
          *reinterpret_cast<u2v*>(xh + at) = __builtin_bit_cast(u2v, h);
          *reinterpret_cast<u2v*>(xl + at) = __builtin_bit_cast(u2v, l);
        } else {
          *reinterpret_cast<u4v*>(xh + at) = __builtin_bit_cast(u4v, h);
          if constexpr (LO) *reinterpret_cast<u4v*>(xl + at) = __builtin_bit_cast(u4v, l);
        }
      } else {
#pragma unroll
        for (int u = 0; u < E; u += 4) *reinterpret_cast<f4v*>(xs + at + u) = f4v{v[u], v[u + 1], v[u + 2], v[u + 3]};
      }
    }
    for (int64_t k = Kz + tid; k < Kz + Kp - K; k += 256) lm_put<T, SPLIT, LO>(xs, xh, xl, lm_xoff(m, k, Kp), 0.0f);
  } else {
    for (int64_t k = tid; k < Kp; k += 256) {
      const int64_t from = k < Kz ? k : k - (Kp - K);
      lm_put<T, SPLIT, LO>(xs, xh, xl, lm_xoff(m, k, Kp),
                           k < Kz || from >= Kz ? __builtin_ldexpf(ElemT<T>::cvt(row[from]), e) : 0.0f);
    }
  }
}

// Workgroups M .. M + NB - 1 (the [K][N] product) find es[nb] instead: the
// power of two that puts the largest |scale| of column block nb (row nb of
// the block-major scales sT [NB][K]) in [2^13, 2^14), 0 for a zero or
// non-finite maximum.  It depends on the weight alone; computed here, it is
// ready before the main kernel starts.
template <typename T, bool SPLIT, bool VEC, bool LO>
__global__ __launch_bounds__(256) void k_linear_mfma_prep_rows(const T* __restrict__ x, int64_t M, int64_t K,
                                                               int64_t Kp, float* __restrict__ xs,
                                                               _Float16* __restrict__ xh, _Float16* __restrict__ xl,
                                                               int* __restrict__ ex, const float* __restrict__ sT,
                                                               int* __restrict__ es) {
  __shared__ float red[4];
  const int tid = threadIdx.x;
  if ((int64_t)blockIdx.x >= M) {
    const int64_t nb = (int64_t)blockIdx.x - M;
    const float* s = sT + nb * K;
    float mx = 0.0f;
    int64_t k = tid;
    for (; k + 7 * 256 < K; k += 8 * 256) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = s[k + 256 * u];
#pragma unroll
      for (int u = 0; u < 8; ++u) mx = fmaxf(mx, __builtin_fabsf(v[u]));
    }
    for (; k < K; k += 256) mx = fmaxf(mx, __builtin_fabsf(s[k]));
    mx = group_max<64>(mx);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    if (tid == 0) {
      mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
      const int be = (int)((__float_as_uint(mx) >> 23) & 0xFFu);
      es[nb] = (be == 0xFF || mx == 0.0f) ? 0 : 140 - (be == 0 ? 1 : be);
    }
    return;
  }
  lm_prep_row<T, SPLIT, SPLIT ? LM_X_TOP : 0, VEC, LO>(x, lm_prep_m(blockIdx.x, M), K, Kp, K, xs, xh, xl, ex, red);
}

inline size_t lm_round(size_t v) { return (v + 255) & ~(size_t)255; }

// rows of x (and, with sT, the NB column-block exponents of a [K][N] weight)
template <typename T, bool SPLIT>
void lm_prep_rows_t(const T* x, int64_t M, int64_t K, int64_t Kp, float* xs, _Float16* xh, _Float16* xl, int* ex,
                    const float* sT, int64_t NB, int* es, hipStream_t st) {
  // 16-bit x has no lo part (lm_put)
  constexpr bool LO = !SPLIT || sizeof(T) == 4;
  const dim3 grid((unsigned)(M + (sT ? NB : 0)));
  if (aligned16(x) && (K * (int64_t)sizeof(T)) % 16 == 0)
    hipLaunchKernelGGL((k_linear_mfma_prep_rows<T, SPLIT, true, LO>), grid, dim3(256), 0, st, x, M, K, Kp, xs, xh, xl, ex,
                       sT, es);
  else
    hipLaunchKernelGGL((k_linear_mfma_prep_rows<T, SPLIT, false, LO>), grid, dim3(256), 0, st, x, M, K, Kp, xs, xh, xl,
                       ex, sT, es);
}

template <bool SPLIT>
void lm_prep_rows(const void* x, int x_type, int64_t M, int64_t K, int64_t Kp, float* xs, _Float16* xh, _Float16* xl,
                  int* ex, const float* sT, int64_t NB, int* es, hipStream_t st) {
  if (x_type == MXK_IN_F32) lm_prep_rows_t<float, SPLIT>((const float*)x, M, K, Kp, xs, xh, xl, ex, sT, NB, es, st);
  else if (x_type == MXK_IN_F16)
    lm_prep_rows_t<__half, SPLIT>((const __half*)x, M, K, Kp, xs, xh, xl, ex, sT, NB, es, st);
  else lm_prep_rows_t<hip_bfloat16, SPLIT>((const hip_bfloat16*)x, M, K, Kp, xs, xh, xl, ex, sT, NB, es, st);
}

}  // namespace

}  // namespace mxk

// Hadamard rotation of rows of 129 .. 8192 elements ('h' dtypes: weights and
// activations of real widths; rows of 128 have kernels of their own), alone or
// fused with the quantizer behind it and the decoder before it.
//
//   rotate    (WHT(pad(x[r]) * signs) / sqrt(n))[:d]   mxtorch.py:2866-2889
//   unrotate  (WHT(pad(x[r])) / sqrt(n) * signs)[:d]   mxtorch.py:2891-2904
//
// n = next_pow2(d); butterflies of half-width n/2, n/4, ..., 1 in that order
// (mxtorch.py:2811-2832), so every value is the reference's bit for bit.
//
// n / 16 threads hold a row, 16 values each in registers, and take four levels
// at a time: first the top four bits of the index in registers, then through
// LDS the next four, then through LDS the rest.  A row crosses LDS twice where
// one level per pass crossed it up to 12 times with a barrier each: at
// 4096 x 4096 bf16 the rotation and the quantizer behind it took 64.5 + 12.0
// us, the decoder and the unrotation 15.4 + 68.7 us (the rotated copy in fp32
// between them); one kernel each here: 20.1 and 21.9 us, against 8 and 15
// us for the bytes alone.  VALU bounds both: 40 and 42 instructions per
// element, which at 4 cycles a wave fill the SIMDs' time.
//
// LDS place of element i: i + 4 (i / 16) + 16 (i / 256): the strided reads of
// a pass (lanes 2^k apart) and the 16-byte reads of the last one meet
// different banks.
#include "mxk_internal.h"

#include <algorithm>
#include <cmath>

namespace mxk {

namespace {

constexpr int ROT_E = 16;

// (rot_at(base + step e) = rot_at(base) + rot_at(step e) for every pair of
// base and step below: with n known to the compiler the second is an offset
// in the instruction)
__host__ __device__ __forceinline__ constexpr int rot_at(int i) { return i + 4 * (i >> 4) + 16 * (i >> 8); }

// levels of half-width 8, 4, 2, 1 among the 16 registers, those below `lim` only
template <bool ALL = true>
__device__ __forceinline__ void rot_levels(float (&v)[ROT_E], int lim = 16) {
#pragma unroll
  for (int s = 8; s >= 1; s >>= 1) {
    if (!ALL && s >= lim) continue;
#pragma unroll
    for (int e = 0; e < ROT_E; ++e)
      if (!(e & s)) {
        const float u = v[e], w = v[e + s];
        v[e] = u + w;
        v[e + s] = u - w;
      }
  }
}

// one level between lanes `o` holds the partner's values of; `low`: this lane holds the sum
__device__ __forceinline__ float rot_cross(float v, float o, bool low) { return low ? v + o : o - v; }

// From v[e] = element t + e n/16 to the transform, with v[] = elements 16 t +
// e (QUADS false) or 4 t + n/4 (e / 4) + e % 4 (QUADS true: the 16-byte stores
// of a wave then cover whole lines).  `slot`: the row's LDS.  All threads of
// the workgroup call it together.
template <bool QUADS>
__device__ __forceinline__ void rot_row(float (&v)[ROT_E], float* __restrict__ slot, int t, int logn) {
  const int T = 1 << (logn - 4);
  rot_levels(v);
#pragma unroll
  for (int e = 0; e < ROT_E; ++e) slot[rot_at(t) + rot_at(T * e)] = v[e];
  __syncthreads();
  if (logn > 8) {
    const int S = 1 << (logn - 8);
    const int base = (t & (S - 1)) + T * (t >> (logn - 8));
#pragma unroll
    for (int e = 0; e < ROT_E; ++e) v[e] = slot[rot_at(base) + rot_at(S * e)];
    rot_levels(v);
#pragma unroll
    for (int e = 0; e < ROT_E; ++e) slot[rot_at(base) + rot_at(S * e)] = v[e];
    __syncthreads();
  }
  const int left = logn > 8 ? logn - 8 : 4;  // levels 2^(left - 1) .. 1 are left
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const f32x4v w = *reinterpret_cast<const f32x4v*>(slot + (QUADS ? rot_at(4 * t) + rot_at(4 * T * q) : rot_at(16 * t) + 4 * q));
#pragma unroll
    for (int c = 0; c < 4; ++c) v[4 * q + c] = w[c];
  }
  if constexpr (QUADS) {
    if (left > 4) {  // half-width 16: lanes 4 apart
#pragma unroll
      for (int e = 0; e < ROT_E; ++e)
        v[e] = rot_cross(v[e], __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v[e]), 0x101F)), !(t & 4));
    }
    if (left > 3) {
#pragma unroll
      for (int e = 0; e < ROT_E; ++e)
        v[e] = rot_cross(v[e], __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v[e]), 0x4E, 0xF, 0xF, true)),
                         !(t & 2));
    }
    if (left > 2) {
#pragma unroll
      for (int e = 0; e < ROT_E; ++e)
        v[e] = rot_cross(v[e], __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v[e]), 0xB1, 0xF, 0xF, true)),
                         !(t & 1));
    }
    if (left > 1) {
#pragma unroll
      for (int e = 0; e < ROT_E; ++e)
        if (!(e & 2)) {
          const float u = v[e], w = v[e + 2];
          v[e] = u + w;
          v[e + 2] = u - w;
        }
    }
#pragma unroll
    for (int e = 0; e < ROT_E; e += 2) {
      const float u = v[e], w = v[e + 1];
      v[e] = u + w;
      v[e + 1] = u - w;
    }
  } else {
    if (left > 4) {  // half-width 16: the next lane
#pragma unroll
      for (int e = 0; e < ROT_E; ++e)
        v[e] = rot_cross(v[e], __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v[e]), 0xB1, 0xF, 0xF, true)),
                         !(t & 1));
    }
    rot_levels<false>(v, 1 << left);
  }
}

// Elements t + n/16 e of row rl of the workgroup's step of `take` rows from r0
// on (zeros past d and past the rows; x of any input type), as bounds-checked
// buffer loads: a branch per element around plain loads waited on each of them
// (4096 x 4096 bf16 to int4: 36.8 -> 20.1 us).
struct RotX {
  const void* x;
  int type;
};
constexpr uint32_t ROT_OOB = 0x80000000u;
__device__ __forceinline__ void rot_load(float (&v)[ROT_E], const RotX& X, int64_t r0, int take, int rl, int t, int T16,
                                         int d) {
  const int esz = X.type == MXK_IN_F32 ? 4 : 2;
  const __amdgpu_buffer_rsrc_t rs =
      make_rsrc((const uint8_t*)X.x + r0 * d * esz, take > 0 ? (uint32_t)(take * d * esz) : 0u);
#pragma unroll
  for (int e = 0; e < ROT_E; ++e) {
    const int i = t + T16 * e;
    const uint32_t off = i < d ? (uint32_t)((rl * d + i) * esz) : ROT_OOB;
    if (X.type == MXK_IN_F32) {
      v[e] = __uint_as_float(buf_load_b32(rs, off, 0u));
    } else {
      const uint16_t h = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, (int)off, 0, 0);
      v[e] = __uint_as_float(h);  // converted where it is used
    }
  }
}
// the loaded elements as floats
__device__ __forceinline__ void rot_cvt(float (&v)[ROT_E], int type) {
  if (type == MXK_IN_F32) return;
#pragma unroll
  for (int e = 0; e < ROT_E; ++e) {
    const uint16_t h = (uint16_t)__float_as_uint(v[e]);
    v[e] = type == MXK_IN_F16 ? (float)__builtin_bit_cast(_Float16, h) : __uint_as_float((uint32_t)h << 16);
  }
}

// A workgroup's rows: blockDim / (n/16) of them side by side, in steps of the grid
struct RotRows {
  int64_t rows, d;
  int logn;
  float rdiv, rinv;
};

// rotated (FWD) or unrotated rows to fp32; in and out may be the same buffer
template <int LOGN, bool FWD>
__global__ __launch_bounds__(512) void k_rot_rows(RotX in, float* out, RotRows R, const float* __restrict__ signs,
                                                  int vec) {
  extern __shared__ __attribute__((aligned(16))) float sh[];
  const int logn = LOGN ? LOGN : R.logn;
  const int n = 1 << logn, T16 = n >> 4, d = (int)R.d;
  const int t = threadIdx.x & (T16 - 1), rl = threadIdx.x >> (logn - 4), rpw = blockDim.x >> (logn - 4);
  const int64_t step = (int64_t)gridDim.x * rpw;
  float* slot = sh + rl * rot_at(n);
  uint32_t neg = 0u;  // bit e: the sign of input (FWD) or output element e is negative
#pragma unroll
  for (int e = 0; e < ROT_E; ++e)
    neg |= (signs[FWD ? t + T16 * e : 4 * t + 4 * T16 * (e >> 2) + (e & 3)] < 0.0f ? 1u : 0u) << e;
  float vn[ROT_E];
  auto fetch = [&](int64_t r0) { rot_load(vn, in, r0, (int)min((int64_t)rpw, R.rows - r0), rl, t, T16, d); };
  fetch((int64_t)blockIdx.x * rpw);
  for (int64_t r0 = (int64_t)blockIdx.x * rpw; r0 < R.rows; r0 += step) {
    const int64_t r = r0 + rl;
    const bool live = r < R.rows;
    rot_cvt(vn, in.type);
    float v[ROT_E];
#pragma unroll
    for (int e = 0; e < ROT_E; ++e) v[e] = FWD ? __uint_as_float(__float_as_uint(vn[e]) ^ ((neg >> e) << 31)) : vn[e];
    if (r0 + step < R.rows) fetch(r0 + step);
    __syncthreads();  // the slot's last readers
    rot_row<true>(v, slot, t, logn);
    div_rn_all<ROT_E>(v, R.rdiv, R.rinv);
    if (live) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = 4 * t + 4 * T16 * q;
        if (i >= d) continue;
        f32x4v w;
#pragma unroll
        for (int c = 0; c < 4; ++c)
          w[c] = FWD ? v[4 * q + c] : __uint_as_float(__float_as_uint(v[4 * q + c]) ^ ((neg >> (4 * q + c)) << 31));
        if (vec) {
          *reinterpret_cast<f32x4v*>(out + r * d + i) = w;
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (i + c < d) out[r * d + i + c] = w[c];
        }
      }
    }
  }
}

// quantize of rotated rows, blocks of 128, d a multiple of 128: 8 threads hold
// a block, 16 consecutive values each, as in k_quant_had128
template <int LOGN, int MODE, int BITS>
__global__ __launch_bounds__(512) void k_rot_quant(RotX x, RotRows R, const float* __restrict__ signs,
                                                   uint8_t* __restrict__ packed, float* __restrict__ scales, float qf) {
  constexpr int NW = (ROT_E * BITS + 31) / 32, NB = ROT_E * BITS / 8;
  constexpr uint32_t MASK = (1u << BITS) - 1u;
  constexpr bool VOTE = MODE == Q_INT1 || MODE == Q_FP;  // the modes whose codes read a tiny quotient's bits
  extern __shared__ __attribute__((aligned(16))) float sh[];
  __shared__ int2 sK[fp_keys_n<MODE, BITS>()];
  const float* sP = fp_mids<MODE == Q_FP ? BITS : 4>();  // read only by the non-finite path
  const int logn = LOGN ? LOGN : R.logn;
  const int n = 1 << logn, T16 = n >> 4, d = (int)R.d;
  const int t = threadIdx.x & (T16 - 1), rl = threadIdx.x >> (logn - 4), rpw = blockDim.x >> (logn - 4);
  const int64_t step = (int64_t)gridDim.x * rpw;
  float* slot = sh + rl * rot_at(n);
  if constexpr (MODE == Q_FP) load_fp_keys<BITS>(sK);
  uint32_t neg = 0u;  // bit e: the sign of this thread's element e is negative
#pragma unroll
  for (int e = 0; e < ROT_E; ++e) neg |= (signs[t + T16 * e] < 0.0f ? 1u : 0u) << e;
  float vn[ROT_E];
  auto fetch = [&](int64_t r0) { rot_load(vn, x, r0, (int)min((int64_t)rpw, R.rows - r0), rl, t, T16, d); };
  fetch((int64_t)blockIdx.x * rpw);
  for (int64_t r0 = (int64_t)blockIdx.x * rpw; r0 < R.rows; r0 += step) {
    const int64_t r = r0 + rl;
    const bool live = r < R.rows;
    rot_cvt(vn, x.type);
    float v[ROT_E];
#pragma unroll
    for (int e = 0; e < ROT_E; ++e) v[e] = __uint_as_float(__float_as_uint(vn[e]) ^ ((neg >> e) << 31));
    if (r0 + step < R.rows) fetch(r0 + step);
    __syncthreads();  // the slot's last readers (and the key table)
    rot_row<false>(v, slot, t, logn);
    uint32_t mxb = 0u, mnb = 0xFFFFFFFFu;
#pragma unroll
    for (int e = 0; e < ROT_E; ++e) {
      mxb = max(mxb, mag_bits(v[e]));
      if constexpr (VOTE) mnb = min(mnb, (__float_as_uint(v[e]) << 1) - 1u);
    }
    const float gmx = __uint_as_float(group_max_u<8>(mxb));
    float am;
    if (VOTE && __builtin_expect(__ballot(mnb < 2u * 0x0F800000u - 1u) != 0ull, 0)) {
#pragma unroll
      for (int e = 0; e < ROT_E; ++e) v[e] = v[e] / R.rdiv;
      am = gmx / R.rdiv;
    } else {
#pragma unroll
      for (int e = 0; e < ROT_E; ++e) {
        const float q0 = v[e] * R.rinv;
        v[e] = __builtin_fmaf(__builtin_fmaf(-q0, R.rdiv, v[e]), R.rinv, q0);
      }
      am = finite_scale(gmx) ? div_rn(gmx, R.rdiv, R.rinv) : gmx;
    }
    const BlockParams bp = block_params<MODE>(amax_clamped(mag_bits(am)), qf);
    uint32_t w[NW];
#pragma unroll
    for (int k = 0; k < NW; ++k) w[k] = 0u;
    if (__builtin_expect(MODE != Q_INT1 && !finite_scale(bp.s), 0)) {
#pragma unroll
      for (int e = 0; e < ROT_E; ++e)
        w[(e * BITS) >> 5] |= ((uint32_t)encode_nonfinite<MODE, BITS>(v[e], bp, qf, sP) & MASK) << ((e * BITS) & 31);
    } else {
#pragma unroll
      for (int e = 0; e < ROT_E; ++e)
        w[(e * BITS) >> 5] |= ((uint32_t)encode_keyed<MODE, BITS>(v[e], bp, qf, sP, sK) & MASK) << ((e * BITS) & 31);
    }
    const int i = 16 * t;
    if (live && i < d) {
      const int64_t at = r * d + i;
      store_bytes<NB>(packed, at * BITS / 8, R.rows * d * BITS / 8, w);
      if ((t & 7) == 0) scales[at >> 7] = bp.s;
    }
  }
}

// unrotated rows of packed codes, blocks of 128, d a multiple of 128
template <int LOGN, int MODE, int BITS>
__global__ __launch_bounds__(512) void k_rot_dequant(const uint8_t* __restrict__ packed, const float* __restrict__ scales,
                                                     RotRows R, const float* __restrict__ signs,
                                                     float* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) float sh[];
  __shared__ float sG[MODE == Q_FP && BITS == 4 ? 16 : 1];
  if constexpr (MODE == Q_FP && BITS == 4) load_fp_grid<BITS>(sG);
  const int logn = LOGN ? LOGN : R.logn;
  const int n = 1 << logn, T16 = n >> 4, d = (int)R.d;
  const int t = threadIdx.x & (T16 - 1), rl = threadIdx.x >> (logn - 4), rpw = blockDim.x >> (logn - 4);
  const int64_t step = (int64_t)gridDim.x * rpw;
  float* slot = sh + rl * rot_at(n);
  uint32_t neg = 0u;  // bit 4q + c: the sign of output element 4 t + n/4 q + c is negative
#pragma unroll
  for (int e = 0; e < ROT_E; ++e) neg |= (signs[4 * t + 4 * T16 * (e >> 2) + (e & 3)] < 0.0f ? 1u : 0u) << e;
  uint32_t c[ROT_E];
  float s[ROT_E];
  // the step's codes (d a multiple of 128: its rows start on bytes) and scales
  auto load = [&](int64_t r0) {
    const int take = (int)min((int64_t)rpw, R.rows - r0);
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(packed + r0 * d / 8 * BITS, (uint32_t)(take * d / 8 * BITS));
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(scales + r0 * d / 128, (uint32_t)(take * d / 32));
#pragma unroll
    for (int e = 0; e < ROT_E; ++e) {
      const int i = t + T16 * e, at = rl * d + i;
      c[e] = (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(rc, i < d ? (int)((uint32_t)(at * BITS) >> 3) : (int)ROT_OOB, 0, 0);
      s[e] = __uint_as_float(buf_load_b32(rs, i < d ? (uint32_t)(at >> 7) * 4u : ROT_OOB, 0u));
    }
  };
  load((int64_t)blockIdx.x * rpw);
  for (int64_t r0 = (int64_t)blockIdx.x * rpw; r0 < R.rows; r0 += step) {
    const int64_t r = r0 + rl;
    const bool live = r < R.rows;
    __syncthreads();  // the slot's last readers (and the grid)
    float v[ROT_E];
#pragma unroll
    for (int e = 0; e < ROT_E; ++e) {
      const int i = t + T16 * e;  // (d is a multiple of 128: the place in its byte depends on i alone)
      v[e] = (live && i < d) ? decode_field<MODE, BITS>(c[e] >> ((i * BITS) & 7), 0, s[e], sG) : 0.0f;
    }
    if (r0 + step < R.rows) load(r0 + step);
    rot_row<true>(v, slot, t, logn);
    div_rn_all<ROT_E>(v, R.rdiv, R.rinv);
    if (live) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = 4 * t + 4 * T16 * q;
        if (i >= d) continue;
        f32x4v w;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          w[k] = __uint_as_float(__float_as_uint(v[4 * q + k]) ^ ((neg >> (4 * q + k)) << 31));
        __builtin_nontemporal_store(w, reinterpret_cast<f32x4v*>(out + r * d + i));
      }
    }
  }
}

// threads, LDS bytes and workgroups (a row's slot is n + n/4 + n/16 floats)
struct RotLaunch {
  RotRows R;
  dim3 grid, block;
  size_t lds;
};

RotLaunch rot_launch(int64_t rows, int64_t d) {
  RotLaunch p;
  const int64_t n = next_pow2(d);
  int logn = 0;
  while ((int64_t(1) << logn) < n) ++logn;
  const int threads = (int)std::max<int64_t>(256, n / 16);
  const int rpw = (int)(threads / (n / 16));
  p.R = RotRows{rows, d, logn, (float)std::sqrt((double)n), 0.0f};
  p.R.rinv = 1.0f / p.R.rdiv;
  p.block = dim3(threads);
  p.grid = dim3((unsigned)std::min<int64_t>(ceil_div(rows, rpw), (int64_t)num_cus() * 16));
  p.lds = (size_t)rpw * rot_at((int)n) * sizeof(float);
  return p;
}

// n of 1024 .. 8192 known to the compiler (LDS places in the instructions: 134
// -> 70 VGPRs), shorter rows by the general form
#define ROT_LOGN(K, ...)                                                                     \
  switch (p.R.logn) {                                                                        \
    case 10: hipLaunchKernelGGL((K<10, __VA_ARGS__>), p.grid, p.block, p.lds, st, ROT_ARGS); break; \
    case 11: hipLaunchKernelGGL((K<11, __VA_ARGS__>), p.grid, p.block, p.lds, st, ROT_ARGS); break; \
    case 12: hipLaunchKernelGGL((K<12, __VA_ARGS__>), p.grid, p.block, p.lds, st, ROT_ARGS); break; \
    case 13: hipLaunchKernelGGL((K<13, __VA_ARGS__>), p.grid, p.block, p.lds, st, ROT_ARGS); break; \
    default: hipLaunchKernelGGL((K<0, __VA_ARGS__>), p.grid, p.block, p.lds, st, ROT_ARGS);  \
  }

}  // namespace

bool rot_fits(int64_t d) { return d > 128 && next_pow2(d) <= 8192; }

int rot_rows(const void* in, int x_type, bool fwd, float* out, int64_t rows, int64_t d, const float* signs,
             hipStream_t st) {
  const RotLaunch p = rot_launch(rows, d);
  const int vec = aligned16(out) && d % 4 == 0;
  const RotX X{in, fwd ? x_type : MXK_IN_F32};
#define ROT_ARGS X, out, p.R, signs, vec
  if (fwd) {
    ROT_LOGN(k_rot_rows, true)
  } else {
    ROT_LOGN(k_rot_rows, false)
  }
#undef ROT_ARGS
  return check_launch("rotate");
}

int rot_quantize(const void* x, int x_type, int64_t n, int64_t d, int mode, int bits, int block, const float* signs,
                 uint8_t* packed, float* scales, int64_t n_store, float qf, hipStream_t st) {
  if (!rot_fits(d) || block != 128 || d % 128 != 0 || n_store != n || !aligned16(packed)) return MXK_EUNSUPPORTED;
  const RotLaunch p = rot_launch(n / d, d);
  const RotX X{x, x_type};
#define ROT_ARGS X, p.R, signs, packed, scales, qf
#define MXK_ROT_Q(MODE, BITS)                    \
  if (mode == MODE && bits == BITS) {            \
    ROT_LOGN(k_rot_quant, MODE, BITS)            \
    return check_launch("quantize(rotated)");    \
  }
  MXK_ROT_Q(Q_INT1, 1)
  MXK_ROT_Q(Q_INT, 2)
  MXK_ROT_Q(Q_INT, 4)
  MXK_ROT_Q(Q_INT, 8)
  MXK_ROT_Q(Q_FP, 4)
  MXK_ROT_Q(Q_FP, 8)
#undef MXK_ROT_Q
#undef ROT_ARGS
  return MXK_EUNSUPPORTED;
}

int rot_dequantize(const uint8_t* packed, int64_t packed_nbytes, const float* scales, int64_t nb, int64_t n, int64_t d,
                   int mode, int bits, int block, const float* signs, float* out, hipStream_t st) {
  if (!rot_fits(d) || block != 128 || d % 128 != 0 || n % d != 0 || nb != n / 128 || !aligned16(out) ||
      packed_nbytes < n / 8 * bits)
    return MXK_EUNSUPPORTED;
  const RotLaunch p = rot_launch(n / d, d);
#define ROT_ARGS packed, scales, p.R, signs, out
#define MXK_ROT_D(MODE, BITS)                    \
  if (mode == MODE && bits == BITS) {            \
    ROT_LOGN(k_rot_dequant, MODE, BITS)          \
    return check_launch("dequantize(rotated)");  \
  }
  MXK_ROT_D(Q_INT1, 1)
  MXK_ROT_D(Q_INT, 2)
  MXK_ROT_D(Q_INT, 4)
  MXK_ROT_D(Q_INT, 8)
  MXK_ROT_D(Q_FP, 4)
  MXK_ROT_D(Q_FP, 8)
#undef MXK_ROT_D
#undef ROT_ARGS
  return MXK_EUNSUPPORTED;
}

}  // namespace mxk

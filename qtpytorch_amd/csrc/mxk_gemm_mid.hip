// Packed block-scaled GEMM of middle sizes for gfx950 (mxk_gemm.hip states the
// arithmetic): int8 or int4 operands as stored, blocks of 128 or 64, any M, K
// and N.  It runs the shapes that the 256x128 loop does not take: grids below
// one such tile per CU, blocks of 64, rows that do not start on 16 bytes.  BT
// is the linear's form: [N][K] weights (B goes to LDS like A), scales by two
// strides, and K in gridDim.y parts where the tiles alone leave CUs idle.
//
// A workgroup owns a 128x128 tile (8 waves of 32x64) or a 64x64 tile (4 waves
// of 32x32).  A stage is 128 codes of K: one block of 128 or two of 64.  Its
// operands come as whole aligned dwords into registers one stage ahead, rows
// that start inside a dword are brought together with v_alignbit (SHIFT), and
// go to LDS as int8 bytes: A's rows K-contiguous, B's rows as stored, read
// back transposed (ds_read_b64_tr_b8).  int4 codes c become bytes 16 c (two
// instructions per eight codes), with K permuted alike in A and in the rows B
// is read in, and the products carry a factor 256.  The scales of a stage go
// through LDS with it, straight from the stored arrays.  No pass before the
// product; with REQ (128-tiles, N a multiple of the block) none after it
// either: the requantization of C runs in the epilogue.
//
// What bounds it: VALU (4 per output and block, 5 for int4, as C's bits need
// them; 62% of the SIMDs' time at 2048^3 in blocks of 64, 57% at int4 1500 x 2048 x
// 1800), LDS reads and MFMA (11%) one after the other in each wave; several
// workgroups per CU (64-tiles) or a barrier every other stage (128-tiles: 2048^3
// in blocks of 64 39.1 -> 34.3 us) let waves overlap them.  2048^3: 70.8 -> 28.9
// us; the sizes and the rule between the kernels stand at plan_mid.
#include "mxk_internal.h"

#include <algorithm>

namespace mxk {

namespace {

typedef int32_t i4v __attribute__((ext_vector_type(4)));
typedef int32_t i2v __attribute__((ext_vector_type(2)));

struct MidArgs {
  const uint8_t* A;  // [M][K] codes
  const uint8_t* B;  // [K][N] codes, or (BT) [N][K]
  const float* sa;   // of row m, block kb: sa[m * sa_m + kb * sa_k], or (BT) that index >> sa_sh
  const float* sb;   // of column n: sb[kb * N + n], or (BT) sb[(n * sb_n + kb * sb_k) >> sb_sh]
  float* C;          // fp32 C, or null
  int32_t* acc;      // [KB][M][N] integer products, or null
  uint8_t* cq;       // REQ: packed codes and scales of C
  float* cq_scales;
  const float* bias; // added to C when written (or null)
  int64_t sa_m, sa_k, sb_n, sb_k;
  uint32_t a_bytes, b_bytes, sa_bytes, sb_bytes;
  int M, K, N, KB, a_ok, b_ok, tiles_n, tiles;
  int sa_sh, sb_sh;
  int per;           // (BT) stages per K split: split z of gridDim.y writes C + z * M * N
};

constexpr uint32_t MID_OOB = 0x80000000u;

// 16-byte slot of chunk c in A row r (128 bytes) and in B row r (16 TN / 16
// bytes): the rows that one read touches spread over the banks
__device__ __forceinline__ int mid_aslot(int r, int c) { return c ^ ((r >> 1) & 7); }
template <int TN>
__device__ __forceinline__ int mid_bslot(int r, int c) {
  return TN == 128 ? c ^ (((r >> 1) & 3) | ((r >> 2) & 4)) : c ^ ((r >> 1) & 3);
}
// column (and K row) at place l of an unpacked group of 8 int4 codes: 0,2,4,6,1,3,5,7
template <int BITS>
__device__ __forceinline__ int mid_perm(int l) {
  return BITS == 4 ? ((l & 8) | ((l & 3) << 1) | ((l >> 2) & 1)) : l;
}

// 16 bytes of codes as loaded: with SHIFT one dword more
template <bool SHIFT>
struct MidRaw {
  u32x4 v;
  uint32_t e;
};

// the 16 bytes at code index f
template <int BITS, bool SHIFT>
__device__ __forceinline__ void mid_load(MidRaw<SHIFT>& r, __amdgpu_buffer_rsrc_t rs, uint32_t f, bool ok) {
  const uint32_t off = ok ? (BITS == 8 ? f & ~3u : (f >> 3) * 4u) : MID_OOB;
  r.v = buf_load_b128(rs, off, 0u);
  if constexpr (SHIFT) r.e = buf_load_b32(rs, off + 16u, 0u);
}
template <int BITS, bool SHIFT>
__device__ __forceinline__ u32x4 mid_take(const MidRaw<SHIFT>& r, uint32_t f) {
  if constexpr (!SHIFT) return r.v;
  const uint32_t sh = BITS == 8 ? (f & 3u) * 8u : (f & 7u) * 4u;
  return u32x4{__builtin_amdgcn_alignbit(r.v[1], r.v[0], sh), __builtin_amdgcn_alignbit(r.v[2], r.v[1], sh),
               __builtin_amdgcn_alignbit(r.v[3], r.v[2], sh), __builtin_amdgcn_alignbit(r.e, r.v[3], sh)};
}
__device__ __forceinline__ u32x4 mid_unpack16(uint32_t w0, uint32_t w1) {
  return u32x4{(w0 << 4) & 0xF0F0F0F0u, w0 & 0xF0F0F0F0u, (w1 << 4) & 0xF0F0F0F0u, w1 & 0xF0F0F0F0u};
}

template <int BITS, int BLK, int TM, bool SHIFT, bool BT, int REQ, bool ACC>
__global__ __launch_bounds__(TM * 4, TM == 128 ? 2 : 3) void k_qgemm_mid(MidArgs g) {
  constexpr int TN = TM, THREADS = TM * 4, H = 128 / BLK;
  constexpr int WN = 2, CT = TN / (16 * WN), RT = 2;
  constexpr int Q = BITS == 8 ? 2 : 1;          // 16-byte pieces of A (and of B) per thread and stage
  constexpr int APR = BITS == 8 ? 8 : 4;        // pieces per A row (128 codes)
  constexpr int BPR = BT ? APR : TN * BITS / 128;  // pieces per B row
  static_assert(REQ == 0 || TM == 128, "a block of C inside one tile");
  constexpr int STAGE = TM * 128;  // bytes of an operand's stage (TN = TM)
  constexpr int SC = H * (TM + TN);
  // 128-tiles (one workgroup per CU): four stages in LDS and a barrier every
  // other one, so that the waves of a SIMD drift apart; 64-tiles: two
  constexpr int NBUF = TM == 128 ? 4 : 2;
  constexpr int LDS_BYTES = NBUF * (2 * STAGE + SC * 4);
  static_assert(REQ == 0 || 2048 + TM * TN * REQ / 8 <= LDS_BYTES, "requantized tile");
  __shared__ __attribute__((aligned(16))) uint8_t lds[LDS_BYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int lr = lane & 15, lg = lane >> 4;
  // an XCD (workgroup b % 8) takes consecutive tiles, row of tiles by row
  const int per = (g.tiles + 7) / 8;
  const int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (tile >= g.tiles) return;
  const int m0 = (tile / g.tiles_n) * TM, n0 = (tile % g.tiles_n) * TN;
  const __amdgpu_buffer_rsrc_t rA = make_rsrc(g.A, g.a_bytes), rB = make_rsrc(g.B, g.b_bytes);
  const __amdgpu_buffer_rsrc_t rSA = make_rsrc(g.sa, g.sa_bytes), rSB = make_rsrc(g.sb, g.sb_bytes);

  const int st0 = BT ? (int)blockIdx.y * g.per : 0;
  const int stages = BT ? std::min((g.K + 127) / 128, st0 + g.per) : (g.K + 127) / 128;
  // this thread's pieces: code index at stage 0, and what a stage adds
  uint32_t fa[Q], fb[Q];
  bool oka[Q], okb[Q];
  int kb_row[Q];  // (B as stored) K row of the piece
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int idx = tid + THREADS * q;
    const int ra = idx / APR, pa = idx % APR;
    fa[q] = (uint32_t)(m0 + ra) * (uint32_t)g.K + (uint32_t)(pa * (128 / APR));
    oka[q] = m0 + ra < g.M;
    const int rb = idx / BPR, pb = idx % BPR;
    if constexpr (BT) {
      fb[q] = (uint32_t)(n0 + rb) * (uint32_t)g.K + (uint32_t)(pb * (128 / APR));
      okb[q] = n0 + rb < g.N;
      kb_row[q] = 0;
    } else {
      fb[q] = (uint32_t)rb * (uint32_t)g.N + (uint32_t)(n0 + pb * (128 / BITS));
      okb[q] = n0 + pb * (128 / BITS) < g.N;
      kb_row[q] = rb;
    }
  }
  const uint32_t bstep = BT ? 128u : 128u * (uint32_t)g.N;
  // this thread's scale of a stage: half h, A row or B column `sx`
  const int sh_h = tid / (TM + TN), sx = tid % (TM + TN);
  const bool s_on = tid < SC, s_a = sx < TM;
  const bool s_ok = s_on && (s_a ? m0 + sx < g.M : n0 + sx - TM < g.N);
  const bool s_one = s_a ? !g.a_ok : !g.b_ok;

  struct Set {  // a stage's pieces and scale on their way to LDS
    MidRaw<SHIFT> a[Q], b[Q];
    float s;
  };
  auto load = [&](Set& S, int st) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      // A codes past K meet zero rows of B (BT: B's are cut below)
      mid_load<BITS, SHIFT>(S.a[q], rA, fa[q] + 128u * st, oka[q] && st < stages);
      mid_load<BITS, SHIFT>(S.b[q], rB, fb[q] + bstep * st, okb[q] && (BT ? st < stages : kb_row[q] + 128 * st < g.K));
    }
    const int kb = st * H + sh_h;
    const bool ok = s_ok && kb < g.KB && !s_one;
    const int64_t sa_i = (m0 + sx) * g.sa_m + kb * g.sa_k;
    const int64_t sb_i = BT ? (n0 + sx - TM) * g.sb_n + kb * g.sb_k : (int64_t)kb * g.N + n0 + sx - TM;
    const uint32_t off = ok ? (uint32_t)(BT ? (s_a ? sa_i >> g.sa_sh : sb_i >> g.sb_sh) : (s_a ? sa_i : sb_i)) * 4u
                            : MID_OOB;
    // (two loads, one of them past its buffer: the resource is the wave's)
    const uint32_t va = buf_load_b32(rSA, s_a ? off : MID_OOB, 0u), vb = buf_load_b32(rSB, s_a ? MID_OOB : off, 0u);
    S.s = s_ok && kb < g.KB ? (s_one ? 1.0f : __uint_as_float(va | vb)) : 0.0f;
  };
  auto put = [&](const Set& S, int st, int buf) {
    uint8_t* sA = lds + buf * STAGE;
    uint8_t* sB = lds + NBUF * STAGE + buf * STAGE;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int idx = tid + THREADS * q;
      const int arow = idx / APR, pa = idx % APR, brow = idx / BPR, pb = idx % BPR;
      u32x4 a = mid_take<BITS, SHIFT>(S.a[q], fa[q] + 128u * st), b = mid_take<BITS, SHIFT>(S.b[q], fb[q] + bstep * st);
      if constexpr (BT) {
        // past K the next row begins: cut one operand's codes there
        const int left = g.K - 128 * st - pb * (128 / APR);  // codes of this piece before K's end
        if (left < 128 / APR) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int c = left - u * (32 / BITS);
            b[u] = c >= 32 / BITS ? b[u] : c <= 0 ? 0u : b[u] & ((1u << (c * BITS)) - 1u);
          }
        }
      }
      auto bput = [&](int c, u32x4 v) {
        if constexpr (BT) *reinterpret_cast<u32x4*>(sB + brow * 128 + mid_aslot(brow, c) * 16) = v;
        else *reinterpret_cast<u32x4*>(sB + brow * TN + mid_bslot<TN>(brow, c) * 16) = v;
      };
      if constexpr (BITS == 8) {
        *reinterpret_cast<u32x4*>(sA + arow * 128 + mid_aslot(arow, pa) * 16) = a;
        bput(pb, b);
      } else {
        *reinterpret_cast<u32x4*>(sA + arow * 128 + mid_aslot(arow, 2 * pa) * 16) = mid_unpack16(a[0], a[1]);
        *reinterpret_cast<u32x4*>(sA + arow * 128 + mid_aslot(arow, 2 * pa + 1) * 16) = mid_unpack16(a[2], a[3]);
        bput(2 * pb, mid_unpack16(b[0], b[1]));
        bput(2 * pb + 1, mid_unpack16(b[2], b[3]));
      }
    }
    if (s_on) reinterpret_cast<float*>(lds + 2 * NBUF * STAGE)[buf * SC + tid] = S.s;
  };

  float c[RT][CT][4];
#pragma unroll
  for (int a = 0; a < RT; ++a)
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) c[a][t][i] = 0.0f;
  const int lcol = BT ? lr : mid_perm<BITS>(lr);
  // fragment places of this lane in stage buffer 0
  const int kl = 16 * lg + mid_perm<BITS>(lr >> 1);

  // one stage on its way in registers, two in LDS (stages past the last read
  // zeros); a second one in registers measured no faster
  Set S;
  load(S, st0);
  put(S, st0, 0);
  load(S, st0 + 1);
  if constexpr (NBUF > 2) {
    put(S, st0 + 1, 1);
    load(S, st0 + 2);
  }
  __syncthreads();
  for (int st = st0; st < stages; ++st) {
    const int buf = (st - st0) & (NBUF - 1);
    const uint8_t* sA = lds + buf * STAGE;
    const uint8_t* sB = lds + NBUF * STAGE + buf * STAGE;
    const float* sS = reinterpret_cast<const float*>(lds + 2 * NBUF * STAGE) + buf * SC;
    i4v af[RT][2], bf[2][CT];
#pragma unroll
    for (int a = 0; a < RT; ++a)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int r = wm * 32 + a * 16 + lr;
        af[a][h] = *reinterpret_cast<const i4v*>(sA + r * 128 + mid_aslot(r, 4 * h + lg) * 16);
      }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < CT; ++t) {
        if constexpr (BT) {
          const int r = wn * 16 * CT + 16 * t + lr;
          bf[h][t] = *reinterpret_cast<const i4v*>(sB + r * 128 + mid_aslot(r, 4 * h + lg) * 16);
        } else {
          typedef __attribute__((address_space(3))) i2v* tr_ptr;
          const uint8_t* at = sB + (kl + 64 * h) * TN + mid_bslot<TN>(kl, CT * wn + t) * 16 + 8 * (lr & 1);
          const i2v x = __builtin_amdgcn_ds_read_tr8_b64_v2i32((tr_ptr)at);
          const i2v y = __builtin_amdgcn_ds_read_tr8_b64_v2i32((tr_ptr)(at + 8 * TN));
          bf[h][t] = i4v{x[0], x[1], y[0], y[1]};
        }
      }
    // the readers of that buffer passed the last barrier
    constexpr int AHEAD = NBUF / 2;
    put(S, st + AHEAD, (st - st0 + AHEAD) & (NBUF - 1));
    load(S, st + AHEAD + 1);
#pragma unroll
    for (int hb = 0; hb < H; ++hb) {
      const float* sh = sS + hb * (TM + TN);
      float sb[CT];
#pragma unroll
      for (int t = 0; t < CT; ++t) sb[t] = sh[TM + wn * 16 * CT + 16 * t + lcol];
#pragma unroll
      for (int a = 0; a < RT; ++a) {
        const f32x4v sa = *reinterpret_cast<const f32x4v*>(sh + wm * 32 + a * 16 + lg * 4);
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          i4v p = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[a][hb], bf[hb][t], i4v{0, 0, 0, 0}, 0, 0, 0);
          if constexpr (H == 1) p = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[a][1], bf[1][t], p, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int pi = BITS == 4 ? p[i] >> 8 : p[i];
            const float v = ((float)pi * sa[i]) * sb[t];
            c[a][t][i] = c[a][t][i] + v;
          }
          if constexpr (ACC) {
            const int kb = st * H + hb, col = n0 + wn * 16 * CT + 16 * t + lcol;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int row = m0 + wm * 32 + a * 16 + lg * 4 + i;
              if (kb < g.KB && row < g.M && col < g.N)
                g.acc[((int64_t)kb * g.M + row) * g.N + col] = BITS == 4 ? p[i] >> 8 : p[i];
            }
          }
        }
      }
    }
    if (NBUF == 2 || ((st - st0) & 1)) __syncthreads();
  }
  if constexpr (NBUF > 2) __syncthreads();

  if (g.C) {
    float* C = BT ? g.C + (int64_t)blockIdx.y * g.M * g.N : g.C;
#pragma unroll
    for (int a = 0; a < RT; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = m0 + wm * 32 + a * 16 + lg * 4 + i;
        if (row >= g.M) continue;
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          const int col = n0 + wn * 16 * CT + 16 * t + lcol;
          if (col < g.N) C[(int64_t)row * g.N + col] = g.bias ? c[a][t][i] + g.bias[col] : c[a][t][i];
        }
      }
  }
  if constexpr (REQ > 0) {
    // blocks of BLK columns of C: the wave's own 64, or both column halves
    // (the row's maximum meets in LDS); then whole packed rows out of LDS
    constexpr int RB = TN * REQ / 8;
    uint32_t* smax = reinterpret_cast<uint32_t*>(lds);  // [wn][TM]
    uint8_t* tile_q = lds + 2048;
    uint32_t mx[RT][4];
#pragma unroll
    for (int a = 0; a < RT; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint32_t m = 0u;
#pragma unroll
        for (int t = 0; t < CT; ++t) m = max(m, mag_bits(c[a][t][i]));
        mx[a][i] = group_max_u<16>(m);
        if (BLK == 128 && lr == 0) smax[wn * TM + wm * 32 + a * 16 + lg * 4 + i] = mx[a][i];
      }
    if constexpr (BLK == 128) __syncthreads();
    constexpr float qf = (float)((1 << (REQ - 1)) - 1);
#pragma unroll
    for (int a = 0; a < RT; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int rl = wm * 32 + a * 16 + lg * 4 + i;
        const uint32_t m = BLK == 128 ? max(smax[rl], smax[TM + rl]) : mx[a][i];
        const BlockParams bp = block_params<Q_VEC>(amax_clamped(m), qf);
        const bool nf = !finite_scale(bp.s);
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          const int cl = wn * 16 * CT + 16 * t + lcol;
          const int code = nf ? encode_nonfinite<Q_VEC, REQ>(c[a][t][i], bp, qf, nullptr)
                              : encode<Q_VEC, REQ>(c[a][t][i], bp, qf, nullptr);
          if constexpr (REQ == 16) reinterpret_cast<int16_t*>(tile_q + rl * RB)[cl] = (int16_t)code;
          else tile_q[rl * RB + cl] = (uint8_t)code;
        }
        const int64_t row = m0 + rl;
        const int cb = n0 + (BLK == 128 ? 0 : wn * 64);
        if ((BLK == 64 || wn == 0) && lr == 0 && row < g.M && cb < g.N) g.cq_scales[(row * g.N + cb) / BLK] = bp.s;
      }
    __syncthreads();
    for (int idx = tid; idx < TM * RB / 16; idx += THREADS) {
      const int rl = idx / (RB / 16), ch = idx % (RB / 16);
      const int64_t row = m0 + rl;
      if (row < g.M && n0 + ch * (128 / REQ) < g.N)
        *reinterpret_cast<u32x4*>(g.cq + (row * g.N + n0) * REQ / 8 + ch * 16) =
            *reinterpret_cast<const u32x4*>(tile_q + rl * RB + ch * 16);
    }
  }
}

template <int BITS, int BLK, int TM, bool BT, int REQ, bool ACC = false>
void mid_launch_s(const MidArgs& g, bool shift, hipStream_t st) {
  const dim3 grid((unsigned)(8 * ceil_div(g.tiles, 8)));
  // (the integer products are a diagnostic output: one form of it)
  if (shift || ACC) hipLaunchKernelGGL((k_qgemm_mid<BITS, BLK, TM, true, BT, REQ, ACC>), grid, dim3(TM * 4), 0, st, g);
  else hipLaunchKernelGGL((k_qgemm_mid<BITS, BLK, TM, false, BT, REQ, false>), grid, dim3(TM * 4), 0, st, g);
}

template <int BITS, int BLK>
void mid_launch(MidArgs g, int tm, bool req, bool shift, hipStream_t st) {
  if (g.acc) tm = 64;
  g.tiles_n = (int)ceil_div(g.N, tm);
  g.tiles = (int)(ceil_div(g.M, tm) * g.tiles_n);
  if (g.acc) return mid_launch_s<BITS, BLK, 64, false, 0, true>(g, shift, st);
  if (tm == 64) return mid_launch_s<BITS, BLK, 64, false, 0>(g, shift, st);
  if (req) return mid_launch_s<BITS, BLK, 128, false, 2 * BITS>(g, shift, st);
  mid_launch_s<BITS, BLK, 128, false, 0>(g, shift, st);
}

}  // namespace

// Which shapes, and which tile (us, start of the file's kernels | 64-tiles |
// 128-tiles; int8 and int4 codes, blocks of 128 unless said):
//   512^3             6.7 | 8.8 | 11.6     int4 31.5 | 9.0 | 12.1
//   1024^3           15.8 | 14.1 | 16.3         40.8 | 13.9 | 16.3
//   1500x2048x1800   55.2 | 30.9 | 31.4         70.7 | 31.0 | 31.2
//   2048^3           70.8 | 34.9 | 28.9         73.7 | 35.1 | 25.9
//     blocks of 64   77.9 | 41.0 | 34.3        135.5 | 41.1 | 31.8
//   3000x2048x3000   87.6 | 75.4 | 79.9        113.9 | 68.1 | 79.0
//   4096^3 block 64   755 | 255 | 266            853 | 243 | 273
//   4096x4096x4100    212 | 249 | 230            275 | 245 | 270
// So: 128-tiles when they fill most of one round of the CUs, else 64-tiles;
// int8 grids of fewer 64-tiles than half the CUs stay with the 32x32 kernel
// (operands on 16 bytes), and grids of two (int4: three) 256x128 tiles per CU
// and more in blocks of 128 with the 256x128 loop, whose unpacking pass then
// pays.
MidPlan plan_mid(int64_t M, int64_t K, int64_t N, int bits, int block, int out_bits) {
  MidPlan p;
  const int64_t lim = int64_t(1) << 31;
  if ((bits != 4 && bits != 8) || (block != 64 && block != 128)) return p;
  const int64_t KB = ceil_div(K, block);
  if ((M + 128) * (K + 256) >= lim || (K + 256) * (N + 128) >= lim || KB * M * 4 >= lim || KB * (N + 128) * 4 >= lim)
    return p;
  // whole aligned dwords are read
  if ((M * K * bits / 8) % 4 != 0 || (K * N * bits / 8) % 4 != 0 || (M * K * bits) % 8 != 0 || (K * N * bits) % 8 != 0)
    return p;
  const int64_t t128 = ceil_div(M, 128) * ceil_div(N, 128), t64 = ceil_div(M, 64) * ceil_div(N, 64);
  if (bits == 8 && K % block == 0 && N % 16 == 0 && t64 < num_cus() / 2) return p;
  if (block == 128 && ceil_div(M, 256) * ceil_div(N, 128) >= (bits == 8 ? 2 : 3) * (int64_t)num_cus()) return p;
  p.tm = 4 * t128 > 3 * num_cus() && t128 <= num_cus() ? 128 : 64;
  p.req = p.tm == 128 && out_bits == 2 * bits && N % block == 0;
  return p;
}

int run_mid(const MidPlan& p, const void* a, const float* sa, int a_ok, const void* b, const float* sb, int b_ok,
            int64_t M, int64_t K, int64_t N, int bits, int block, bool req, void* cq, float* cq_scales, float* C,
            int32_t* acc, hipStream_t st) {
  MidArgs g;
  const int64_t KB = ceil_div(K, block);
  g.A = (const uint8_t*)a;
  g.B = (const uint8_t*)b;
  g.sa = sa;
  g.sb = sb;
  g.C = C;
  g.acc = acc;
  g.sb_n = g.sb_k = 0;
  g.sa_sh = g.sb_sh = 0;
  g.per = 0;
  g.cq = (uint8_t*)cq;
  g.cq_scales = cq_scales;
  g.bias = nullptr;
  g.sa_m = KB;
  g.sa_k = 1;
  g.a_bytes = (uint32_t)(M * K * bits / 8);
  g.b_bytes = (uint32_t)(K * N * bits / 8);
  g.sa_bytes = a_ok ? (uint32_t)(KB * M * 4) : 0u;
  g.sb_bytes = b_ok ? (uint32_t)(KB * N * 4) : 0u;
  g.M = (int)M;
  g.K = (int)K;
  g.N = (int)N;
  g.KB = (int)KB;
  g.a_ok = a_ok;
  g.b_ok = b_ok;
  const bool shift = (K * bits) % 32 != 0 || (N * bits) % 32 != 0;
  if (bits == 8 && block == 128) mid_launch<8, 128>(g, p.tm, req, shift, st);
  else if (bits == 8) mid_launch<8, 64>(g, p.tm, req, shift, st);
  else if (block == 128) mid_launch<4, 128>(g, p.tm, req, shift, st);
  else mid_launch<4, 64>(g, p.tm, req, shift, st);
  return check_launch("qgemm");
}

// C = the sum of S partial products in order (+ bias)
__global__ __launch_bounds__(256) void k_mid_reduce(const float* __restrict__ part, int S, int64_t n, int64_t N,
                                                    const float* __restrict__ bias, float* __restrict__ C) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    float v = part[i];
    for (int z = 1; z < S; ++z) v += part[z * n + i];
    C[i] = bias ? v + bias[i % N] : v;
  }
}

// One scale per row, or per power of two of the kernel's K blocks (block 128
// on rows of odd multiples of 64: a scale may reach over two rows;
// 9x5056x6968 with x's quantization 243 -> 31 us)
static bool mid_scale_form(int64_t block, int64_t K, int kblk) {
  const int64_t r = block / kblk;
  return block == K || (r & (r - 1)) == 0;
}

// Which int8 x int8 linears (us, scales per token of x and per block of w;
// 128 x 128 kernels and their passes | 64-tiles | 256 x 128 loop):
//   8x512x512          12.1 |  5.8           8x4096x4096        51.0 | 11.0
//   64x4096x4096       53.9 | 14.1           128x8192x1024      96.3 | 15.0
//   512x2048x2048      32.0 | 17.8           1000x4096x4096     60.9 | 53.2
//   300x4160x4000       199 | 34.9  (blocks of 64)
//   2001x4160x4096      393 |  127  (blocks of 64)
//   8x4096x32768          - | 33.6 | 46.5    1100x4096x4096     62.3 |    - | 49.4
//   1500x4096x4096     64.0 | 83.4 | 52.2    3500x4096x2048     64.3 | 81.6 | 55.3
//   int4: 8x4096x4096   134 | 11.2           1000x4096x4096      152 | 53.3
//   int4: 1500x4096x4096 161 | 76.5 | 146   2000x4096x4096      163 | 98.3
// The 64-tiles read scales and codes as they are stored, one launch.  They
// take up to four tiles per CU (int4, which the 256 x 128 loop unpacks first:
// eight) and, in blocks of 64, which that loop does not have, all sizes.  A
// grid of fewer tiles than the CUs hold at once (three each) splits K into
// parts of at least six stages; 8x4096x4096 unsplit 23.1 -> 11.0, in 16 parts
// 13.0; 128x8192x1024 43.5 -> 15.0.
MidLin plan_mid_lin(int64_t M, int64_t K, int64_t N, int bits, int64_t x_block, int64_t w_block, int kblk) {
  MidLin p;
  const int64_t lim = int64_t(1) << 31, KB = K / kblk;
  if ((bits != 4 && bits != 8) || !mid_scale_form(x_block, K, kblk) || !mid_scale_form(w_block, K, kblk)) return p;
  if ((M + 128) * (K + 256) >= lim || (K + 256) * (N + 128) >= lim || KB * (M + 128) * 4 >= lim ||
      KB * (N + 128) * 4 >= lim)
    return p;
  const int64_t stages = ceil_div(K, 128), tiles = ceil_div(M, 64) * ceil_div(N, 64);
  if (kblk == 128 && tiles > (bits == 8 ? 4 : 8) * (int64_t)num_cus()) return p;
  p.taken = true;
  const int64_t S = std::max<int64_t>(1, std::min<int64_t>(3 * num_cus() / tiles, stages / 6));
  p.per = (int)ceil_div(stages, S);
  p.splits = (int)ceil_div(stages, p.per);
  return p;
}

int run_mid_lin(const MidLin& p, const void* x, const float* sx, int64_t x_block, const void* w, const float* sw,
                int64_t w_block, int64_t M, int64_t K, int64_t N, int bits, int kblk, const float* bias, float* out,
                float* part, hipStream_t st) {
  const int64_t KB = K / kblk;
  MidArgs g{};
  const bool split = p.splits > 1 && part;
  g.A = (const uint8_t*)x;
  g.B = (const uint8_t*)w;
  g.sa = sx;
  g.sb = sw;
  g.C = split ? part : out;
  g.bias = split ? nullptr : bias;
  g.sa_m = x_block == K ? 1 : KB;
  g.sa_k = x_block == K ? 0 : 1;
  g.sb_n = w_block == K ? 1 : KB;
  g.sb_k = w_block == K ? 0 : 1;
  g.sa_sh = x_block == K ? 0 : __builtin_ctzll((uint64_t)(x_block / kblk));
  g.sb_sh = w_block == K ? 0 : __builtin_ctzll((uint64_t)(w_block / kblk));
  g.a_bytes = (uint32_t)(M * K * bits / 8);
  g.b_bytes = (uint32_t)(K * N * bits / 8);
  g.sa_bytes = (uint32_t)(ceil_div(M * K, x_block) * 4);
  g.sb_bytes = (uint32_t)(ceil_div(N * K, w_block) * 4);
  g.M = (int)M;
  g.K = (int)K;
  g.N = (int)N;
  g.KB = (int)KB;
  g.a_ok = g.b_ok = 1;
  g.tiles_n = (int)ceil_div(N, 64);
  g.tiles = (int)(ceil_div(M, 64) * g.tiles_n);
  g.per = split ? p.per : (int)ceil_div(K, 128);
  const dim3 grid((unsigned)(8 * ceil_div(g.tiles, 8)), split ? (unsigned)p.splits : 1u), wg(256);
  if (bits == 8 && kblk == 128)
    hipLaunchKernelGGL((k_qgemm_mid<8, 128, 64, false, true, 0, false>), grid, wg, 0, st, g);
  else if (bits == 8)
    hipLaunchKernelGGL((k_qgemm_mid<8, 64, 64, false, true, 0, false>), grid, wg, 0, st, g);
  else if (kblk == 128)
    hipLaunchKernelGGL((k_qgemm_mid<4, 128, 64, false, true, 0, false>), grid, wg, 0, st, g);
  else
    hipLaunchKernelGGL((k_qgemm_mid<4, 64, 64, false, true, 0, false>), grid, wg, 0, st, g);
  if (split)
    hipLaunchKernelGGL(k_mid_reduce, dim3((unsigned)std::min<int64_t>(ceil_div(M * N, 256), 8 * num_cus())), dim3(256),
                       0, st, part, p.splits, M * N, N, bias, out);
  return check_launch("linear_i8");
}

}  // namespace mxk

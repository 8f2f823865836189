// Attention of many query rows over the FP32 KV cache (QK_SHADER,
// SOFTMAX_SHADER and ATTN_OUT_SHADER, gpu-runtime.js:1204-1248) on the 16-bit
// matrix cores.
//
// Numerics.  The 16-bit matrix forms run at 16 times the FP32 form's rate, so
// q, k, v and p are taken as three BF16 parts each (exact: 3 x 8 bits of FP32's
// 24, and FP32's exponents), six v_mfma_f32_16x16x32_bf16 per product, the sums
// in FP32.  What is dropped is below 2^-26 of each product by itself, so a small
// value keeps its bits beside any large one (below 2^-110 the last parts leave
// BF16's range).  Two FP16 parts under shared
// exponents were less: for the scores 1.3-1.7 times the FP32 form's error at head
// dim 512, and a value 1e-8 of the largest of its key lost half of its bits.
//
// Two launches, three where the keys are split over blocks:
//   attn_kv_split_kernel    the parts of k and v of the visible keys in the order
//                           the matrix instructions read them
//   attn_rows_split_kernel  64 rows of [qrows * heads, hd] per block
//   attn_rows_merge_kernel  adds the key splits
//
// Measured (us per call, 8 heads, against the FP32 matrix kernels in
// g4_ops.hip; error against binary64 in parentheses):
//   head dim 512, all keys   2048 rows, 4096 keys   1384 (8.0e-7) -> 670 (3.7e-7)
//                            1500 rows, 3000 keys    784 (7.1e-7) -> 431 (3.6e-7)
//                            1000 rows, 1000 keys    171 (3.7e-7) -> 101 (2.5e-7)
//                            20 rows, 2020 keys      213 (6.5e-7) -> 40 (3.7e-7)
//                            512 rows, 512 keys       62 (3.0e-7) -> 55 (2.2e-7)
//   head dim 256, window 512 1500 rows, 3000 keys    106 (4.8e-7) -> 77 (3.0e-7)
//                            20 rows, 2020 keys       34 (5.0e-7) -> 23 (2.9e-7)
// The long case is 154 TFLOP/s in FP32 terms.  Its block step of 32 keys takes
// about 5.2 us against 2.7 us of matrix work: with the tile loads left out the
// call takes 82% of its time, without the score products 67%, without the output
// products 78%, with softmax and barriers alone 25%.  (v and p as two FP16 parts,
// three products, took 568 us there and 365 over 3000 keys.)
#include <limits.h>
#include <math.h>
#include <string.h>

#include <type_traits>

#include "g4_gemv.h"
#include "g4_internal.h"
#include "g4_ops.h"

namespace g4 {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int kTile = 32;      // keys per tile
constexpr int kRows = 64;      // query rows (of qrows * heads) per block
constexpr int kMaxSplits = 64;  // key splits of one call
constexpr int kTileFlags = 2;  // per tile: K's and V's

struct RowsArgs {
  const float *q, *k, *v;
  float *out;
  uint4 *xt;  // the prefill GEMM's x' (w4_gemm_prepare), instead of out
  int *xe;
  int Mp;
  u32x4 *kv;   // split tiles: 32 hd 6 bytes of K, then of V
  int *flags;  // per tile kTileFlags
  float *part;  // [splits][nrows][hd] unnormalised outputs
  float2 *ml;   // [splits][nrows] (max, sum)
  int H, hd, keylen, qpos0, sliding, window, qrows;
  int tps;  // key tiles per split
  const int *pos_dev;
};

// Positions and key tiles of a call or of one block's rows.
struct Span {
  int qpos0, keylen, nrows;
  __device__ explicit Span(const RowsArgs &a) {
    qpos0 = a.pos_dev ? *a.pos_dev : a.qpos0;
    keylen = a.pos_dev ? qpos0 + a.qrows : a.keylen;
    nrows = a.qrows * a.H;
  }
  __device__ int kmin(const RowsArgs &a, int pos) const {
    const int lo = a.sliding ? pos - a.window + 1 : 0;
    return lo > 0 ? lo : 0;
  }
  // first tile of the call: the tile slots count from it
  __device__ int base(const RowsArgs &a) const { return kmin(a, qpos0) / kTile; }
  __device__ int kmax(int pos) const { return pos < keylen - 1 ? pos : keylen - 1; }
};

__device__ __forceinline__ uint32_t pack_h2(_Float16 a, _Float16 b) {
  return __builtin_bit_cast(uint32_t, (f16x2){a, b});
}

// 8 values as three BF16 parts, each the rounding of what the ones before
// leave (differences of FP32 values that are exact).
__device__ __forceinline__ void split8(const float (&x)[8], bf16x8 (&p)[3]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    p[0][i] = (__bf16)x[i];
    const float r = x[i] - (float)p[0][i];
    p[1][i] = (__bf16)r;
    p[2][i] = (__bf16)(r - (float)p[1][i]);
  }
}

// max over the lanes c, c + 16, c + 32, c + 48
__device__ __forceinline__ float group_max(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNoScore = -1e30f;  // where a row's maximum starts (the shader's masked logit)
constexpr uint32_t kBf16MaxBits = 0x7f7f8000u;  // from here on BF16 rounds to infinity

// Waves that share a row's head dim (its q and output dims), and the place of
// V piece n: first the first halves of every such wave's dims.
template <int HD>
constexpr int kDimWaves = HD > 256 ? 2 : 1;
template <int HD>
__device__ constexpr int v_piece(int n) {
  constexpr int NN = HD / 16, NW = NN / kDimWaves<HD>;
  const int dh = n / NW, i = n % NW;
  return (i / (NW / 2)) * (NN / 2) + dh * (NW / 2) + i % (NW / 2);
}

// K (blockIdx.y 0) or V (1) of one 32-key tile, three parts of 1 KB per piece.
// K piece (sub, j) is the A operand of score step j for keys 16 sub ..: lane
// (c, g) holds key c, dims 32 j + 8 g .. + 7.  V piece n is the A operand of
// output dims 16 n ..: lane (c, g) holds dim 16 n + c of keys 4 g .. + 3 and
// 16 + 4 g .. + 3, the keys whose probabilities lane group g computes.  Rows
// past the last visible key are zeros and are not read.  A value that BF16
// parts cannot hold (not finite, or within 2^-9 of FP32's largest) flags its
// tile, which the attention kernel then computes from the FP32 rows.  Bound by
// the latency of its loads.
template <int HD>
__global__ __launch_bounds__(512) void attn_kv_split_kernel(RowsArgs a) {
  constexpr int KI = (HD / 32 + 3) / 4, VI = (HD / 16 + 7) / 8;
  const Span sp(a);
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, c = lane & 15, g = lane >> 4;
  const int slot = blockIdx.x, k0 = (sp.base(a) + slot) * kTile;
  const int kmax = sp.kmax(sp.qpos0 + a.qrows - 1);
  if (k0 > kmax) return;
  u32x4 *dst = a.kv + (size_t)slot * (24 * HD) + (blockIdx.y ? 12 * HD : 0);
  uint32_t mx = 0;
  auto store = [&](const float (&x)[8], int piece) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t b = __float_as_uint(x[e]) & 0x7fffffffu;
      mx = b > mx ? b : mx;
    }
    bf16x8 p[3];
    split8(x, p);
#pragma unroll
    for (int q = 0; q < 3; ++q) dst[(piece * 3 + q) * 64 + lane] = __builtin_bit_cast(u32x4, p[q]);
  };
  if (blockIdx.y == 0) {
    const int sub = w & 1, key = k0 + 16 * sub + c;
    const float *src = a.k + (size_t)(key <= kmax ? key : kmax) * HD + 8 * g;
    float x[KI][8];
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const int j = (w >> 1) + 4 * i;
      const float4 *p = reinterpret_cast<const float4 *>(src + 32 * (j < HD / 32 ? j : 0));
      const float4 u0 = p[0], u1 = p[1];
      const float y[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) x[i][e] = key <= kmax ? y[e] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const int j = (w >> 1) + 4 * i;
      if (j < HD / 32) store(x[i], sub * (HD / 32) + j);
    }
  } else {
    float x[VI][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int key = k0 + (e < 4 ? 4 * g + e : 12 + 4 * g + e);
      const float *src = a.v + (size_t)(key <= kmax ? key : kmax) * HD + c;
#pragma unroll
      for (int i = 0; i < VI; ++i) {
        const int n = w + 8 * i;
        const float y = src[16 * (n < HD / 16 ? n : 0)];
        x[i][e] = key <= kmax ? y : 0.f;
      }
    }
#pragma unroll
    for (int i = 0; i < VI; ++i) {
      const int n = w + 8 * i;
      if (n < HD / 16) store(x[i], v_piece<HD>(n));
    }
  }
  const int bad = __syncthreads_or(mx >= kBf16MaxBits);
  if (t == 0) a.flags[slot * kTileFlags + blockIdx.y] = bad;
}

// One row's 8-value chunk halves as the prefill GEMM's x' (pair order (0,4)
// (1,5) (2,6) (3,7), hi plane and lo plane): the even lane group of a pair
// holds values 0-3 and writes the hi chunk, the odd one holds 4-7 and writes
// the lo chunk.
__device__ __forceinline__ u32x4 xprep_chunk(const float (&v)[4], int e, bool odd) {
  _Float16 h[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float s = ldexpf(v[i], -e);
    h[i] = (_Float16)s;
    l[i] = (_Float16)(s - (float)h[i]);
  }
  const uint32_t h01 = pack_h2(h[0], h[1]), h23 = pack_h2(h[2], h[3]);
  const uint32_t l01 = pack_h2(l[0], l[1]), l23 = pack_h2(l[2], l[3]);
  const uint32_t r01 = __shfl_xor(odd ? h01 : l01, 16, 64);
  const uint32_t r23 = __shfl_xor(odd ? h23 : l23, 16, 64);
  const uint32_t a01 = odd ? r01 : h01, a23 = odd ? r23 : h23;  // values 0-3
  const uint32_t b01 = odd ? l01 : r01, b23 = odd ? l23 : r23;  // values 4-7
  return (u32x4){(a01 & 0xffffu) | (b01 << 16), (a01 >> 16) | (b01 & 0xffff0000u),
                 (a23 & 0xffffu) | (b23 << 16), (a23 >> 16) | (b23 & 0xffff0000u)};
}

// A block owns 64 rows of [qrows * heads, hd] (row R at position qpos0 +
// R / H, seeing the keys (pos - window, pos] or [0, pos]), 16 per wave (head
// dim 512: per two waves with half of the dims each, which add their scores
// through LDS, so that two waves' registers fit a SIMD), and key tiles blockIdx.y tps .. of its rows' range.  Lane (c, g) of a wave
// works for row c throughout:
//   S^T = K . Q^T   lane (c, g) gets keys 4 g .. + 3 and 16 + 4 g .. + 3
//   softmax         a lane's 8 scores, then lane groups by two exchanges
//   O^T += V^T . P^T  the lane's probabilities are its operand as they are,
//                   so P never leaves the registers
// Tiles reach LDS by direct loads, in three buffers: A the K of keys 0-15, B
// that of keys 16-31 and then the second half of V's dims, C the first half.
//   S0 (A) | S1 (B), softmax, O0 (C) | ... O1 (B)
// A's next load leaves after S0, B's after S1 (V) and after O1 (K), C's after
// O0, so each load has at least one phase to land in: one wait and barrier
// per phase.  At head dim 512 whole K and V tiles beside each other would not
// fit 160 KB; at 256 two blocks fit a CU.
// Masked keys get weight exactly 0; tiles that a wave's rows do not see are
// skipped by that wave.
template <int HD>
__global__ __launch_bounds__(256 * kDimWaves<HD>, 2) void attn_rows_split_kernel(RowsArgs a) {
  constexpr int DH = kDimWaves<HD>, WV = 4 * DH, NTH = 64 * WV;
  constexpr int NJ = HD / 32 / DH, NN = HD / 16 / DH;  // of one wave's dims
  constexpr int KP = 3 * NJ * DH, VP = 3 * NN * DH / 2;  // 1 KB pieces of 16 keys of K, of V's half
  constexpr int KW = (KP + WV - 1) / WV, VW = VP / WV;  // and loads per wave
  constexpr int KU = KP * 64, VU = VP * 64;             // units of a buffer
  struct Smem {
    u32x4 a[KU];
    u32x4 b[KU > VU ? KU : VU];
    u32x4 c[VU];
    // partial scores of waves that share rows; before and after the tiles, one
    // value per wave or lane
    f32x4 ex[DH > 1 ? WV : 1][2][64];
  };
  __shared__ Smem sm;  // head dim 512: all of a CU's 160 KB
  typedef __attribute__((address_space(3))) void *lds_ptr;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int rg = w & 3, dh = w >> 2;  // rows 16 rg .., dims dh HD / DH ..
  const Span sp(a);
  const int H = a.H, nrows = sp.nrows;
  // the last rows see the most keys: they start first
  const int R0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * kRows;
  const int Rw = R0 + 16 * rg + c;
  if (R0 >= nrows) {  // x' only: the GEMM's padding rows qrows .. Mp - 1 as zero chunks
    const int nch = H * (HD / 8), q0 = R0 / H, nq = kRows / H;
    for (int i = t; i < nq * nch; i += NTH) {
      const int qr = q0 + i % nq, ch = i / nq;
      if (qr >= a.Mp) continue;
      a.xt[(size_t)ch * a.Mp + qr] = make_uint4(0u, 0u, 0u, 0u);
      a.xt[(size_t)(nch + ch) * a.Mp + qr] = make_uint4(0u, 0u, 0u, 0u);
    }
    return;
  }
  const int Rl = (R0 + kRows < nrows ? R0 + kRows : nrows) - 1;  // the block's last live row
  const int pos_first = sp.qpos0 + R0 / H, pos_last = sp.qpos0 + Rl / H;
  const int kt0 = sp.kmin(a, pos_first) / kTile, kt1 = sp.kmax(pos_last) / kTile;
  const int t0 = kt0 + (int)blockIdx.y * a.tps;
  const int t1 = t0 + a.tps - 1 < kt1 ? t0 + a.tps - 1 : kt1;
  if (t0 > kt1) return;
  // this lane's row, and the tiles that any row of the wave sees
  const bool live = Rw < nrows;
  const int R = live ? Rw : nrows - 1;
  const int rpos = sp.qpos0 + R / H;
  const int rlo = a.sliding ? rpos - a.window : -1;  // keys > rlo are visible
  const int Rf = R0 + 16 * rg < nrows ? R0 + 16 * rg : nrows - 1;
  const int Re = R0 + 16 * rg + 15 < nrows ? R0 + 16 * rg + 15 : nrows - 1;
  const int wt0 = R0 + 16 * rg < nrows ? sp.kmin(a, sp.qpos0 + Rf / H) / kTile : kt1 + 1;
  const int wt1 = sp.kmax(sp.qpos0 + Re / H) / kTile;

  // tiles whose every key every row of the wave sees
  const int in0 = a.sliding ? (sp.qpos0 + Re / H - a.window) / kTile + 1 : 0;
  const int in1 = R0 + 16 * rg + 15 < nrows ? (sp.qpos0 + Rf / H + 1) / kTile - 1 : -1;

  const int base = sp.base(a);
  auto tile = [&](int kt) { return a.kv + (size_t)(kt - base) * (24 * HD); };
  auto flagged = [&](int kt) {
    const int *f = a.flags + (kt - base) * kTileFlags;
    return (f[0] | f[1]) != 0;
  };
  auto load = [&](const u32x4 *src, u32x4 *dst, int pieces, int n) {
#pragma unroll
    for (int i = 0; i < n; ++i) {
      const int u = w + WV * i < pieces ? w + WV * i : pieces - 1;  // the last one twice, same bytes
      __builtin_amdgcn_global_load_lds((const void *)(src + u * 64 + lane), (lds_ptr)(dst + u * 64),
                                       16, 0, 0);
    }
  };
  auto load_k = [&](int kt, int sub) {
    load(tile(kt) + sub * (6 * HD), sub ? sm.b : sm.a, KP, KW);
  };
  auto load_v = [&](int kt, int half) {
    load(tile(kt) + 12 * HD + half * (6 * HD), half ? sm.b : sm.c, VP, VW);
  };
  load_k(t0, 0);
  load_k(t0, 1);
  load_v(t0, 0);

  // q of this lane's row: dims 32 j + 8 g .. + 7, as three parts
  bf16x8 qp[NJ][3];
  bool qslow, any_slow;  // of the block: a q beyond BF16's range; that or a flagged tile
  {
    const float4 *src = reinterpret_cast<const float4 *>(a.q + (size_t)R * HD + dh * (HD / DH) + 8 * g);
    float x[NJ][8];
    uint32_t mx = 0;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const float4 u0 = src[8 * j], u1 = src[8 * j + 1];
      x[j][0] = u0.x, x[j][1] = u0.y, x[j][2] = u0.z, x[j][3] = u0.w;
      x[j][4] = u1.x, x[j][5] = u1.y, x[j][6] = u1.z, x[j][7] = u1.w;
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t b = __float_as_uint(x[j][i]) & 0x7fffffffu;
        mx = b > mx ? b : mx;
      }
    bool f = false;
    for (int kt = t0 + t; kt <= t1; kt += NTH) f = f || flagged(kt);
    int *fl = reinterpret_cast<int *>(sm.ex);
    const int slow = (__any(mx >= kBf16MaxBits) ? 1 : 0) | (__any(f) ? 2 : 0);
    if (lane == 0) fl[w] = slow;
#pragma unroll
    for (int j = 0; j < NJ; ++j) split8(x[j], qp[j]);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    int all = 0;
#pragma unroll
    for (int i = 0; i < WV; ++i) all |= fl[i];
    qslow = __builtin_amdgcn_readfirstlane(all) & 1;
    any_slow = __builtin_amdgcn_readfirstlane(all) != 0;
  }

  float m = kNoScore, l = 0.f;  // l: this lane's keys only
  f32x4 o[NN];
#pragma unroll
  for (int n = 0; n < NN; ++n) o[n] = (f32x4){0.f, 0.f, 0.f, 0.f};

  for (int kt = t0; kt <= t1; ++kt) {
    const bool mine = kt >= wt0 && kt <= wt1;
    bf16x8 pp[3];
    float s[8];
    bool slow = false;
    // the scores of 16 keys over this wave's dims: the leading products in sums
    // of 128 dims.  The order of reads and products is the compiler's, and the
    // wave goes first on its SIMD meanwhile (one step's pieces read ahead by
    // scheduling groups cost 2% of a call of 1500 rows over 3000 keys; for the
    // outputs below the groups are worth 670 against 721 us at 2048 over 4096)
    auto scores = [&](const u32x4 *buf, float *sc) {
      const u32x4 *kb = buf + dh * (NJ * 3 * 64) + lane;
      constexpr int NM = NJ > 4 ? NJ / 4 : 1;
      f32x4 d0[NM], d1 = {0.f, 0.f, 0.f, 0.f}, d2 = d1, d3 = d1;
#pragma unroll
      for (int i = 0; i < NM; ++i) d0[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
      bf16x8 k[NJ][3];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
#pragma unroll
        for (int i = 0; i < 3; ++i) k[j][i] = __builtin_bit_cast(bf16x8, kb[(j * 3 + i) * 64]);
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        f32x4 &d = d0[j % NM];
        d1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[j][0], qp[j][1], d1, 0, 0, 0);
        d2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[j][0], qp[j][2], d2, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[j][0], qp[j][0], d, 0, 0, 0);
        d1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[j][1], qp[j][0], d1, 0, 0, 0);
        d2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[j][1], qp[j][1], d2, 0, 0, 0);
        d3 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[j][2], qp[j][0], d3, 0, 0, 0);
      }
      f32x4 d = d1 + (d2 + d3);
#pragma unroll
      for (int i = 0; i < NM; ++i) d += d0[i];
#pragma unroll
      for (int v = 0; v < 4; ++v) sc[v] = d[v];
    };
    if (mine) {
      __builtin_amdgcn_s_setprio(1);
      scores(sm.a, s);
      __builtin_amdgcn_s_setprio(0);
    }
    // B has landed everywhere, and A is free
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (kt < t1) load_k(kt + 1, 0);
    if (mine) {
      __builtin_amdgcn_s_setprio(1);
      scores(sm.b, s + 4);
      __builtin_amdgcn_s_setprio(0);
      if (DH > 1) {
        sm.ex[w][0][lane] = (f32x4){s[0], s[1], s[2], s[3]};
        sm.ex[w][1][lane] = (f32x4){s[4], s[5], s[6], s[7]};
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // B is free
    load_v(kt, 1);
    if (mine) {
      if (DH > 1) {  // in dim order, so the waves of a row hold the same scores
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const f32x4 d = sm.ex[rg][u][lane] + sm.ex[rg + 4 * (DH - 1)][u][lane];
#pragma unroll
          for (int v = 0; v < 4; ++v) s[4 * u + v] = d[v];
        }
      }
      const bool inner = kt >= in0 && kt <= in1;
      if (any_slow) slow = qslow || __builtin_amdgcn_readfirstlane(flagged(kt) ? 1 : 0) != 0;
      auto key_of = [&](int i) { return kt * kTile + (i < 4 ? 4 * g + i : 12 + 4 * g + i); };
      if (slow) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int key = key_of(i) < sp.keylen ? key_of(i) : sp.keylen - 1;
          const float *qf = a.q + (size_t)R * HD, *kf = a.k + (size_t)key * HD;
          float d = 0.f;
          for (int x = 0; x < HD; ++x) d = fmaf(qf[x], kf[x], d);
          s[i] = d;
        }
      }
      if (!inner) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int key = key_of(i);
          if (!(live && key <= rpos && key < sp.keylen && key > rlo)) s[i] = -INFINITY;
        }
      }
      float tm = s[0];
#pragma unroll
      for (int i = 1; i < 8; ++i) tm = fmaxf(tm, s[i]);
      // (fmaxf drops a NaN score, whose p is NaN.)
      const float mn = fmaxf(m, group_max(tm));
      const float corr = __builtin_amdgcn_exp2f((m - mn) * kLog2e);
      m = mn;
      float ls = 0.f, p[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i] = __builtin_amdgcn_exp2f((s[i] - mn) * kLog2e);  // 0 for a masked key
        ls += p[i];
      }
      l = fmaf(l, corr, ls);
      split8(p, pp);
      if (__any(corr != 1.f)) {
#pragma unroll
        for (int n = 0; n < NN; ++n) o[n] *= corr;
      }
    }
    auto outputs = [&](const u32x4 *buf, auto half) {
      constexpr int n0 = decltype(half)::value * (NN / 2);
      const u32x4 *vb = buf + dh * (NN / 2 * 3 * 64) + lane;
      bf16x8 vv[NN / 2][3];
#pragma unroll
      for (int i = 0; i < NN / 2; ++i)
#pragma unroll
        for (int q = 0; q < 3; ++q) vv[i][q] = __builtin_bit_cast(bf16x8, vb[(3 * i + q) * 64]);
      constexpr int kProducts[6][2] = {{2, 0}, {1, 1}, {0, 2}, {1, 0}, {0, 1}, {0, 0}};
#pragma unroll
      for (int i = 0; i < NN / 2; i += 2) {
        f32x4 d[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
          for (int u = 0; u < 2; ++u)
            d[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv[i + u][kProducts[q][0]],
                                                           pp[kProducts[q][1]], d[u], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 2; ++u) o[n0 + i + u] += d[u];
      }
      constexpr int AHEAD = 2;
      __builtin_amdgcn_sched_group_barrier(0x100, 3 * AHEAD, 0);
#pragma unroll
      for (int i = 0; i < NN / 2; i += 2) {
#pragma unroll
        for (int u = 0; u < 3; ++u) {
          __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
          if (i + AHEAD < NN / 2) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
          if (i > 0) __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        }
      }
    };
    if (mine && !slow) outputs(sm.c, std::integral_constant<int, 0>());
    // B (V) and A have landed everywhere, and C is free
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (kt < t1) load_v(kt + 1, 0);
    if (mine && !slow) outputs(sm.b, std::integral_constant<int, 1>());
    if (slow) {  // keys that the row sees, from the FP32 rows
      for (int gg = 0; gg < 4; ++gg)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float pk = __shfl((float)pp[0][i] + ((float)pp[1][i] + (float)pp[2][i]), 16 * gg + c, 64);
          const int key = kt * kTile + (i < 4 ? 4 * gg + i : 12 + 4 * gg + i);
          if (!(live && key <= rpos && key < sp.keylen && key > rlo)) continue;
          const float *vp = a.v + (size_t)key * HD + dh * (HD / DH) + 4 * g;
#pragma unroll
          for (int n = 0; n < NN; ++n) {
            const float4 vv = *reinterpret_cast<const float4 *>(vp + 16 * n);
            o[n][0] = fmaf(pk, vv.x, o[n][0]);
            o[n][1] = fmaf(pk, vv.y, o[n][1]);
            o[n][2] = fmaf(pk, vv.z, o[n][2]);
            o[n][3] = fmaf(pk, vv.w, o[n][3]);
          }
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // B is free
    if (kt < t1) load_k(kt + 1, 1);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);

  if (gridDim.y > 1) {
    if (!live) return;
    float *pp = a.part + ((size_t)blockIdx.y * nrows + R) * HD + dh * (HD / DH) + 4 * g;
#pragma unroll
    for (int n = 0; n < NN; ++n) *reinterpret_cast<f32x4 *>(pp + 16 * n) = o[n];
    if (g == 0 && dh == 0) a.ml[(size_t)blockIdx.y * nrows + R] = make_float2(m, l);
    return;
  }
#pragma unroll
  for (int n = 0; n < NN; ++n)
#pragma unroll
    for (int v = 0; v < 4; ++v) o[n][v] = live ? o[n][v] / l : 0.f;
  if (!a.xt) {
    if (!live) return;
    float *op = a.out + (size_t)R * HD + dh * (HD / DH) + 4 * g;
#pragma unroll
    for (int n = 0; n < NN; ++n) *reinterpret_cast<f32x4 *>(op + 16 * n) = o[n];
    return;
  }
  // x' of the GEMM: the exponent of a query row from its H heads (H divides
  // 16, so they are lanes of this wave); rows past qrows are zero chunks
  float mx = 0.f;
#pragma unroll
  for (int n = 0; n < NN; ++n)
#pragma unroll
    for (int v = 0; v < 4; ++v) mx = fmaxf(mx, fabsf(o[n][v]));
  for (int d = 1; d < H; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
  if (DH > 1) {
    float *rmx = reinterpret_cast<float *>(sm.ex);
    if (g == 0) rmx[16 * w + c] = mx;
    __syncthreads();
    mx = fmaxf(rmx[16 * rg + c], rmx[16 * (rg + 4 * (DH - 1)) + c]);
  }
  const int e = mx > 0.f && mx <= 3.4e38f ? ilogbf(mx) - 13 : 0;
  const int qr = Rw / H, h = Rw - qr * H;
  if (live && h == 0 && g == 0 && dh == 0) a.xe[qr] = e;
  const size_t lo_plane = (size_t)H * (HD / 8) * a.Mp;
#pragma unroll
  for (int n = 0; n < NN; ++n) {
    const float v[4] = {o[n][0], o[n][1], o[n][2], o[n][3]};
    const u32x4 ch = xprep_chunk(v, e, g & 1);
    const size_t at = (size_t)(h * (HD / 8) + dh * (HD / DH / 8) + 2 * n + (g >> 1)) * a.Mp + qr + ((g & 1) ? lo_plane : 0);
    if (qr < a.Mp) reinterpret_cast<u32x4 *>(a.xt)[at] = ch;
  }
}

// Adds the key splits of one query row: out = sum_s e^(m_s - M) o_s /
// sum_s e^(m_s - M) l_s in split order, as rows of out or as the GEMM's x'.
// A block is one query row (x': all heads, one exponent) or one (query row,
// head); thread t takes 16-byte units t, t + 256, ... of it.
template <int HD, bool X>
__global__ __launch_bounds__(256) void attn_rows_merge_kernel(RowsArgs a) {
  constexpr int U4 = HD / 4;  // units per head
  constexpr int kHeads = 16;
  __shared__ float wt[X ? kHeads : 1][kMaxSplits];
  __shared__ float rl[kHeads];
  __shared__ float red[4];
  const Span sp(a);
  const int t = threadIdx.x, H = a.H, nrows = sp.nrows;
  const int qr = X ? blockIdx.x : blockIdx.x / H, h0 = X ? 0 : blockIdx.x - qr * H;
  const int nh = X ? H : 1;
  if (X && qr >= a.qrows) {
    const int nch = H * (HD / 8);
    for (int ch = t; ch < 2 * nch; ch += 256) a.xt[(size_t)ch * a.Mp + qr] = make_uint4(0u, 0u, 0u, 0u);
    return;
  }
  // splits of a row: those of its 64-row block
  auto splits = [&](int R) {
    const int r0 = R / kRows * kRows;
    const int re = (r0 + kRows < nrows ? r0 + kRows : nrows) - 1;
    const int nt = sp.kmax(sp.qpos0 + re / H) / kTile - sp.kmin(a, sp.qpos0 + r0 / H) / kTile + 1;
    return (nt + a.tps - 1) / a.tps;
  };
  // weights e^(m_s - M) and the sum of each head: 16 lanes per head
  {
    const int hh = t >> 4, li = t & 15;
    const int R = qr * H + h0 + (hh < nh ? hh : 0), ns = splits(R);
    float2 ml[kMaxSplits / 16];
    float M = -2e30f, L = 0.f;
#pragma unroll
    for (int i = 0; i < kMaxSplits / 16; ++i) {
      const int s = li + 16 * i;
      ml[i] = a.ml[(size_t)(s < ns ? s : 0) * nrows + R];
      M = fmaxf(M, ml[i].x);
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
#pragma unroll
    for (int i = 0; i < kMaxSplits / 16; ++i) {
      const int s = li + 16 * i;
      const float e = s < ns ? __builtin_amdgcn_exp2f((ml[i].x - M) * kLog2e) : 0.f;
      if (hh < nh) wt[hh][s] = e;
      L += s < ns ? e * ml[i].y : 0.f;
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) L += __shfl_xor(L, o, 64);
    if (hh < nh && li == 0) rl[hh] = L;
  }
  __syncthreads();
  constexpr int NU = X ? kHeads * U4 / 256 : (U4 + 255) / 256;
  f32x4 v[NU];
  float mx = 0.f;
#pragma unroll
  for (int i = 0; i < NU; ++i) {
    v[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int u = t + 256 * i, h = u / U4, d = u - h * U4;
    if (h >= nh) continue;
    const int R = qr * H + h0 + h, ns = splits(R);
    const float *p = a.part + (size_t)R * HD + 4 * d;
    const size_t step = (size_t)nrows * HD;
    int s = 0;
    for (; s + 4 <= ns; s += 4) {
      f32x4 x[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = *reinterpret_cast<const f32x4 *>(p + (s + k) * step);
#pragma unroll
      for (int k = 0; k < 4; ++k) v[i] += wt[h][s + k] * x[k];
    }
    for (; s < ns; ++s) v[i] += wt[h][s] * *reinterpret_cast<const f32x4 *>(p + s * step);
    const float L = rl[h];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[i][k] = v[i][k] / L;
      mx = fmaxf(mx, fabsf(v[i][k]));
    }
    if (!X) *reinterpret_cast<f32x4 *>(a.out + (size_t)R * HD + 4 * d) = v[i];
  }
  if (!X) return;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  if ((t & 63) == 0) red[t >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const int e = mx > 0.f && mx <= 3.4e38f ? ilogbf(mx) - 13 : 0;
  if (t == 0) a.xe[qr] = e;
  const size_t lo_plane = (size_t)H * (HD / 8) * a.Mp;
#pragma unroll
  for (int i = 0; i < NU; ++i) {
    const int u = t + 256 * i;  // units 2 ch and 2 ch + 1 sit in neighbouring lanes
    _Float16 hv[4], lv[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float s = ldexpf(v[i][k], -e);
      hv[k] = (_Float16)s;
      lv[k] = (_Float16)(s - (float)hv[k]);
    }
    const bool odd = t & 1;
    const uint32_t h01 = pack_h2(hv[0], hv[1]), h23 = pack_h2(hv[2], hv[3]);
    const uint32_t l01 = pack_h2(lv[0], lv[1]), l23 = pack_h2(lv[2], lv[3]);
    const uint32_t r01 = __shfl_xor(odd ? h01 : l01, 1, 64);
    const uint32_t r23 = __shfl_xor(odd ? h23 : l23, 1, 64);
    const uint32_t a01 = odd ? r01 : h01, a23 = odd ? r23 : h23;
    const uint32_t b01 = odd ? l01 : r01, b23 = odd ? l23 : r23;
    if (u / U4 < nh)
      reinterpret_cast<u32x4 *>(a.xt)[(size_t)(u >> 1) * a.Mp + qr + (odd ? lo_plane : 0)] =
          (u32x4){(a01 & 0xffffu) | (b01 << 16), (a01 >> 16) | (b01 & 0xffff0000u),
                  (a23 & 0xffffu) | (b23 << 16), (a23 >> 16) | (b23 & 0xffff0000u)};
  }
}

int cdiv(int a, int b) { return (a + b - 1) / b; }

struct RowsPlan {
  int tiles, tps, splits;
  size_t kv, flags, part, total;  // floats
};

constexpr int kMaxKeys = 16384;  // launch_attention's limit
constexpr int kRing = 2048;
static_assert(2 * (kMaxKeys / kTile + 1) + 4 < kRing, "a block's time fits the ring");

constexpr int kMaxCus = 512;
int cus() {
  const int n = cu_count();
  return n <= 0 ? 256 : n < kMaxCus ? n : kMaxCus;
}

// Most keys that the rows of `positions` consecutive positions see.
int keys_seen(int positions, int max_keylen, bool sliding, int window) {
  const long n = (long)window - 1 + positions;
  return sliding && n < max_keylen ? (int)n : max_keylen;
}

// What a plan depends on besides the scratch.
struct RowsKey {
  int qrows, heads, hd, max_keylen, sliding, window, cus;
};

// Key tiles of the call, and the split of a row block's tiles over blocks (at
// least two tiles each, and no more than `avail` floats of scratch).
// Head dim 256: as many as fill the CUs with two blocks each.
// Head dim 512, one block per CU: the split whose blocks, dealt to the CUs in
// launch order, end first by these costs in halves of a tile's 5.2 us: 2 per
// tile, 4 per block (q's conversion, the first loads, the stores), 1 for a block
// with no tiles (early rows have fewer than late ones, yet every block needs its
// LDS), and with more than one split 3 for the merge and 1 per 36 blocks for its
// planes.  us per call at 8 heads (* as chosen), 1, 2, 3, 4, 5 splits, then 6 and 8:
//   1000 rows, 1000 keys  201 124   96*  127 123  114 126
//    700 rows, 2700 keys  493 271  196*  286 238  217 248
//   1500 rows, 1500 keys  286 173* 222   186 183  195 208
//   2048 rows, 4096 keys  730 766  708   671* 677  726 776
//    300 rows,  900 keys  180 110   83    72  61   56  59*
//   1500 rows, 3000 keys  542 430* 412   458 394  434 442
bool find_plan(const RowsKey &key, size_t avail, RowsPlan *p) {
  const int qrows = key.qrows, heads = key.heads, hd = key.hd, max_keylen = key.max_keylen;
  const int window = key.window;
  const bool sliding = key.sliding != 0;
  const int nrows = qrows * heads, blocks = cdiv(nrows, kRows);
  const int span = cdiv(kRows, heads) + 1;  // positions of a block's rows
  const int all = cdiv(max_keylen, kTile);
  auto tiles_of = [&](int positions) {  // whatever their alignment
    const int n = (keys_seen(positions, max_keylen, sliding, window) + kTile - 2) / kTile + 1;
    return n < all ? n : all;
  };
  p->tiles = tiles_of(qrows);
  p->kv = (size_t)p->tiles * hd * 96;
  p->flags = ((size_t)p->tiles * kTileFlags + 3) & ~size_t(3);
  const int nt = tiles_of(span < qrows ? span : qrows);
  const int slots = key.cus;
  // tiles of row block b (launched last to first), as the kernel counts them
  const int qpos0 = max_keylen - qrows;
  auto block_tiles = [&](int b) {
    const int first = qpos0 + b * kRows / heads;
    const int last = qpos0 + ((b + 1) * kRows < nrows ? (b + 1) * kRows - 1 : nrows - 1) / heads;
    const int lo = sliding && first - window + 1 > 0 ? first - window + 1 : 0;
    return last / kTile - lo / kTile + 1;
  };
  auto fits = [&](int splits) {
    p->splits = splits;
    p->part = splits > 1 ? (size_t)splits * nrows * (hd + 2) : 0;
    p->total = p->kv + p->flags + p->part;
    return p->total <= avail;
  };
  auto tiles_per = [&](int splits) {
    const int t = cdiv(nt, splits);
    return splits == 1 || t > 2 ? t : 2;
  };
  if (hd <= 256) {
    int want = 2 * slots / blocks;
    want = want > kMaxSplits ? kMaxSplits : want < 1 ? 1 : want;
    for (; want >= 1; --want) {
      p->tps = tiles_per(want);
      if (fits(cdiv(nt, p->tps))) return true;
    }
    return false;
  }
  if (blocks > 2 * slots) {  // more than the limit below with any split
    p->tps = nt;
    return fits(1);
  }
  int tiles[2 * kMaxCus];
  for (int b = 0; b < blocks; ++b) tiles[b] = block_tiles(b);
  // CUs that become free at each time, from `now` on (a block takes less than a
  // turn of the ring: see kMaxKeys)
  int free_at[kRing];
  long best = LONG_MAX;
  int best_splits = 0, best_tps = 0, last_tps = 0;
  for (int want = 1; want <= kMaxSplits; want += want < 6 ? 1 : want / 3) {
    const int tps = tiles_per(want), splits = cdiv(nt, tps);
    if (tps == last_tps) continue;
    if (splits > 1 && (long)splits * blocks > 4L * slots) break;
    last_tps = tps;
    if (!fits(splits)) continue;
    for (int &f : free_at) f = 0;
    free_at[0] = slots;
    long end = 0, used = 0;
    unsigned now = 0;
    for (int y = 0; y < splits && end < best; ++y)
      for (int b = blocks - 1; b >= 0 && end < best; --b) {
        int t = tiles[b] - y * tps;
        t = t < tps ? t : tps;
        const int len = t > 0 ? 2 * t + 4 : 1;
        used += t > 0;
        while (free_at[now % kRing] == 0) ++now;
        --free_at[now % kRing];
        ++free_at[(now + len) % kRing];
        if ((long)now + len > end) end = (long)now + len;
      }
    if (splits > 1) end += 3 + used / 36;
    if (end < best) {
      best = end;
      best_splits = splits;
      best_tps = tps;
    }
  }
  p->tps = best_tps;
  return best_splits > 0 && fits(best_splits);
}

// The plan for at most `avail` floats.  At head dim 512 finding it takes 5 to 15 us
// of host time, more than a call's launches, so the one for any scratch is kept
// per thread for the last key (a call asks for its scratch and then launches, an
// engine's layers follow each other); where it fits, it is also the best that
// fits.
bool rows_plan(const RowsKey &key, size_t avail, RowsPlan *p) {
  if (key.hd <= 256) return find_plan(key, avail, p);
  static thread_local RowsKey last{};
  static thread_local RowsPlan plan{};
  if (memcmp(&last, &key, sizeof(key)) != 0) {
    find_plan(key, ~size_t(0), &plan);
    last = key;
  }
  *p = plan;
  return plan.total <= avail || find_plan(key, avail, p);
}

template <int HD>
int launch_rows(const RowsArgs &a, const RowsPlan &p) {
  hipLaunchKernelGGL(attn_kv_split_kernel<HD>, dim3(p.tiles, 2), dim3(512), 0, stream(), a);
  G4_LAUNCH_CHECK("attn_kv_split_kernel");
  const bool pad = a.xt && p.splits == 1;
  const dim3 grid(cdiv((pad ? a.Mp : a.qrows) * a.H, kRows), p.splits);
  hipLaunchKernelGGL(attn_rows_split_kernel<HD>, grid, dim3(256 * kDimWaves<HD>), 0, stream(), a);
  G4_LAUNCH_CHECK("attn_rows_split_kernel");
  if (p.splits == 1) return G4_OK;
  if (a.xt)
    hipLaunchKernelGGL((attn_rows_merge_kernel<HD, true>), dim3(a.Mp), dim3(256), 0, stream(), a);
  else
    hipLaunchKernelGGL((attn_rows_merge_kernel<HD, false>), dim3(a.qrows * a.H), dim3(256), 0,
                       stream(), a);
  G4_LAUNCH_CHECK("attn_rows_merge_kernel");
  return G4_OK;
}

}  // namespace

// Where the FP32 matrix kernels take longer: their time is that of the heaviest
// 16-row block's walk over 16-key tiles (about 1.6 us a tile at head dim 512,
// 0.75 at 256) times the rounds of such blocks over the CUs, and 10 us.  Here a
// call costs 25 to 35 us before keys matter (three launches, q's conversion
// and, growing with the rows, the planes of the key splits).  Measured at 8
// heads, FP32 kernel against this one: head dim 512, 12 rows over 362 keys 47 /
// 33 us, 5 over 290 40 / 30, 80 over 280 38 / 36, 320 over 320 42 / 40; head dim
// 256, 20 rows over 370 keys 26 / 22, 512 over 512 33 / 39, 700 over 700 51 / 45,
// 1000 over 1000 65 / 50.  With 4, 2 and 1 heads (2 to 1000 rows, 0 to 2500 keys
// before them, both head dims) the calls that the rule brings here take 0.15
// to 1 times the FP32 kernels' time, but 1.05 at 2 heads, 1000 rows, window 512.
// One row has kernels of its own.
bool attention_rows_wins(int qrows, int heads, int hd, int max_keylen, bool sliding, int window) {
  if (qrows < 2 || (hd != 256 && hd != 512) || max_keylen > kMaxKeys) return false;
  const int nrows = qrows * heads;
  const int keys = keys_seen(cdiv(16, heads) + 1, max_keylen, sliding, window);
  const int steps = cdiv(keys, 16) * cdiv(nrows, 16 * cus());
  return hd == 512 ? steps >= 18 : steps >= 22 + nrows / 200;
}

size_t attention_rows_floats(int qrows, int heads, int hd, int max_keylen, bool sliding,
                             int window) {
  RowsPlan p{};
  if (!attention_rows_wins(qrows, heads, hd, max_keylen, sliding, window)) return 0;
  rows_plan({qrows, heads, hd, max_keylen, sliding, window, cus()}, ~size_t(0), &p);
  return p.total;
}

int launch_attention_rows(const float *q, const float *k, const float *v, int qrows, int heads,
                          int hd, int keylen, int qpos0, const int *pos_dev, int max_keylen,
                          bool sliding, int window, float *scratch, size_t scratch_floats,
                          float *out, void *xt, int *xe, int Mp, bool *taken) {
  RowsPlan p{};
  *taken = false;
  if (!rows_plan({qrows, heads, hd, max_keylen, sliding, window, cus()}, scratch_floats, &p)) return G4_OK;
  RowsArgs a{};
  a.q = q;
  a.k = k;
  a.v = v;
  a.out = out;
  a.xt = static_cast<uint4 *>(xt);
  a.xe = xe;
  a.Mp = Mp;
  a.kv = reinterpret_cast<u32x4 *>(scratch);
  a.flags = reinterpret_cast<int *>(scratch + p.kv);
  a.part = scratch + p.kv + p.flags;
  a.ml = reinterpret_cast<float2 *>(a.part + (size_t)p.splits * qrows * heads * hd);
  a.H = heads;
  a.hd = hd;
  a.keylen = keylen;
  a.qpos0 = qpos0;
  a.sliding = sliding ? 1 : 0;
  a.window = window;
  a.qrows = qrows;
  a.tps = p.tps;
  a.pos_dev = pos_dev;
  *taken = true;
  return hd == 512 ? launch_rows<512>(a, p) : launch_rows<256>(a, p);
}

}  // namespace g4

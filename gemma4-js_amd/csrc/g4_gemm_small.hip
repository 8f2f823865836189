// The W4A16 product for a few rows of x (a short prompt, a chat message): the
// weights' bytes and the launches count here, not the matrix rate.
//
// Bound: HBM and latency.  The prefill GEMM (g4_gemm.hip) pads such rows to
// tiles of 64, converts x in one or two launches of its own and walks K with a
// barrier per stage: 23 rows through 2 x 12288 outputs at K 1536 took 3.8 +
// 22.8 us, through 1536 outputs at K 12288 4.3 + 4.6 + 20.9 + 4.0.  Here nothing
// is staged and nothing loops: a block owns TN 16-column tiles and up to 32
// rows; each of its 8 waves takes S stages of 64 values of K, issues every load
// of them at once (x straight from the caller's rows, the packed words and
// scales from the stage-major tile copy), converts x in registers, dequantizes
// and multiplies, and the 8 partial tiles meet in LDS, added in wave order.
//
// Numerics are the prefill GEMM's: FP16 q s 2^shift (exact), x 2^-e as FP16
// hi + lo (FP32 x) or hi (BF16 x, exact), FP32 accumulation.  e is the exponent
// of the row's largest value within the wave's S stages (the prefill GEMM's:
// within the whole row), so no value is further below it than there.
// An x value below 2^-21 of that largest keeps fewer than 17 bits: an output whose
// weight is zero at an x 1e8 above the others is good to 5e-5 (to 4e-7 at 1e6).
// The GEMV that two to four FP32 rows leave for this kernel is worse there, since
// it takes 8 times x off again after its sums (0.1 at 1e6).
#include <math.h>

#include "g4_gemv.h"
#include "g4_internal.h"

namespace g4 {

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kWaves = 8;
constexpr int kTileUnits = 36;  // 16-byte units of a tile's stage block
constexpr int kMaxSegs = 3;

struct SmallArgs {
  const void *x;     // [rows, K], or null:
  const u32x4 *xt;   // x' (w4_gemm_prepare) ...
  const int *xe;     // ... and its row exponents
  const u32x4 *tw[kMaxSegs];
  void *y[kMaxSegs];
  const int16_t *rs[kMaxSegs];
  int N[kMaxSegs], shift[kMaxSegs], t0[kMaxSegs + 1];
  int n, glu, y_bf16, rows, K, Mp;
  int per;  // stages per block (blockIdx.y)
  float *part;
  size_t pstride, poff[kMaxSegs];
};

// x modes: FP32 rows, BF16 rows, x' written by x's producer
enum { kXF32, kXBf16, kXPrep };

// max(m, |a|, |b|) in one instruction (fmaxf would first quieten each operand)
__device__ __forceinline__ float max_abs(float m, float a, float b) {
  float r;
  asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
  return r;
}

typedef float f32x2 __attribute__((ext_vector_type(2)));

// 8 values times 2^-e as FP16 pairs (0,4) (1,5) (2,6) (3,7), hi and lo; 3
// instructions a value (packed conversions, the remainders as mixed FMAs).
template <bool LO>
__device__ __forceinline__ void chunk_halves(const float (&v)[8], int e, f16x8 &hi, f16x8 &lo) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x2 s = {ldexpf(v[i], -e), ldexpf(v[i + 4], -e)};
    const f16x2 h = __builtin_convertvector(s, f16x2);
    hi[2 * i] = h[0];
    hi[2 * i + 1] = h[1];
    if (LO) {
      f32x2 r;
      const uint32_t hb = __builtin_bit_cast(uint32_t, h);
      asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r[0]) : "v"(hb), "v"(s[0]));
      asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
          : "=v"(r[1])
          : "v"(hb), "v"(s[1]));
      const f16x2 l = __builtin_convertvector(r, f16x2);
      lo[2 * i] = l[0];
      lo[2 * i + 1] = l[1];
    }
  }
}

template <int TM, int TN, int S, int XM>
__global__ __launch_bounds__(64 * kWaves, 2) void w4_gemm_small_kernel(SmallArgs a) {
  constexpr int NX = XM == kXBf16 ? 1 : 2;
  __shared__ f32x4 red[kWaves][TM * TN][64];
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  const bool glu = a.glu != 0;
  const int cg = blockIdx.x;
  const int si = glu ? 0 : a.n > 2 && cg >= a.t0[2] ? 2 : a.n > 1 && cg >= a.t0[1] ? 1 : 0;
  const int m0 = blockIdx.z * 16 * TM;
  // tile jj of the block: its weight, and its 16 columns
  auto seg_of = [&](int jj) { return glu && jj >= TN / 2 ? 1 : si; };
  auto tile_of = [&](int jj) {
    return glu ? cg * (TN / 2) + (jj >= TN / 2 ? jj - TN / 2 : jj) : (cg - a.t0[si]) * TN + jj;
  };
  const int stages = a.K >> 6;
  int end = ((int)blockIdx.y + 1) * a.per;
  end = end < stages ? end : stages;
  const int st0 = (int)blockIdx.y * a.per + w * S;
  const int nv = end - st0 < S ? (end > st0 ? end - st0 : 0) : S;  // stages of this wave

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  if (nv > 0) {
    // every load first: x (needed first), then the weights.  Stages past the
    // wave's last re-read it, and their x is zeroed.
    u32x4 xr[S][TM][XM == kXBf16 ? 2 : 4];
    int e[TM];
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      const int row = m0 + 16 * m + lr < a.rows ? m0 + 16 * m + lr : a.rows - 1;
      e[m] = XM == kXPrep ? a.xe[row] : 0;
#pragma unroll
      for (int i = 0; i < S; ++i) {
        const int st = st0 + (i < nv ? i : nv - 1);
        if constexpr (XM == kXPrep) {
          // hi and lo of chunks 8 st + 2 lq and + 1
          const u32x4 *p = a.xt + (size_t)(8 * st + 2 * lq) * a.Mp + m0 + 16 * m + lr;
          const size_t lo = (size_t)(a.K >> 3) * a.Mp;
          xr[i][m][0] = p[0];
          xr[i][m][1] = p[a.Mp];
          xr[i][m][2] = p[lo];
          xr[i][m][3] = p[lo + a.Mp];
        } else {
          constexpr int U = XM == kXBf16 ? 2 : 4;  // 16-byte units of a lane's 16 values
          const u32x4 *p = static_cast<const u32x4 *>(a.x) +
                           ((size_t)row * stages + st) * (4 * U) + lq * U;
#pragma unroll
          for (int u = 0; u < U; ++u) xr[i][m][u] = p[u];
        }
      }
    }
    u32x2 wd[S][TN];
    uint32_t sc[S][TN];
    int sh[TN];
#pragma unroll
    for (int jj = 0; jj < TN; ++jj) {
      const int seg = seg_of(jj), T = (a.N[seg] + 15) >> 4;
      const int tile = tile_of(jj) < T ? tile_of(jj) : T - 1;
#pragma unroll
      for (int i = 0; i < S; ++i) {
        const int st = st0 + (i < nv ? i : nv - 1);
        const char *p = reinterpret_cast<const char *>(a.tw[seg] + ((size_t)st * T + tile) * kTileUnits);
        wd[i][jj] = *reinterpret_cast<const u32x2 *>(p + 8 * lane);
        sc[i][jj] = *reinterpret_cast<const uint32_t *>(p + 512 + 4 * lr);
      }
      const int row = 16 * tile + lr < a.N[seg] ? 16 * tile + lr : a.N[seg] - 1;
      sh[jj] = a.rs[seg] ? a.rs[seg][row] : a.shift[seg];
    }

    if (nv < S) {
#pragma unroll
      for (int i = 1; i < S; ++i)
        if (i >= nv)
#pragma unroll
          for (int m = 0; m < TM; ++m)
#pragma unroll
            for (auto &u : xr[i][m]) u = (u32x4){0u, 0u, 0u, 0u};
    }
    // x as the A operands: chunks 2 lq and 2 lq + 1 of each stage
    f16x8 xa[S][TM][NX][2];
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      if constexpr (XM == kXPrep) {
#pragma unroll
        for (int i = 0; i < S; ++i)
#pragma unroll
          for (int h = 0; h < NX; ++h)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              xa[i][m][h][j] = __builtin_bit_cast(f16x8, xr[i][m][2 * h + j]);
            }
      } else {
        auto value = [&](int i, int k) {  // k-th of the lane's 16 values of stage i
          if constexpr (XM == kXBf16) {
            const uint32_t u = xr[i][m][k >> 3][(k >> 1) & 3];
            return bf16_to_f32(k & 1 ? u >> 16 : u & 0xffffu);
          } else {
            return __uint_as_float(xr[i][m][k >> 2][k & 3]);
          }
        };
        float mx = 0.f;
#pragma unroll
        for (int i = 0; i < S; ++i)
#pragma unroll
          for (int k = 0; k < 16; k += 2) mx = max_abs(mx, value(i, k), value(i, k + 1));
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        // all-zero and non-finite rows keep e = 0
        e[m] = mx > 0.f && mx <= 3.4e38f ? __builtin_amdgcn_frexp_expf(mx) - 14 : 0;
#pragma unroll
        for (int i = 0; i < S; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = value(i, 8 * j + k);
            chunk_halves<NX == 2>(v, e[m], xa[i][m][0][j], xa[i][m][NX - 1][j]);
          }
      }
    }

    uint32_t mask = 0x000F000Fu;
    asm("" : "+v"(mask));  // in a VGPR: lets v_and_or_b32 take the magic
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int jj = 0; jj < TN; ++jj) {
        const uint32_t sb = (lq >> 1) ? sc[i][jj] >> 16 : sc[i][jj] & 0xffffu;
        const _Float16 s1 = (_Float16)ldexpf(bf16_to_f32(sb), sh[jj]);
        const f16x2 s2 = {s1, s1}, off = {(_Float16)1032.f, (_Float16)1032.f};
        f16x8 b[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          u32x4 u;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint32_t p = ((wd[i][jj][j] >> (4 * k)) & mask) | 0x64006400u;
            u[k] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(f16x2, p) - off) * s2);
          }
          b[j] = __builtin_bit_cast(f16x8, u);
        }
#pragma unroll
        for (int h = 0; h < NX; ++h)
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int m = 0; m < TM; ++m)
              acc[m][jj] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[i][m][h][j], b[j], acc[m][jj], 0,
                                                                  0, 0);
      }
    // rows 4 lq + r of a tile: their exponents sit in lanes of those numbers
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int er = __shfl(e[m], 4 * lq + r, 64);
#pragma unroll
        for (int jj = 0; jj < TN; ++jj) acc[m][jj][r] = ldexpf(acc[m][jj][r], er - sh[jj]);
      }
  }
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int jj = 0; jj < TN; ++jj) red[w][m * TN + jj][lane] = acc[m][jj];
  __syncthreads();

  auto sum = [&](int tile, int l) {
    f32x4 v = red[0][tile][l];
#pragma unroll
    for (int k = 1; k < kWaves; ++k) v += red[k][tile][l];
    return v;
  };
  const int out_tiles = glu ? TM * (TN / 2) : TM * TN;
  const int per_row = glu ? TN / 2 : TN;
  for (int u = t; u < out_tiles * 64; u += 64 * kWaves) {
    const int o = u >> 6, m = o / per_row, jj = o - m * per_row;
    const int seg = seg_of(jj), N = a.N[seg];
    const int n = 16 * tile_of(jj) + lr;
    f32x4 v = sum(m * TN + jj, lane);
    if (glu) {
      const f32x4 up = sum(m * TN + jj + TN / 2, lane);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = gelu_tanh(v[r]) * up[r];
    }
    if (n >= N) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m0 + 16 * m + 4 * lq + r;
      if (row >= a.rows) continue;
      const size_t at = (size_t)row * N + n;
      if (gridDim.y > 1)
        (a.part + blockIdx.y * a.pstride + a.poff[seg])[at] = v[r];
      else if (a.y_bf16)
        static_cast<uint16_t *>(a.y[seg])[at] = (uint16_t)f32_to_bf16_rne(v[r]);
      else
        static_cast<float *>(a.y[seg])[at] = v[r];
    }
  }
}

template <int XM>
int launch_small(const SmallArgs &a, const GemmSmallPlan &p, dim3 grid) {
#define G4_SMALL(M, T, SS)                                                                   \
  if (p.tm == M && p.tn == T && p.s == SS) {                                                 \
    hipLaunchKernelGGL((w4_gemm_small_kernel<M, T, SS, XM>), grid, dim3(64 * kWaves), 0,     \
                       stream(), a);                                                         \
    G4_LAUNCH_CHECK("w4_gemm_small_kernel");                                                 \
    return G4_OK;                                                                            \
  }
#define G4_SMALL_T(M, T) G4_SMALL(M, T, 3) G4_SMALL(M, T, 4)
  G4_SMALL_T(1, 1) G4_SMALL_T(1, 2) G4_SMALL_T(1, 3) G4_SMALL_T(1, 6)
  G4_SMALL_T(2, 1) G4_SMALL_T(2, 2) G4_SMALL_T(2, 3) G4_SMALL_T(2, 6)
#undef G4_SMALL_T
#undef G4_SMALL
  return fail(G4_E_ARG, "w4_gemm_small: no tile %dx%d of %d stages", p.tm, p.tn, p.s);
}

}  // namespace

// The call is taken where its blocks fit the CUs in one round (one block of 8
// waves per CU) with at most 8 slices of K (what the consumers of unsummed
// planes add), by the narrowest tile that does: fewer columns per block mean
// more loads in flight.  Measured with FP32 x, cold-ish weights, us per call,
// prefill GEMM with its pre-pass (and sum) / this kernel (and sum):
//   K x N          5 rows        32 rows       64 rows       128 rows
//   1536 x 6144    21.6 /  7.1   22.1 / 11.4   22.1 / 13.2   22.8 / 17.9
//   1536 x 12288   21.5 /  8.3   22.2 / 13.0   22.4 / 18.0   (two rounds: 28 / 35)
//   6144 x 1536    24.1 /  9.7   24.8 / 14.0   25.3 / 16.0   26.7 / 20.6
//   12288 x 1536   32.0 / 11.9   33.3 / 17.1   33.8 / 22.1   (two rounds: 35 / 39)
//   1536 x 256     13.5 /  5.8   14.1 / 10.1   14.2 / 10.1   14.5 / 10.2
// Below 8 stages most waves have nothing to do, and tiles of 6 lose to the
// prefill GEMM (K 320 x N 4000, 128 rows: 9.7 / 10.2).
bool gemm_small_plan(const g4_w4 *const *w, int nw, int rows, bool glu, bool sum,
                     GemmSmallPlan *p) {
  if (rows < 2 || w[0]->G % 2 != 0) return false;
  for (int i = 0; i < nw; ++i)
    if (!w[i]->tiles) return false;
  const int cus = cu_count() > 0 ? cu_count() : 256;
  const int stages = w[0]->G / 2;
  p->tm = rows <= 16 ? 1 : 2;
  p->groups = (rows + 16 * p->tm - 1) / (16 * p->tm);
  // slices of K: a block's 8 waves hold 3 stages each where that divides K
  // evenly (E2B's widths but 2048 and 4096), else up to 4
  p->slices = stages % (3 * kWaves) == 0 ? stages / (3 * kWaves)
                                         : (stages + 4 * kWaves - 1) / (4 * kWaves);
  if (p->slices > 8 || (p->slices > 1 && ((nw > 1 && sum) || glu))) return false;
  p->per = (stages + p->slices - 1) / p->slices;
  p->s = p->per <= 3 * kWaves ? 3 : 4;
  for (int tn : {1, 2, 3, 6}) {
    if ((glu && tn % 2) || (tn > 3 && stages < kWaves)) continue;
    const int c = glu ? tn / 2 : tn;
    long blocks = 0;
    for (int i = 0; i < (glu ? 1 : nw); ++i) blocks += ((w[i]->N + 15) / 16 + c - 1) / c;
    p->tn = tn;
    if (blocks * p->slices * p->groups <= cus) return true;
  }
  return false;
}

int launch_gemm_small(const GemmSmallPlan &p, const g4_w4 *const *w, int nw, const void *x,
                      bool f32x, const uint4 *xt, const int *xe, int Mp, int rows, void *const *y,
                      bool y_bf16, float *part, size_t pstride, bool glu) {
  SmallArgs a{};
  a.x = x;
  a.xt = reinterpret_cast<const u32x4 *>(xt);
  a.xe = xe;
  a.Mp = Mp;
  a.n = nw;
  a.glu = glu;
  a.y_bf16 = y_bf16;
  a.rows = rows;
  a.K = w[0]->K;
  a.per = p.per;
  a.part = part;
  a.pstride = pstride;
  size_t off = 0;
  const int c = glu ? p.tn / 2 : p.tn;
  for (int i = 0; i < nw; ++i) {
    a.tw[i] = reinterpret_cast<const u32x4 *>(w[i]->tiles);
    a.y[i] = y[i];
    a.rs[i] = w[i]->row_shift ? w[i]->rshift : nullptr;
    a.N[i] = w[i]->N;
    a.shift[i] = w[i]->shift;
    a.t0[i + 1] = a.t0[i] + ((w[i]->N + 15) / 16 + c - 1) / c;
    a.poff[i] = off;
    off += (size_t)rows * w[i]->N;
  }
  const dim3 grid(glu ? a.t0[1] : a.t0[nw], p.slices, p.groups);
  if (!x) return launch_small<kXPrep>(a, p, grid);
  return f32x ? launch_small<kXF32>(a, p, grid) : launch_small<kXBf16>(a, p, grid);
}

}  // namespace g4

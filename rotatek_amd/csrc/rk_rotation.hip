// Top-k eigenbasis by truncated subspace iteration with Cholesky-QR
// orthonormalisation (rotation.py:21-91), for the 128 x 128 Key covariances
// of every (batch, KV head), k <= 128 (k <= 64 here; wider bases in
// power_iter128_kernel below).
//
// Per iteration, as the reference:
//   W = C V;  G = W^T W;  G += eps * mean(diag G) * I;  G = L L^T;  V = W L^-T
// One 256-thread workgroup owns one matrix.  C stays in registers, V^T, W^T,
// G, X = L^-1 and L in LDS (19 / 48 / 120 KB at KP = 16 / 32 / 64, so
// several matrices share a CU at KP <= 32).  The products run on
// v_mfma_f32_16x16x4_f32, 32 cycles each on the wave's SIMD, which bounds C V
// and the solve; each is formed transposed, so that the accumulators of one
// are the operands of the next:
//   W^T = V^T C^T      KP/16 x 8 tiles of 16 x 16, two columns of them a wave
//   G = W^T W          the lower tiles; those off the diagonal beside the
//                      first panel's elimination
//   Cholesky, L^-1     16-column panels: the diagonal block is inverted in
//                      wave 0 by DPP elimination (invert_block), the rest is
//                      MFMA products on waves 1-3 while wave 0 inverts the
//                      next one
//   V^T = X W^T        from W^T's registers
// Cycles of one iteration (wave 0, KP = 16 / 32 / 64): W 2400 / 4500 /
// 8800, diagonal of G 1400, ridge 350, panels 2100 / 5300 / 11900, V 360 /
// 950 / 2800.  32 matrices, 5 iterations: 26.4 -> 20.0 us at k = 16, 47.6 ->
// 34.5 at 32, 115 -> 65 at 64; 1024 matrices 109 -> 50, 194 -> 109, 455 -> 279.
// Padding columns of V are zero, so their rows and columns of G are too: a
// unit diagonal there makes that block the identity, and V keeps them zero.
// The start block V0 comes from the caller (the reference draws it with
// torch.randn from a seeded device generator, rotation.py:88-90).
#include <math.h>

#include <utility>

#include "rk_common.h"
#include "rk_host.h"
#include "rotatek_hip.h"

namespace rk {
namespace rot {

typedef __attribute__((address_space(3))) float lds_f32;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;

constexpr int kD = 128;
constexpr int kThreads = 256;

// D = A B + D on v_mfma_f32_16x16x4_f32 (A 16x4, B 4x16): lane (g, n) supplies
// A[n][g] and B[g][n] and holds D[4g + i][n], i = 0..3.
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 d) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, d, 0, 0, 0);
}

// The LDS address of p, through an empty asm the compiler cannot see into.
__device__ __forceinline__ lds_f32* opaque_lds(float* p) {
  unsigned a = (unsigned)(uintptr_t)(lds_f32*)p;
  asm volatile("" : "+v"(a));
  return (lds_f32*)(uintptr_t)a;
}

// LDS written and read within one wave: no barrier, but the compiler may
// not move the accesses across this point.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Lane J of each 16-lane row, in every lane of the row (DPP row_newbcast).
template <int J>
__device__ __forceinline__ float row_bcast(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + J, 0xf, 0xf, true));
}

// The sum over each 16-lane row, in every lane of the row (DPP rotations).
__device__ __forceinline__ float row_sum(float v) {
  auto rot = [](float x, auto ctrl) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  v += rot(v, std::integral_constant<int, 0x128>{});  // row_ror:8
  v += rot(v, std::integral_constant<int, 0x124>{});
  v += rot(v, std::integral_constant<int, 0x122>{});
  v += rot(v, std::integral_constant<int, 0x121>{});
  return v;
}
__device__ __forceinline__ float lane_value(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

// v += m * (v of lane J of the 16-lane row), for a group of registers.  As
// v_fmac_f32 with the DPP row broadcast on its first source: written out,
// since from the builtin the compiler keeps a v_mov_dpp per value, all
// through one register, with the two wait states a DPP read needs before
// each (3.1 against 2.8 us an iteration at k = 16).  The wait states stand
// around the group instead: in front for values that the instructions before
// may have written, behind for DPP reads of these results.  The instructions
// of a group do not depend on each other.
#define RK_F(d) "v_fmac_f32_dpp " d ", " d ", %[m] row_newbcast:%c[j] row_mask:0xf bank_mask:0xf\n\t"
#define RK_F4(d0, d1, d2, d3) RK_F(d0) RK_F(d1) RK_F(d2) RK_F(d3)
#define RK_V4(v) "+v"((v)[0]), "+v"((v)[1]), "+v"((v)[2]), "+v"((v)[3])
#define RK_F8 RK_F4("%0", "%1", "%2", "%3") RK_F4("%4", "%5", "%6", "%7")
#define RK_F12 RK_F8 RK_F4("%8", "%9", "%10", "%11")
#define RK_F16 RK_F12 RK_F4("%12", "%13", "%14", "%15")
#define RK_F20 RK_F16 RK_F4("%16", "%17", "%18", "%19")
// G0: the first group of four columns of a that still changes
template <int J, int G0>
__device__ __forceinline__ void fmac_bcast(float (&a)[16], float (&y)[4], float m) {
  if constexpr (G0 == 0)
    asm volatile("s_nop 1\n\t" RK_F20 "s_nop 1"
                 : RK_V4(a), RK_V4(a + 4), RK_V4(a + 8), RK_V4(a + 12), RK_V4(y)
                 : [m] "v"(m), [j] "n"(J));
  else if constexpr (G0 == 1)
    asm volatile("s_nop 1\n\t" RK_F16 "s_nop 1"
                 : RK_V4(a + 4), RK_V4(a + 8), RK_V4(a + 12), RK_V4(y)
                 : [m] "v"(m), [j] "n"(J));
  else if constexpr (G0 == 2)
    asm volatile("s_nop 1\n\t" RK_F12 "s_nop 1" : RK_V4(a + 8), RK_V4(a + 12), RK_V4(y) : [m] "v"(m), [j] "n"(J));
  else
    asm volatile("s_nop 1\n\t" RK_F8 "s_nop 1" : RK_V4(a + 12), RK_V4(y) : [m] "v"(m), [j] "n"(J));
}
#undef RK_F20
#undef RK_F16
#undef RK_F12
#undef RK_F8
#undef RK_V4
#undef RK_F4
#undef RK_F

// Step J of invert_block: subtract a_nJ / a_JJ times row J from the rows
// n > J, in the block (whole groups of four columns from J + 1 on: the
// columns up to J are not read again) and in the identity being turned
// into its inverse.
template <int J>
__device__ __forceinline__ void eliminate(float (&a)[16], float (&y)[4], float& own, int n, bool& bad) {
  const float piv = row_bcast<J>(a[J]);
  bad |= !__builtin_amdgcn_classf(piv, 0x180);  // positive, finite, not zero
  own = n == J ? piv : own;
  if constexpr (J < 15)  // no row follows the last
    fmac_bcast<J, (J + 1) / 4>(a, y, n > J ? -(a[J] * __builtin_amdgcn_rcpf(piv)) : 0.f);
}

template <int... J>
__device__ __forceinline__ void eliminate_all(float (&a)[16], float (&y)[4], float& own, int n, bool& bad,
                                              std::integer_sequence<int, J...>) {
  (eliminate<J>(a, y, own, n, bad), ...);
}

// X = L^-1 of a symmetric positive definite 16 x 16 block A = L L^T, in one
// wave: lane (g, n) brings row n (every g the same) and leaves with
// X[n][4 g + c], c = 0..3, which is the A operand of an MFMA over X's
// columns.  Gaussian elimination on [A | I]: A's rows in every 16-lane
// row, four columns of I each; the eliminated identity is D^1/2 X with D
// the pivots.  Rows are passed by DPP, so a step is a short chain (the
// pivot's broadcast, its reciprocal, the multiplier, the next pivot's
// update) with no LDS round trip; about 130 cycles a step, most of it the
// issue of its fused multiply-adds.
__device__ __forceinline__ f32x4 invert_block(float (&a)[16], int g, int n, bool& bad) {
  float y[4], own = 1.f;
#pragma unroll
  for (int c = 0; c < 4; ++c) y[c] = n == 4 * g + c ? 1.f : 0.f;
  eliminate_all(a, y, own, n, bad, std::make_integer_sequence<int, 16>{});
  const float r = __builtin_amdgcn_rsqf(own);
  return f32x4{y[0] * r, y[1] * r, y[2] * r, y[3] * r};
}

template <int KP>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(KP > 32 ? 1 : 2))) power_iter_kernel(
    const float* cov, int64_t c_sb, int64_t c_sh, int64_t c_sr, int64_t c_sc, const float* v0, int64_t v_sb,
    int64_t v_sh, int64_t v_sr, int64_t v_sc, float* out, int64_t o_sb, int64_t o_sh, int64_t o_sr,
    int64_t o_sc, int H, int k, int iters, float eps, int32_t* info, int cvec, int D) {
  constexpr int NT = KP / 16;  // 16-column tiles of V / W, 16-column panels of G
  // Row strides of 4 mod 16 floats: 16-byte reads of rows n = 0..15 at column
  // 4g, and accumulator writes of rows 4g + i at column n, cover all 64 banks
  constexpr int VS = kD + 4;
  constexpr int GS = KP + 4;
  __shared__ __align__(16) float sVt[KP * VS];  // V^T
  __shared__ __align__(16) float sWt[KP * VS];  // W^T
  __shared__ __align__(16) float sG[KP * GS];   // G, lower tiles
  __shared__ __align__(16) float sX[KP * GS];   // X = L^-1, lower tiles
  __shared__ __align__(16) float sL[NT > 1 ? KP * GS : 4];  // L, tiles below the diagonal

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, n = lane & 15;
  const int bh = blockIdx.x, b = bh / H, h = bh - b * H;
  const float* C = cov + b * c_sb + (int64_t)h * c_sh;
  const float* V0 = v0 + b * v_sb + (int64_t)h * v_sh;

  // C stays in registers over the iterations: wave w owns its row tiles 2w
  // and 2w + 1, lane (g, n) of k-group q the entries C[16 ti + n][16 q + 4 g + r].
  // With a head_dim D < 128 the rows and columns past D are zeros (their
  // loads re-read an in-bounds entry): W = C V, G, L and V = W L^-T then
  // equal the D x D iteration's, with exact zeros in the padded rows.
  f32x4 cf[2][8];
  if (cvec) {  // (D == 128, 16-byte rows)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int q = 0; q < 8; ++q)
        cf[t][q] = *(const f32x4*)(C + (int64_t)(16 * (2 * wave + t) + n) * c_sr + 16 * q + 4 * g);
  } else {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int row = 16 * (2 * wave + t) + n;
      const float* cr = C + (int64_t)min(row, D - 1) * c_sr;
#pragma unroll
      for (int q = 0; q < 8; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int col = 16 * q + 4 * g + r;
          const float x = cr[(int64_t)min(col, D - 1) * c_sc];
          cf[t][q][r] = row < D && col < D ? x : 0.f;
        }
    }
  }
  // V0 transposed into LDS, a batch of loads at a time
  constexpr int kVB = kD * KP / kThreads < 16 ? kD * KP / kThreads : 16;
  static_assert((kD * KP) % (kThreads * kVB) == 0, "whole batches");
  for (int e0 = 0; e0 < kD * KP; e0 += kThreads * kVB) {
    float v[kVB];
#pragma unroll
    for (int i = 0; i < kVB; ++i) {
      const int e = e0 + i * kThreads + tid, r = e / KP, c = e - r * KP;
      const float x = V0[min(r, D - 1) * v_sr + min(c, k - 1) * v_sc];
      v[i] = c < k && r < D ? x : 0.f;
    }
#pragma unroll
    for (int i = 0; i < kVB; ++i) {
      const int e = e0 + i * kThreads + tid, r = e / KP, c = e - r * KP;
      sVt[c * VS + r] = v[i];
    }
  }
  __syncthreads();

  bool bad = false;  // a pivot that is not positive and finite (wave 0)
  f32x4 vt[NT][2];   // V^T tiles (tj, 2w + t): lane (g, n) holds V^T[16 tj + 4 g + i][16 ti + n]
  if (iters == 0) {
#pragma unroll
    for (int tj = 0; tj < NT; ++tj)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) vt[tj][t][i] = sVt[(16 * tj + 4 * g + i) * VS + 16 * (2 * wave + t) + n];
  }

  for (int it = 0; it < iters; ++it) {
    // LDS bases, opaque to the compiler once per iteration: every access
    // below is one of these plus a lane part plus an immediate offset
    // (< 64 KB), so no per-access address is kept in a register across
    // iterations
    lds_f32* const lV = opaque_lds(sVt);
    lds_f32* const lW = opaque_lds(sWt);
    lds_f32* const lG = opaque_lds(sG);
    lds_f32* const lX = opaque_lds(sX);
    lds_f32* const lL = opaque_lds(sL);

    // ---- W^T = V^T C^T: the accumulators leave each lane with
    // W^T[16 tj + 4 g + i][16 ti + n], the B operand of the solve below
    f32x4 wt[NT][2];
#pragma unroll
    for (int tj = 0; tj < NT; ++tj) wt[tj][0] = wt[tj][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < kD / 16; ++q) {
      f32x4 a[NT];
#pragma unroll
      for (int tj = 0; tj < NT; ++tj) a[tj] = *(const lds_f32x4*)&lV[(16 * tj + n) * VS + 16 * q + 4 * g];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int tj = 0; tj < NT; ++tj)
#pragma unroll
          for (int t = 0; t < 2; ++t) wt[tj][t] = mfma4(a[tj][r], cf[t][q][r], wt[tj][t]);
    }
#pragma unroll
    for (int tj = 0; tj < NT; ++tj)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) lW[(16 * tj + 4 * g + i) * VS + 16 * (2 * wave + t) + n] = wt[tj][t][i];
    __syncthreads();

    // ---- G = W^T W: the diagonal tiles now, one to a wave; the others
    // below the diagonal by waves 1-3 while wave 0 eliminates the first
    // panel, which needs only the diagonal.  Two accumulators per tile so
    // consecutive MFMAs do not wait on each other.
    auto g_tile = [&](int ti, int tj) {
      f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int q = 0; q < kD / 16; ++q) {
        const f32x4 av = *(const lds_f32x4*)&lW[(16 * tj + n) * VS + 16 * q + 4 * g];
        const f32x4 bv = ti == tj ? av : *(const lds_f32x4*)&lW[(16 * ti + n) * VS + 16 * q + 4 * g];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r & 1] = mfma4(av[r], bv[r], acc[r & 1]);
      }
      *(lds_f32x4*)&lG[(16 * ti + n) * GS + 16 * tj + 4 * g] = acc[0] + acc[1];
    };
#pragma unroll
    for (int ti = 0; ti < NT; ++ti)
      if (wave == ti) g_tile(ti, ti);
    __syncthreads();

    // ---- ridge: G += eps * mean(diag G) * I (wave 0); the padding rows and
    // columns of G are zero (V's padding columns are): a unit diagonal there
    // makes them the identity
    if (wave == 0) {
      const int lr = min(lane, KP - 1);
      const float dii = lG[lr * GS + lr];
      const float dg = row_sum(lane < k ? dii : 0.f);
      float tr = lane_value(dg, 0);
#pragma unroll
      for (int t = 1; t < NT; ++t) tr += lane_value(dg, 16 * t);
      const float ridge = eps * (tr / (float)k);
      if (lane < KP) lG[lane * GS + lane] = lane < k ? dii + ridge : 1.f;
    } else {
      int t = 0;
#pragma unroll
      for (int ti = 1; ti < NT; ++ti)
#pragma unroll
        for (int tj = 0; tj < ti; ++tj)
          if (t++ % 3 == wave - 1) g_tile(ti, tj);
    }

    // ---- blocked Cholesky G = L L^T and X = L^-1 over 16-column panels,
    // one barrier per panel.  Wave 0 eliminates panel p's diagonal block
    // (X_pp = L_pp^-1) and publishes it; then it alone prepares the next
    // diagonal block and eliminates that, while waves 1-3 update the other
    // trailing tiles G_ij -= L_ip L_jp^T and form row p of X,
    // X_pr = -X_pp sum_{s=r}^{p-1} L_ps X_sr.  L_qp = G_qp X_pp^T is formed
    // by every wave that needs it, transposed (X_pp G_qp^T), so that the
    // accumulators are the operands of the next product.
#pragma unroll
    for (int p = 0; p < NT; ++p) {
      if (wave == 0) {
        wave_lds_fence();
        float a[16];
#pragma unroll
        for (int c4 = 0; c4 < 4; ++c4) {
          const f32x4 v = *(const lds_f32x4*)&lG[(16 * p + n) * GS + 16 * p + 4 * c4];
#pragma unroll
          for (int i = 0; i < 4; ++i) a[4 * c4 + i] = v[i];
        }
        *(lds_f32x4*)&lX[(16 * p + n) * GS + 16 * p + 4 * g] = invert_block(a, g, n, bad);
      }
      __syncthreads();
      const f32x4 xp = *(const lds_f32x4*)&lX[(16 * p + n) * GS + 16 * p + 4 * g];
      auto l_t = [&](int q) {  // L_qp[n][4 g + i]
        const f32x4 gq = *(const lds_f32x4*)&lG[(16 * q + n) * GS + 16 * p + 4 * g];
        f32x4 d = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; ++r) d = mfma4(xp[r], gq[r], d);
        return d;
      };
      auto update = [&](int ti, int tj) {  // G_ij -= L_ip L_jp^T; a diagonal tile's wave keeps L_ip
        const f32x4 li = l_t(ti);
        const f32x4 lj = ti == tj ? li : l_t(tj);
        f32x4 d = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; ++r) d = mfma4(lj[r], li[r], d);
        lds_f32x4* pg = (lds_f32x4*)&lG[(16 * ti + n) * GS + 16 * tj + 4 * g];
        *pg = *pg - d;
        if (ti == tj) *(lds_f32x4*)&lL[(16 * ti + n) * GS + 16 * p + 4 * g] = li;
      };
      auto x_tile = [&](int r) {  // X_pr
        f32x4 s_acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NT - 1; ++s) {
          if (s >= r && s < p) {
            const f32x4 lv = *(const lds_f32x4*)&lL[(16 * p + n) * GS + 16 * s + 4 * g];
#pragma unroll
            for (int i = 0; i < 4; ++i)
              s_acc = mfma4(lv[i], lX[(16 * s + 4 * g + i) * GS + 16 * r + n], s_acc);
          }
        }
        f32x4 d = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) d = mfma4(xp[i], s_acc[i], d);
#pragma unroll
        for (int i = 0; i < 4; ++i) lX[(16 * p + 4 * g + i) * GS + 16 * r + n] = -d[i];
      };
      if (p + 1 < NT) {
        if (wave == 0) {
          update(p + 1, p + 1);
        } else {
          int t = 0;
#pragma unroll
          for (int ti = p + 1; ti < NT; ++ti)
#pragma unroll
            for (int tj = p + 1; tj <= ti; ++tj) {
              if (ti == p + 1 && tj == p + 1) continue;
              if (t++ % 3 == wave - 1) update(ti, tj);
            }
#pragma unroll
          for (int r = 0; r < p; ++r)
            if (t++ % 3 == wave - 1) x_tile(r);
        }
      } else if (p > 0) {
#pragma unroll
        for (int r = 0; r < p; ++r)
          if (r % 4 == wave) x_tile(r);
        __syncthreads();
      }
    }

    // ---- V^T = X W^T (X lower triangular): tile (tj, ti) over q <= tj, W^T
    // from the registers it was formed in
#pragma unroll
    for (int tj = 0; tj < NT; ++tj) {
      vt[tj][0] = vt[tj][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q <= tj; ++q) {
        const f32x4 xa = *(const lds_f32x4*)&lX[(16 * tj + n) * GS + 16 * q + 4 * g];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int t = 0; t < 2; ++t) vt[tj][t] = mfma4(xa[r], wt[q][t][r], vt[tj][t]);
      }
    }
    if (it + 1 < iters) {
#pragma unroll
      for (int tj = 0; tj < NT; ++tj)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) lV[(16 * tj + 4 * g + i) * VS + 16 * (2 * wave + t) + n] = vt[tj][t][i];
      __syncthreads();
    }
  }

  if (info && tid == 0) info[bh] = bad ? 1 : 0;  // thread 0 is in wave 0, which ran the pivots
  float* O = out + b * o_sb + (int64_t)h * o_sh;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int row = 16 * (2 * wave + t) + n;
    if (row < D) {
#pragma unroll
      for (int tj = 0; tj < NT; ++tj)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (16 * tj + 4 * g + i < k) O[row * o_sr + (16 * tj + 4 * g + i) * o_sc] = vt[tj][t][i];
    }
  }
}

// ---- 64 < k <= 128.  C, V/W, G, L and L^-1 do not all fit in LDS at this
// width, so C is read from global memory (each matrix's 64 KB stays in its
// XCD's L2 across the iterations) and G, L and X = L^-1 share one array:
//   strict lower triangle  L (rows below the diagonal)
//   diagonal               r_j = 1 / L_jj (= X_jj)
//   strict upper triangle  X^T (X is lower triangular)
// The Cholesky is blocked by 16-column panels as at k = 64 (wave 0 factors
// a panel with two rows per lane; all waves apply the trailing update on
// the MFMA), X's off-diagonal blocks follow by block rows, and V = W X^T
// reads X^T from the upper triangle (masked to zero below it).
constexpr int kW = 128;       // padded basis width
constexpr int kWS = kW + 4;   // V / W row stride
constexpr int kWG = kW + 1;   // G row stride

// X^T[m][j] from the packed array (zero below the diagonal, where L lives)
__device__ __forceinline__ float xt_at(const lds_f32* P, int m, int j) {
  const float v = P[m * kWG + j];
  return m <= j ? v : 0.f;
}

__global__ void __launch_bounds__(kThreads) power_iter128_kernel(
    const float* cov, int64_t c_sb, int64_t c_sh, int64_t c_sr, int64_t c_sc, const float* v0, int64_t v_sb,
    int64_t v_sh, int64_t v_sr, int64_t v_sc, float* out, int64_t o_sb, int64_t o_sh, int64_t o_sr,
    int64_t o_sc, int H, int k, int iters, float eps, int32_t* info, int cvec, int D) {
  __shared__ __align__(16) float sV[kD * kWS];
  __shared__ __align__(16) float sP[kW * kWG];
  __shared__ float sT[4 * 256];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, n = lane & 15;
  const int bh = blockIdx.x, b = bh / H, h = bh - b * H;
  const float* C = cov + b * c_sb + (int64_t)h * c_sh;
  const float* V0 = v0 + b * v_sb + (int64_t)h * v_sh;
  constexpr int kB = 16;
  for (int e0 = 0; e0 < kD * kW; e0 += kThreads * kB) {
    float v[kB];
#pragma unroll
    for (int i = 0; i < kB; ++i) {
      const int e = e0 + i * kThreads + tid, r = e >> 7, c = e & 127;
      v[i] = c < k && r < D ? V0[r * v_sr + c * v_sc] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < kB; ++i) {
      const int e = e0 + i * kThreads + tid;
      sV[(e >> 7) * kWS + (e & 127)] = v[i];
    }
  }
  __syncthreads();
  bool bad = false;
  lds_f32* const lV = (lds_f32*)sV;
  lds_f32* const lP = (lds_f32*)sP;
  lds_f32* const lT = (lds_f32*)sT + wave * 256;
  const int tjw = 2 * wave;  // this wave's output column tiles in C V and W X^T: tjw, tjw + 1

  for (int it = 0; it < iters; ++it) {
    // ---- W = C V: tiles (ti, tjw + t2), ti = 0..7; in k-group q lane (g, n)
    // supplies k = 16 q + 4 g + r (one 16-byte read of C's row feeds four steps)
    {
      f32x4 acc[8][2];
#pragma unroll
      for (int ti = 0; ti < 8; ++ti) acc[ti][0] = acc[ti][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int q = 0; q < kD / 16; ++q) {
        float a[8][4];
#pragma unroll
        for (int ti = 0; ti < 8; ++ti) {
          if (cvec) {  // (D == 128)
            const float* cr = C + (int64_t)(16 * ti + n) * c_sr;
            const float4 v = *(const float4*)(cr + 16 * q + 4 * g);
            a[ti][0] = v.x, a[ti][1] = v.y, a[ti][2] = v.z, a[ti][3] = v.w;
          } else {  // rows and columns of C past D are zeros
            const int row = 16 * ti + n;
            const float* cr = C + (int64_t)min(row, D - 1) * c_sr;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int col = 16 * q + 4 * g + r;
              const float x = cr[(int64_t)min(col, D - 1) * c_sc];
              a[ti][r] = row < D && col < D ? x : 0.f;
            }
          }
        }
        float bv[2][4];
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
          for (int r = 0; r < 4; ++r) bv[t2][r] = lV[(16 * q + 4 * g + r) * kWS + 16 * (tjw + t2) + n];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int ti = 0; ti < 8; ++ti)
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2) acc[ti][t2] = mfma4(a[ti][r], bv[t2][r], acc[ti][t2]);
      }
      __syncthreads();
#pragma unroll
      for (int ti = 0; ti < 8; ++ti)
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
          for (int i = 0; i < 4; ++i) lV[(16 * ti + 4 * g + i) * kWS + 16 * (tjw + t2) + n] = acc[ti][t2][i];
    }
    __syncthreads();

    // ---- G = W^T W, the 36 lower tiles (ti >= tj), tile t to wave t mod 4
    {
      int t = 0;
      for (int ti = 0; ti < 8; ++ti) {
        for (int tj = 0; tj <= ti; ++tj, ++t) {
          if (t % 4 != wave) continue;  // wave-uniform
          f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
          for (int q = 0; q < kD / 4; ++q)
            acc = mfma4(lV[(4 * q + g) * kWS + 16 * ti + n], lV[(4 * q + g) * kWS + 16 * tj + n], acc);
#pragma unroll
          for (int i = 0; i < 4; ++i) lP[(16 * ti + 4 * g + i) * kWG + 16 * tj + n] = acc[i];
        }
      }
    }
    __syncthreads();

    // ---- ridge: G += eps * mean(diag G) * I over the first k; padding
    // rows and columns are zero (V's padding columns are): unit diagonal
    if (wave == 0) {
      const float d0 = lP[lane * kWG + lane], d1 = lP[(lane + 64) * kWG + lane + 64];
      float dg = (lane < k ? d0 : 0.f) + (lane + 64 < k ? d1 : 0.f);
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) dg += shfl_xor(dg, off);
      const float ridge = eps * (dg / (float)k);
      lP[lane * kWG + lane] = lane < k ? d0 + ridge : 1.f;
      lP[(lane + 64) * kWG + lane + 64] = lane + 64 < k ? d1 + ridge : 1.f;
    }
    __syncthreads();

    // ---- blocked Cholesky and the diagonal blocks of X
    for (int p = 0; p < kW / 16; ++p) {
      const int P0 = 16 * p;
      if (wave == 0) {
        // lane holds rows lane and lane + 64 (entries of panel columns P0..P0+15)
        float a0[16], a1[16], lc0[16], lc1[16], xv[16];
        const bool hi = P0 >= 64;  // the panel's rows sit in the second half
        const int prow = (hi ? lane + 64 : lane);  // the half whose lanes hold the panel rows
#pragma unroll
        for (int c = 0; c < 16; ++c) {
          a0[c] = lP[lane * kWG + P0 + c];
          a1[c] = lP[(lane + 64) * kWG + P0 + c];
          xv[c] = prow == P0 + c ? 1.f : 0.f;
        }
#pragma unroll
        for (int jj = 0; jj < 16; ++jj) {
          const int j = P0 + jj;
          const float pv = hi ? a1[jj] : a0[jj];
          const float piv = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, pv), j & 63));
          bad |= !(piv > 0.f && piv <= 3.402823466e38f);
          const float rj = __builtin_amdgcn_rsqf(piv);
          const float l0 = lane > j ? a0[jj] * rj : (lane == j ? rj : 0.f);
          const float l1 = lane + 64 > j ? a1[jj] * rj : (lane + 64 == j ? rj : 0.f);
          lc0[jj] = l0;
          lc1[jj] = l1;
          xv[jj] *= rj;
          const float lp = hi ? l1 : l0;  // column j of L in the panel rows' half
#pragma unroll
          for (int mm = jj + 1; mm < 16; ++mm) {
            const float c = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, lp), (P0 + mm) & 63));
            a0[mm] = fmaf(-l0, c, a0[mm]);
            a1[mm] = fmaf(-l1, c, a1[mm]);
            xv[mm] = fmaf(-c, xv[jj], xv[mm]);
          }
        }
        // L (lower triangle and diagonal) in place of G
#pragma unroll
        for (int jj = 0; jj < 16; ++jj) {
          if (lane >= P0 + jj) lP[lane * kWG + P0 + jj] = lc0[jj];
          if (lane + 64 >= P0 + jj) lP[(lane + 64) * kWG + P0 + jj] = lc1[jj];
        }
        // X's diagonal block, transposed into the upper triangle: row prow
        // of X^T holds column prow of X (lanes whose row is in the panel)
        if (prow >= P0 && prow < P0 + 16) {
#pragma unroll
          for (int mm = 0; mm < 16; ++mm)
            if (P0 + mm > prow) lP[prow * kWG + P0 + mm] = xv[mm];
        }
      }
      __syncthreads();
      if (p + 1 < kW / 16) {
        // G[16 ti + a][16 tj + b] -= sum_c L[16 ti + a][P0 + c] L[16 tj + b][P0 + c], p < tj <= ti
        int t = 0;
        for (int ti = p + 1; ti < kW / 16; ++ti) {
          for (int tj = p + 1; tj <= ti; ++tj, ++t) {
            if (t % 4 != wave) continue;  // wave-uniform
            f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < 4; ++st) {
              const int cc = P0 + 4 * st + g;
              acc = mfma4(lP[(16 * ti + n) * kWG + cc], lP[(16 * tj + n) * kWG + cc], acc);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) lP[(16 * ti + 4 * g + i) * kWG + 16 * tj + n] -= acc[i];
          }
        }
        __syncthreads();
      }
    }

    // ---- X's blocks below the diagonal by block rows q:
    // X_qr = -X_qq sum_{s=r}^{q-1} L_qs X_sr, stored transposed in the upper triangle
    for (int q = 1; q < kW / 16; ++q) {
      for (int r = wave; r < q; r += 4) {  // wave-uniform
        f32x4 tacc = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int kk0 = 16 * r; kk0 < 16 * q; kk0 += 4) {
          const int kk = kk0 + g;
          tacc = mfma4(lP[(16 * q + n) * kWG + kk], xt_at(lP, 16 * r + n, kk), tacc);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) lT[(4 * g + i) * 16 + n] = tacc[i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        f32x4 xacc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          const int kk = 4 * st + g;
          xacc = mfma4(xt_at(lP, 16 * q + kk, 16 * q + n), lT[kk * 16 + n], xacc);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int i = 0; i < 4; ++i) lP[(16 * r + n) * kWG + 16 * q + 4 * g + i] = -xacc[i];
      }
      __syncthreads();
    }

    // ---- V = W X^T: V[r][j] = sum_{m <= j} W[r][m] X^T[m][j], tiles (ti, tjw + t2)
    {
      f32x4 acc[8][2];
#pragma unroll
      for (int ti = 0; ti < 8; ++ti) acc[ti][0] = acc[ti][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int q = 0; q <= tjw + 1; ++q) {  // k-blocks of 16 up to the wave's last column tile
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          const int m = 16 * q + 4 * st + g;
          float bv[2];
#pragma unroll
          for (int t2 = 0; t2 < 2; ++t2) bv[t2] = xt_at(lP, m, 16 * (tjw + t2) + n);
#pragma unroll
          for (int ti = 0; ti < 8; ++ti) {
            const float av = lV[(16 * ti + n) * kWS + m];
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2) acc[ti][t2] = mfma4(av, bv[t2], acc[ti][t2]);
          }
        }
      }
      __syncthreads();
#pragma unroll
      for (int ti = 0; ti < 8; ++ti)
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
          for (int i = 0; i < 4; ++i) lV[(16 * ti + 4 * g + i) * kWS + 16 * (tjw + t2) + n] = acc[ti][t2][i];
    }
    __syncthreads();
  }

  if (info && tid == 0) info[bh] = bad ? 1 : 0;
  float* O = out + b * o_sb + (int64_t)h * o_sh;
  for (int e = tid; e < D * k; e += kThreads) {
    const int r = e / k, c = e - (e / k) * k;
    O[r * o_sr + c * o_sc] = sV[r * kWS + c];
  }
}

template <int KP>
hipError_t launch(const rk_tensor* cov, const rk_tensor* v0, const rk_tensor* out, int64_t BH, int H, int k,
                  int iters, float eps, int32_t* info, int cvec, int D, hipStream_t s) {
  hipLaunchKernelGGL((power_iter_kernel<KP>), dim3((unsigned)BH), dim3(kThreads), 0, s, (const float*)cov->data,
                     cov->stride[0], cov->stride[1], cov->stride[2], cov->stride[3], (const float*)v0->data,
                     v0->stride[0], v0->stride[1], v0->stride[2], v0->stride[3], (float*)out->data, out->stride[0],
                     out->stride[1], out->stride[2], out->stride[3], H, k, iters, eps, info, cvec, D);
  return hipGetLastError();
}

}  // namespace rot
}  // namespace rk

extern "C" int rk_power_iteration(const rk_tensor* cov, const rk_tensor* v0, const rk_tensor* out,
                                  int32_t num_iters, float eps, int32_t* info, void* stream) {
  using namespace rk::rot;
  if (!cov || !v0 || !out) return RK_ERR_NULL;
  int st;
  if ((st = rk::check_desc(cov, 4)) || (st = rk::check_desc(v0, 4)) || (st = rk::check_desc(out, 4))) return st;
  if (cov->dtype != RK_F32 || v0->dtype != RK_F32 || out->dtype != RK_F32) return RK_ERR_DTYPE;
  // any head_dim D <= 128 (rotation.py:86-91 takes D = cov.shape[-1])
  const int64_t D = cov->shape[2];
  if (D < 1 || D > kD || cov->shape[3] != D) return RK_ERR_HEAD_DIM;
  const int64_t B = cov->shape[0], H = cov->shape[1], k = v0->shape[3];
  for (const rk_tensor* t : {v0, out})
    if (t->shape[0] != B || t->shape[1] != H || t->shape[2] != D || t->shape[3] != k) return RK_ERR_SHAPE;
  if (k < 1 || k > D) return RK_ERR_KEEP_DIM;
  if (num_iters < 0 || !(eps >= 0.f)) return RK_ERR_ARG;
  if (B * H == 0) return RK_OK;
  if (B * H > (INT64_C(1) << 31) || H > (INT64_C(1) << 30)) return RK_ERR_SHAPE;
  if (!cov->data || !v0->data || !out->data) return RK_ERR_NULL;
  hipStream_t s = (hipStream_t)stream;
  hipError_t e;
  // 16-byte loads of whole rows of C
  const int cvec = D == kD && cov->stride[3] == 1 && cov->stride[2] % 4 == 0 && cov->stride[1] % 4 == 0 &&
                   cov->stride[0] % 4 == 0 && (((uintptr_t)cov->data) & 15) == 0;
  if (k <= 16)
    e = launch<16>(cov, v0, out, B * H, (int)H, (int)k, num_iters, eps, info, cvec, (int)D, s);
  else if (k <= 32)
    e = launch<32>(cov, v0, out, B * H, (int)H, (int)k, num_iters, eps, info, cvec, (int)D, s);
  else if (k <= 64)
    e = launch<64>(cov, v0, out, B * H, (int)H, (int)k, num_iters, eps, info, cvec, (int)D, s);
  else {
    hipLaunchKernelGGL(power_iter128_kernel, dim3((unsigned)(B * H)), dim3(kThreads), 0, s, (const float*)cov->data,
                       cov->stride[0], cov->stride[1], cov->stride[2], cov->stride[3], (const float*)v0->data,
                       v0->stride[0], v0->stride[1], v0->stride[2], v0->stride[3], (float*)out->data,
                       out->stride[0], out->stride[1], out->stride[2], out->stride[3], (int)H, (int)k, num_iters, eps,
                       info, cvec, (int)D);
    e = hipGetLastError();
  }
  return e == hipSuccess ? RK_OK : RK_ERR_HIP;
}

// Dense layers on the fp32 matrix cores with the passes around them fused into
// the epilogue: C[M, N] = epi(A[M, K] B[N, K]^T), A and B row-major with K
// contiguous (torch Linear's in W^T; a backward in_adj = out_adj W uses W's
// transposed copy, so every GEMM has this one form).
//
// Epilogue, per element (i, j) in this order:
//   v = acc                                  (the product, fp32, fixed k order)
//   v = v * row_scale[i]                     (a row scale: RMSNorm's 1/rms, its weight folded into B)
//   v = v + bias[j]
//   v = v + beta * C_in[i, j]                (a residual, C_in may be C itself)
//   pre[i, j] = v                            (kept for a backward, when asked)
//   v = act(v)                               (SiLU, or SwiGLU on (v_2c, g_2c+1) pairs to column c)
// so the bias fills, residual sums and activation passes of the model need no
// memory round trip of their own.
//
// Tiling for gfx950: a 256-thread workgroup (4 waves in 2 x 2) computes a BM x BN
// tile, each wave (BM/2) x (BN/2) in 16 x 16 v_mfma_f32_16x16x4_f32 tiles. The
// K loop steps 16 at a time through LDS, double-buffered: each thread loads the
// next step's A and B slices into registers before the current step's MFMAs and
// stores them to the other buffer after, one barrier a step. Within a step the
// four MFMA k-slices take k = 4g + s (lane group g, slice s), so a lane reads
// one contiguous float4 of an A row and of a B row per 16 x 16 tile (the sum's
// order is fixed: results repeat bit for bit).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <atomic>
#include <mutex>
#include <type_traits>
#include <cstdlib>

#include "../../include/pet_model.h"
#include "gemm_common.h"
#include "split_bf16.h"

namespace pet_gemm {

using pet_split::mfma6;
using pet_split::pack_hi;
using pet_split::split3;
using pet_split::split8;
using pet_split::pair2;
using pet_split::pair_scale;

__device__ __forceinline__ f4 mfma(float a, float b, const f4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
std::atomic<uint64_t> g_flops[4];

// The epilogue of one result element v at (i, j), shared by the kernels. Every
// lane of the wave calls it together (SwiGLU pairs neighbouring lanes):
// (i, j) may lie outside the result, which is then left alone.
__device__ __forceinline__ void epi_elem(float v, int i, int j, int c, int M, int N, float* C, int64_t ldc,
                                         const Epi& epi) {
  if (epi.act >= 3) {
    // v is an activation's output adjoint; cin the saved pre-activation
    // (bias the pre-activation's bias, null when cin holds it already).
    // 3: C[i, j] = v silu'(z); 4 (SwiGLU, (value, gate) pairs of cin):
    // C[i, 2j] = v sigmoid(g), C[i, 2j + 1] = v u sigmoid(g) (1 - sigmoid(g))
    if (i >= M || j >= N) return;
    const float* z = epi.cin + int64_t(i) * epi.ldcin;
    if (epi.act == 3) {
      const float x = z[j] + (epi.bias ? epi.bias[j] : 0.f), sg = sig_fast(x);
      C[int64_t(i) * ldc + j] = v * (sg * (1.0f + x * (1.0f - sg)));
    } else {
      const float u = z[2 * j] + (epi.bias ? epi.bias[2 * j] : 0.f);
      const float sg = sig_fast(z[2 * j + 1] + (epi.bias ? epi.bias[2 * j + 1] : 0.f));
      *reinterpret_cast<float2*>(C + int64_t(i) * ldc + 2 * j) = make_float2(v * sg, v * u * sg * (1.0f - sg));
    }
    return;
  }
  if (epi.row_scale && i < M) v *= epi.row_scale[i];
  if (epi.bias && j < N) v += epi.bias[j];
  if (epi.cin && i < M && j < N) v += epi.beta * epi.cin[int64_t(i) * epi.ldcin + j];
  if (epi.pre && i < M && j < N) epi.pre[int64_t(i) * epi.ldpre + j] = v;
  if (epi.act == 2) {
    // SwiGLU: columns 2c' (value) and 2c'+1 (gate) sit in lanes c and c + 1
    const float gate = __shfl_down(v, 1, 16);
    if ((c & 1) == 0 && i < M && j < N) C[int64_t(i) * ldc + j / 2] = v * sig_fast(gate);
  } else if (i < M && j < N) {
    C[int64_t(i) * ldc + j] = epi.act == 1 ? v * sig_fast(v) : v;
  }
}
// The tile kernels' epilogue: lane (c, g) of tile (a, b) holds rows 4g + r,
// column c of the wave's WM x WN share.
template <int WM, int WN>
__device__ __forceinline__ void epilogue(const f4 (&acc)[WM / 16][WN / 16], int m0, int n0, int wm, int wn, int c,
                                         int g, int M, int N, float* C, int64_t ldc, const Epi& epi) {
  constexpr int TM = WM / 16, TN = WN / 16;
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        epi_elem(acc[a][b][r], m0 + wm * WM + 16 * a + 4 * g + r, n0 + wn * WN + 16 * b + c, c, M, N, C, ldc, epi);
}

// The epilogue through LDS, for a tile whose columns all lie in the result:
// the waves' results (already unscaled) go to a BM x BN fp32 tile in LDS
// (float4 slot q of row R at q ^ s(R), s(R) = 4 (R / 4) mod BN / 4, so the
// four row groups of a store fall on distinct banks), then each thread takes
// float4 runs of a row and applies epi_elem's arithmetic, in its order, with
// 16-byte loads and stores (C, pre, cin, bias) in place of a wave's 4-byte
// stores to four rows. False (nothing written) where a pointer or leading
// dimension does not allow the 16-byte accesses; the caller then uses
// epilogue(). tile: BM BN floats of LDS no wave still reads.
template <int BM, int BN, int WGM, int WGN, int PASSES = 1>
__device__ __forceinline__ bool staged_epilogue(const f4 (&acc)[BM / WGM / 16][BN / WGN / 16], float* tile, int m0,
                                                int n0, int M, int N, float* C, int64_t ldc, const Epi& epi) {
  constexpr int T = 64 * WGM * WGN, WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16, F = BN / 4;
  constexpr int RB = BM / PASSES;  // the tile's rows a pass (the rows of WGM / PASSES wave rows)
  static_assert(T % F == 0 && WGM % PASSES == 0, "whole rows a pass, whole wave rows a pass");
  auto a16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const bool act4 = epi.act == 4, act2 = epi.act == 2;
  // C's columns: 2 N (act 4), N / 2 (act 2), else N; j stays a multiple of 4
  const bool ok = n0 + BN <= N && a16(C) && ldc % 4 == 0 && (!epi.bias || a16(epi.bias)) &&
                  (!epi.cin || (a16(epi.cin) && epi.ldcin % 4 == 0)) && (!epi.pre || (a16(epi.pre) && epi.ldpre % 4 == 0));
  if (!ok) return false;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, c = l & 15, g = l >> 4;
  const int wm = w / WGN, wn = w % WGN;
  auto slot = [](int R, int q) { return R * BN + 4 * (q ^ ((4 * (R >> 2)) & (F - 1))); };
  const int q = tid % F;
  const int j = n0 + 4 * q;
  // a thread's NO outputs of row i from output column jo on
  auto put = [&](int i, int jo, const float* o, auto no_c) {
    constexpr int NO = decltype(no_c)::value;
    float* dst = C + int64_t(i) * ldc + jo;
    if constexpr (NO == 2) *reinterpret_cast<float2*>(dst) = make_float2(o[0], o[1]);
    if constexpr (NO >= 4) *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
    if constexpr (NO == 8) *reinterpret_cast<float4*>(dst + 4) = make_float4(o[4], o[5], o[6], o[7]);
  };
  using c2 = std::integral_constant<int, 2>;
  using c4 = std::integral_constant<int, 4>;
  using c8 = std::integral_constant<int, 8>;
  float4 bj = make_float4(0.f, 0.f, 0.f, 0.f), bj2 = bj;
  if (epi.bias) {
    if (act4) {
      bj = *reinterpret_cast<const float4*>(epi.bias + 2 * j);
      bj2 = *reinterpret_cast<const float4*>(epi.bias + 2 * j + 4);
    } else {
      bj = *reinterpret_cast<const float4*>(epi.bias + j);
    }
  }
  for (int h = 0; h < PASSES; ++h) {
  __syncthreads();  // every wave done with the LDS the tile reuses
  if (wm / (WGM / PASSES) == h) {
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TN; ++b)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int R = wm * WM + 16 * a + 4 * g + rr - h * RB, Cc = wn * WN + 16 * b + c;
          tile[slot(R, Cc >> 2) + (Cc & 3)] = acc[a][b][rr];
        }
  }
  __syncthreads();
  for (int R = tid / F; R < RB; R += T / F) {
    const int i = m0 + h * RB + R;
    if (i >= M) break;
    const float4 t4 = *reinterpret_cast<const float4*>(tile + slot(R, q));
    float v[4] = {t4.x, t4.y, t4.z, t4.w};
    if (epi.act >= 3) {
      const float* z = epi.cin + int64_t(i) * epi.ldcin;
      if (!act4) {
        const float4 z4 = *reinterpret_cast<const float4*>(z + j);
        const float zz[4] = {z4.x, z4.y, z4.z, z4.w}, bb[4] = {bj.x, bj.y, bj.z, bj.w};
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = zz[e] + (epi.bias ? bb[e] : 0.f), sg = sig_fast(x);
          o[e] = v[e] * (sg * (1.0f + x * (1.0f - sg)));
        }
        put(i, j, o, c4{});
      } else {
        const float4 z0 = *reinterpret_cast<const float4*>(z + 2 * j), z1 = *reinterpret_cast<const float4*>(z + 2 * j + 4);
        const float zz[8] = {z0.x, z0.y, z0.z, z0.w, z1.x, z1.y, z1.z, z1.w};
        const float bb[8] = {bj.x, bj.y, bj.z, bj.w, bj2.x, bj2.y, bj2.z, bj2.w};
        float o[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float u = zz[2 * e] + (epi.bias ? bb[2 * e] : 0.f);
          const float sg = sig_fast(zz[2 * e + 1] + (epi.bias ? bb[2 * e + 1] : 0.f));
          o[2 * e] = v[e] * sg, o[2 * e + 1] = v[e] * u * sg * (1.0f - sg);
        }
        put(i, 2 * j, o, c8{});
      }
      continue;
    }
    if (epi.row_scale) {
      const float rs = epi.row_scale[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= rs;
    }
    if (epi.bias) v[0] += bj.x, v[1] += bj.y, v[2] += bj.z, v[3] += bj.w;
    if (epi.cin) {
      const float4 c4 = *reinterpret_cast<const float4*>(epi.cin + int64_t(i) * epi.ldcin + j);
      v[0] += epi.beta * c4.x, v[1] += epi.beta * c4.y, v[2] += epi.beta * c4.z, v[3] += epi.beta * c4.w;
    }
    if (epi.pre) *reinterpret_cast<float4*>(epi.pre + int64_t(i) * epi.ldpre + j) = make_float4(v[0], v[1], v[2], v[3]);
    if (act2) {
      const float o[2] = {v[0] * sig_fast(v[1]), v[2] * sig_fast(v[3])};
      put(i, j / 2, o, c2{});
    } else {
      if (epi.act == 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] * sig_fast(v[e]);
      put(i, j, v, c4{});
    }
  }
  }
  return true;
}

template <int BM, int BN, int BK = 32>
__global__ void __launch_bounds__(256) gemm_nt_kernel(int M, int N, int K, const float* __restrict__ A, int64_t lda,
                                                      const float* __restrict__ B, int64_t ldb, float* C, int64_t ldc,
                                                      Epi epi) {
  constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 16, TN = WN / 16, PK = BK + 4, Q4 = BK / 4;
  // float4 slots of a step's A / B slice (4 a row), and a thread's share
  constexpr int AQ = BM * BK / 4, BQ = BN * BK / 4, AL = (AQ + 255) / 256, BL = (BQ + 255) / 256;
  __shared__ float lds_ab[2 * (BM + BN) * PK];  // both buffers of A's and B's slices, one array
  float (*const As)[BM * PK] = reinterpret_cast<float (*)[BM * PK]>(lds_ab);
  float (*const Bs)[BN * PK] = reinterpret_cast<float (*)[BN * PK]>(lds_ab + 2 * BM * PK);
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, c = l & 15, g = l >> 4;
  const int wm = w >> 1, wn = w & 1;
  // a 1-D grid of tiles, a row block's column tiles consecutive
  const int NT = (N + BN - 1) / BN, tile = blockIdx.x;
  const int m0 = (tile / NT) * BM, n0 = (tile % NT) * BN;

  f4 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b) acc[a][b] = f4{0.f, 0.f, 0.f, 0.f};

  // thread t loads float4 slots q = t + 256 u: row q / 4, columns 4 (q % 4) ..
  float4 ra[AL], rb[BL];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < AL; ++u) {
      const int q = tid + 256 * u, r = q / Q4, i = m0 + r;
      ra[u] = q < AQ && i < M ? *reinterpret_cast<const float4*>(A + int64_t(i) * lda + k0 + 4 * (q % Q4))
                              : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < BL; ++u) {
      const int q = tid + 256 * u, r = q / Q4, j = n0 + r;
      rb[u] = q < BQ && j < N ? *reinterpret_cast<const float4*>(B + int64_t(j) * ldb + k0 + 4 * (q % Q4))
                              : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int u = 0; u < AL; ++u) {
      const int q = tid + 256 * u;
      if (q < AQ) *reinterpret_cast<float4*>(&As[buf][(q / Q4) * PK + 4 * (q % Q4)]) = ra[u];
    }
#pragma unroll
    for (int u = 0; u < BL; ++u) {
      const int q = tid + 256 * u;
      if (q < BQ) *reinterpret_cast<float4*>(&Bs[buf][(q / Q4) * PK + 4 * (q % Q4)]) = rb[u];
    }
  };

  const int steps = K / BK;  // K a multiple of BK
  load(0);
  store(0);
  __syncthreads();
  for (int s = 0; s < steps; ++s) {
    const int cur = s & 1;
    if (s + 1 < steps) load((s + 1) * BK);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {  // 16 k a sub-step: k = kk + 4g + slice
      float4 av[TM], bv[TN];
#pragma unroll
      for (int a = 0; a < TM; ++a)
        av[a] = *reinterpret_cast<const float4*>(&As[cur][(wm * WM + 16 * a + c) * PK + kk + 4 * g]);
#pragma unroll
      for (int b = 0; b < TN; ++b)
        bv[b] = *reinterpret_cast<const float4*>(&Bs[cur][(wn * WN + 16 * b + c) * PK + kk + 4 * g]);
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) {
          acc[a][b] = mfma(av[a].x, bv[b].x, acc[a][b]);
          acc[a][b] = mfma(av[a].y, bv[b].y, acc[a][b]);
          acc[a][b] = mfma(av[a].z, bv[b].z, acc[a][b]);
          acc[a][b] = mfma(av[a].w, bv[b].w, acc[a][b]);
        }
    }
    if (s + 1 < steps) {
      store(cur ^ 1);
      __syncthreads();
    }
  }
  // through LDS (both slice buffers, done with), a pass per wave row
  static_assert((BM / 2) * BN <= 2 * (BM + BN) * PK, "a wave row's results fit the slices' LDS");
  if (!staged_epilogue<BM, BN, 2, 2, 2>(acc, &As[0][0], m0, n0, M, N, C, ldc, epi))
    epilogue<WM, WN>(acc, m0, n0, wm, wn, c, g, M, N, C, ldc, epi);
}

// The same product with the fp32 matrix cores' work moved to the bf16 ones:
// B comes split once (pet_linear_split_weights: per row, per 8-element k
// group, its three bf16 parts, 48 bytes), A is split as each k step of 32 is
// staged, and a 16 x 16 x 32 step is the six part products of split_bf16.h
// (6 x 16 nominal cycles against 8 x 32 on the fp32 instruction, at fp32's
// error; measured with all waves issuing, ~33 against ~42 cycles an instruction).
// Tiles of WGM x WGN waves (64 WGM WGN threads): 64 x 64 or 128 x 64 of 2 x 2,
// 128 x 128 of 2 x 4. K steps of 32 go through one LDS buffer, the next
// step's slices loaded into registers under the current step's products. A
// row's step is 4 groups x 3 parts x 16 bytes plus a 32-byte pad (14 u4: the
// 8-byte stores of an A slice's neighbouring rows then fall on distinct banks,
// while the 128-bit operand reads stay conflict-free; measured 3-4% faster
// than a 16-byte pad at the model's large shapes, 131072 x 1536 x 512 1160
// against 1208 us): 28 / 42 / 56 KB a workgroup. K a multiple of 32.
// Measured against torch's GEMM at the model's shapes: even at K = 128
// (27318 x 128 x 128: 15 against 20 us), ahead at 26670 x 1024 x 128 (59-62
// against 86 us) and 131072 x 1536 x 512 (1160 against 1555 us); rocBLAS's
// fp32 kernel takes 12.8 us on the first.
//
// BF: B comes as fp32 rows [N, K] (ld ldb) and is split as it is staged, like
// A (for a caller with no room to keep a split copy: twice the staging VALU).
template <int BM, int BN, int WGM = 2, int WGN = 2, bool BF = false>
__global__ void __launch_bounds__(64 * WGM * WGN) gemm_nt_split_kernel(int M, int N, int K,
                                                                       const float* __restrict__ A, int64_t lda,
                                                                       const u4* __restrict__ Bs, float* C,
                                                                       int64_t ldc, Epi epi,
                                                                       const float* __restrict__ Bf, int64_t ldb,
                                                                       int /* one tile an item */) {
  constexpr int T = 64 * WGM * WGN, WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16, RP = 14;
  constexpr int AQ = BM * 8, AL = (AQ + T - 1) / T;   // float4 of a step's A slice, a thread's share
  constexpr int BQ = BF ? BN * 8 : BN * 12, BL = (BQ + T - 1) / T;  // B slice: float4 (BF) or u4 slots
  __shared__ u4 lds_ab[(BM + BN) * RP];  // A's and B's step slices, one array (the epilogue's tile spans both)
  u4* const As = lds_ab;
  u4* const Bt = lds_ab + BM * RP;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, c = l & 15, g = l >> 4;
  const int wm = w / WGN, wn = w % WGN;
  // Workgroups go to the 8 XCDs in turn (an L2 each): XCD k takes a
  // contiguous run of tiles in row-block order, so a row block's column tiles
  // share an L2 (509730 x 512 x 512: 1547 against 1624 us in launch order).
  // A bijection of the tiles whatever the hardware's order.
  // A 1-D grid of all the tiles, tile t = (row block t / NT, column tile t % NT).
  const int NT = (N + BN - 1) / BN, total = gridDim.x, L = blockIdx.x;
  const int q = total / 8, r = total % 8, x = L % 8;
  const int t = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + L / 8;
  const int tm = t / NT, tn = t % NT;
  const int m0 = tm * BM, n0 = tn * BN, KG = K / 8;

  f4 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b) acc[a][b] = f4{0.f, 0.f, 0.f, 0.f};

  // A: thread t's float4 slots q = t + 256 u, row q / 8, k 4 (q % 8) .. ;
  // B: u4 slots q, row q / 12, part (q % 12) of the row's step
  float4 ra[AL];
  u4 rb[BF ? 1 : BL];
  float4 rbf[BF ? BL : 1];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < AL; ++u) {
      const int q = tid + T * u, i = m0 + q / 8;
      ra[u] = q < AQ && i < M ? *reinterpret_cast<const float4*>(A + int64_t(i) * lda + k0 + 4 * (q % 8))
                              : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < BL; ++u) {
      if constexpr (BF) {
        const int q = tid + T * u, j = n0 + q / 8;
        rbf[u] = q < BQ && j < N ? *reinterpret_cast<const float4*>(Bf + int64_t(j) * ldb + k0 + 4 * (q % 8))
                                 : make_float4(0.f, 0.f, 0.f, 0.f);
      } else {
        const int q = tid + T * u, j = n0 + q / 12;
        rb[u] = q < BQ && j < N ? Bs[(int64_t(j) * KG + k0 / 8) * 3 + q % 12] : u4{0u, 0u, 0u, 0u};
      }
    }
  };
  // a float4 of row `row`'s k slots 4 (q % 8) .. into its split row (parts of
  // k group (q % 8) / 2, half q & 1) of tile X
  auto store_split = [&](u4* X, int row, int q, const float4& v) {
    float h[3][4];
    split3(v.x, h[0][0], h[1][0], h[2][0]);
    split3(v.y, h[0][1], h[1][1], h[2][1]);
    split3(v.z, h[0][2], h[1][2], h[2][2]);
    split3(v.w, h[0][3], h[1][3], h[2][3]);
    unsigned* dst = reinterpret_cast<unsigned*>(&X[row * RP + ((q % 8) / 2) * 3]) + 2 * (q & 1);
#pragma unroll
    for (int p = 0; p < 3; ++p)
      *reinterpret_cast<uint2*>(dst + 4 * p) = make_uint2(pack_hi(h[p][0], h[p][1]), pack_hi(h[p][2], h[p][3]));
  };
  auto store = [&]() {
#pragma unroll
    for (int u = 0; u < AL; ++u) {
      // the float4 is half of k group (q % 8) / 2: its parts go to that half of each part's 16 bytes
      const int q = tid + T * u;
      if (q < AQ) store_split(As, q / 8, q, ra[u]);
    }
#pragma unroll
    for (int u = 0; u < BL; ++u) {
      const int q = tid + T * u;
      if constexpr (BF) {
        if (q < BQ) store_split(Bt, q / 8, q, rbf[u]);
      } else {
        if (q < BQ) Bt[(q / 12) * RP + q % 12] = rb[u];
      }
    }
  };

  const int steps = K / 32;
  load(0);
  store();
  __syncthreads();
  for (int s = 0; s < steps; ++s) {
    if (s + 1 < steps) load((s + 1) * 32);
    u4 av[TM][3], bv[TN][3];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int p = 0; p < 3; ++p) av[a][p] = As[(wm * WM + 16 * a + c) * RP + 3 * g + p];
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int p = 0; p < 3; ++p) bv[b][p] = Bt[(wn * WN + 16 * b + c) * RP + 3 * g + p];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TN; ++b) acc[a][b] = mfma6(av[a], bv[b], acc[a][b]);
    if (s + 1 < steps) {
      __syncthreads();  // every wave is done with the step's slices
      store();
      __syncthreads();
    }
  }
  // through LDS (the slices', done with), a pass per wave row
  static_assert((BM / WGM) * BN * 4 <= (BM + BN) * RP * 16, "a wave row's results fit the slices' LDS");
  if (!staged_epilogue<BM, BN, WGM, WGN, WGM>(acc, reinterpret_cast<float*>(lds_ab), m0, n0, M, N, C, ldc, epi))
    epilogue<WM, WN>(acc, m0, n0, wm, wn, c, g, M, N, C, ldc, epi);
}

// W^T as split rows, W [K, N] (ld ldw): out[(n K/8 + j) 3 + p] = part p of
// column n's k group j.
__global__ void split_rows_t_kernel(const float* __restrict__ W, int N, int K, int64_t ldw, u4* __restrict__ out) {
  const int KG = K / 8;
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= int64_t(N) * KG) return;
  const int n = int(t % N), j = int(t / N);  // consecutive threads, consecutive columns of a row
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = W[int64_t(8 * j + e) * ldw + n];
  u4 parts[3];
  split8(x, parts);
#pragma unroll
  for (int p = 0; p < 3; ++p) out[(int64_t(n) * KG + j) * 3 + p] = parts[p];
}

// W [N, K] (ld ldw) as split rows: out[(n K/8 + j) 3 + p] = part p of k group j.
__global__ void split_rows_kernel(const float* __restrict__ W, int N, int K, int64_t ldw, u4* __restrict__ out) {
  const int KG = K / 8;
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= int64_t(N) * KG) return;
  const int n = int(t / KG), j = int(t % KG);
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = W[int64_t(n) * ldw + 8 * j + e];
  u4 parts[3];
  split8(x, parts);
#pragma unroll
  for (int p = 0; p < 3; ++p) out[t * 3 + p] = parts[p];
}

// pair2's lo parts of x and y with their ties (a remainder halfway between two
// fp16 numbers: every fourth weight) broken so that the errors of a group of
// eight, summed in carry, cancel: the same in every product with the weight, they
// add up over a structure (eight 648-atom structures on a 512-wide model 3.7e-6 eV
// an atom (rms) from float64 with ties to even, 3.0e-6 so).
__device__ __forceinline__ unsigned even_ties(float x, float y, unsigned hi, unsigned lo, float& carry) {
  const pet_split::h2v h = __builtin_bit_cast(pet_split::h2v, hi);
  pet_split::h2v l = __builtin_bit_cast(pet_split::h2v, lo);
  const float v[2] = {x, y};
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float err = v[e] - float(h[e]) - float(l[e]), other = float(l[e]) + 2.f * err;
    const bool flip = err * carry > 0.f && float(_Float16(other)) == other;
    carry += flip ? -err : err;
    if (flip) l[e] = _Float16(other);
  }
  return __builtin_bit_cast(unsigned, l);
}

// Rows of B = W (transposed false: W [N, K], ld ldw) or B = W^T (transposed
// true: W [K, N]) as P fp16 parts: out[(n K/8 + j) P + p] = part p of row n's
// k group j, scaled by the row's s_n (P 2: hi and lo, pair2; P 3: hi, mid and
// lo, pair3, W exactly); then at byte N K 2 P the N inverse scales 1 / s_n.
// alt (P 2): the values of odd steps of 32 negated, and the inverse scales too, which
// tells the product that reads them (gemm_rows.hip, add_step) to subtract
// those steps' sums; lo's ties by even_ties.
// One workgroup a row: its largest |x|, then its groups.
template <int P>
__global__ void __launch_bounds__(256) pair_rows_kernel(const float* __restrict__ W, int N, int K, int64_t ldw,
                                                         bool transposed, bool alt, u4* __restrict__ out) {
  static_assert(P == 2 || P == 3, "two or three parts");
  __shared__ float red[4];
  const int n = blockIdx.x, tid = threadIdx.x, KG = K / 8;
  auto at = [&](int k) { return transposed ? W[int64_t(k) * ldw + n] : W[int64_t(n) * ldw + k]; };
  float m = 0.f;
  for (int k = tid; k < K; k += 256) {
    const float x = fabsf(at(k));
    m = fmaxf(m, P == 3 && x > pet_split::kFltMax ? 0.f : x);  // (infinities: pair3)
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
  const float s = pair_scale(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
  for (int j = tid; j < KG; j += 256) {
    u4 pt[P];
    float carry = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float sj = P == 2 && alt && (j & 4) ? -s : s;
      const float x = at(8 * j + 2 * e) * sj, y = at(8 * j + 2 * e + 1) * sj;
      unsigned h, md, lw;
      if constexpr (P == 2) {
        pair2(x, y, h, lw);
        if (alt) lw = even_ties(x, y, h, lw, carry);
        pt[0][e] = h, pt[1][e] = lw;
      } else {
        pet_split::pair3(x, y, h, md, lw);
        pt[0][e] = h, pt[1][e] = md, pt[2][e] = lw;
      }
    }
#pragma unroll
    for (int p = 0; p < P; ++p) out[(int64_t(n) * KG + j) * P + p] = pt[p];
  }
  if (tid == 0) reinterpret_cast<float*>(out + int64_t(N) * KG * P)[n] = (alt ? -1.f : 1.f) / s;
}

// Rows of an activation X [M, K] (ld ldx) as fp16 pairs in pair_rows_kernel's
// layout (the M inverse scales after the pairs), one wave a row: lane j takes
// k groups j, j + 64, ..., held in registers from the row's largest |x| to
// its split (NGL groups a lane; NGL 0: any K, the row read twice, the second
// time from cache). Each lane writes 32 contiguous bytes a group.
template <int NGL>
__global__ void __launch_bounds__(256) pair_act_kernel(const float* __restrict__ X, int M, int K, int64_t ldx,
                                                        u4* __restrict__ out) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63, KG = K / 8;
  if (row >= M) return;
  const float* x = X + int64_t(row) * ldx;
  constexpr int NV = NGL > 0 ? 2 * NGL : 2;
  float4 v[NV];
  float m = 0.f;
  auto amax = [](const float4& a) { return fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))); };
  if constexpr (NGL > 0) {
#pragma unroll
    for (int i = 0; i < NGL; ++i) {
      const int j = l + 64 * i;
      if (j < KG) {
        v[2 * i] = *reinterpret_cast<const float4*>(x + 8 * j);
        v[2 * i + 1] = *reinterpret_cast<const float4*>(x + 8 * j + 4);
        m = fmaxf(m, fmaxf(amax(v[2 * i]), amax(v[2 * i + 1])));
      }
    }
  } else {
    for (int j = l; j < KG; j += 64)
      m = fmaxf(m, fmaxf(amax(*reinterpret_cast<const float4*>(x + 8 * j)),
                         amax(*reinterpret_cast<const float4*>(x + 8 * j + 4))));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
  const float s = pair_scale(m);
  auto put = [&](int j, const float4& a, const float4& b) {
    u4 hi, lo;
    unsigned h, lw;
    pair2(a.x * s, a.y * s, h, lw), hi[0] = h, lo[0] = lw;
    pair2(a.z * s, a.w * s, h, lw), hi[1] = h, lo[1] = lw;
    pair2(b.x * s, b.y * s, h, lw), hi[2] = h, lo[2] = lw;
    pair2(b.z * s, b.w * s, h, lw), hi[3] = h, lo[3] = lw;
    u4* o = out + (int64_t(row) * KG + j) * 2;
    o[0] = hi, o[1] = lo;
  };
  if constexpr (NGL > 0) {
#pragma unroll
    for (int i = 0; i < NGL; ++i)
      if (l + 64 * i < KG) put(l + 64 * i, v[2 * i], v[2 * i + 1]);
  } else {
    for (int j = l; j < KG; j += 64)
      put(j, *reinterpret_cast<const float4*>(x + 8 * j), *reinterpret_cast<const float4*>(x + 8 * j + 4));
  }
  if (l == 0) reinterpret_cast<float*>(out + int64_t(M) * KG * 2)[row] = 1.f / s;
}

}  // namespace pet_gemm

using namespace pet_gemm;

// Which split a K takes: fp16 pairs from K = 256 (three matrix instructions a
// product where the bf16 form takes six, and a first pass over A's rows for
// their scales, which pays once the K loop is long enough: measured 131072 x
// 1536 x 512 908-923 against 1220 us, 122688 x 768 x 256 289 against 345 us,
// but 26670 x 1024 x 128 78 against 70 us), three bf16 parts below. The
// weights' split and the product both follow it, so a split copy matches the
// kernel that reads it.
static bool pair_form(int K) { return K >= 256; }

// The tile shape for a problem: wide outputs take 128 x 128; narrow ones
// (N <= 64) or too few tiles to fill 256 CUs take smaller tiles.
int pet_gemm_nt_fused(int M, int N, int K, const float* A, int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc,
                const float* row_scale, const float* bias, const float* cin, int64_t ldcin, float beta, float* pre,
                int64_t ldpre, int act, hipStream_t st) {
  if (M < 0 || N < 0 || K < 0) return PET_ATTN_EINVAL;
  if (M == 0 || N == 0) return PET_ATTN_OK;
  if (K == 0) return PET_ATTN_EINVAL;
  if (K % 16 || lda % 4 || ldb % 4 || (reinterpret_cast<uintptr_t>(A) & 15) || (reinterpret_cast<uintptr_t>(B) & 15))
    return PET_ATTN_EALIGN;
  if (act == 2 && N % 2) return PET_ATTN_EINVAL;
  Epi e;
  e.row_scale = row_scale, e.bias = bias, e.cin = cin, e.ldcin = ldcin, e.beta = beta, e.pre = pre, e.ldpre = ldpre;
  e.act = act;
  auto tiles = [&](int bm, int bn) { return int64_t((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  const bool k32 = K % 32 == 0;
  auto go = [&](auto kern, int bm, int bn) {  // a 1-D grid: every tile, no extent limit below 2^31 tiles
    hipLaunchKernelGGL(kern, dim3(unsigned(tiles(bm, bn))), dim3(256), 0, st, M, N, K, A, lda, B, ldb, C, ldc, e);
  };
  if (tiles(64, 32) >= (int64_t(1) << 31)) return PET_ATTN_EINDEX;
  if (N > 64 && tiles(128, 128) >= 512)
    k32 ? go(gemm_nt_kernel<128, 128, 32>, 128, 128) : go(gemm_nt_kernel<128, 128, 16>, 128, 128);
  else if (N > 32 && tiles(128, 64) >= 512)
    k32 ? go(gemm_nt_kernel<128, 64, 32>, 128, 64) : go(gemm_nt_kernel<128, 64, 16>, 128, 64);
  else
    k32 ? go(gemm_nt_kernel<64, 32, 32>, 64, 32) : go(gemm_nt_kernel<64, 32, 16>, 64, 32);
  tally(0, M, N, K);
  return hipGetLastError() == hipSuccess ? PET_ATTN_OK : PET_ATTN_ELAUNCH;
}

// The epilogue arguments of the public entry points: C's and cin's widths
// per act (act 4 writes and reads 2N columns), cin required by the backward
// codes 3 and 4, which take no row scale and no pre.
static bool epi_args_ok(int N, const float* C, int64_t ldc, const float* row_scale, const float* cin, int64_t ldcin,
                        const float* pre, int64_t ldpre, int act) {
  if (act < 0 || act > 4 || !C) return false;
  if (act >= 3) {
    const int64_t w = act == 4 ? 2 * int64_t(N) : N;
    // act 4 stores (value, gate) adjoint pairs as 8-byte words
    const bool pairs_ok = act == 3 || ((reinterpret_cast<uintptr_t>(C) & 7) == 0 && ldc % 2 == 0);
    return cin && ldcin >= w && ldc >= w && !row_scale && !pre && pairs_ok;
  }
  return ldc >= (act == 2 ? N / 2 : N) && (!cin || ldcin >= N) && (!pre || ldpre >= N);
}

extern "C" int pet_linear_fused(int M, int N, int K, const float* A, int64_t lda, const float* W, int64_t ldw,
                                float* C, int64_t ldc, const float* row_scale, const float* bias, const float* cin,
                                int64_t ldcin, float beta, float* pre, int64_t ldpre, int act, void* stream) {
  if ((M > 0 && N > 0) && (!A || !W || !C || lda < K || ldw < K || !epi_args_ok(N, C, ldc, row_scale, cin, ldcin,
                                                                                    pre, ldpre, act)))
    return PET_ATTN_EINVAL;
  return pet_gemm_nt_fused(M, N, K, A, lda, W, ldw, C, ldc, row_scale, bias, cin, ldcin, beta, pre, ldpre, act,
                           reinterpret_cast<hipStream_t>(stream));
}

int pet_gemm_nt_pp(int M, int N, int K, const void* Ap, const void* Bs, float* C, int64_t ldc, const Epi& e,
                   hipStream_t st);
int pet_gemm_pair_rows(const float* X, int M, int K, int64_t ldx, void* out, hipStream_t st);

// From which N A's rows are split into the scratch first: below, their scales
// are found by each tile (62291 rows on MI355X: N 512 K 1024 236 us against 75 + 176,
// N 2048 K 512 519 against 45 + 408; the same bits). Block pairs out ask for the
// scratch from N = 512.
constexpr int kPairsMinN = 1024, kBlocksMinN = 512;

// The split-product GEMM with the epilogue e (block pairs out where e.pout).
int split_impl(int M, int N, int K, const float* A, int64_t lda, const void* Bs, float* C, int64_t ldc, Epi e,
               hipStream_t st, void* scratch, size_t scratch_bytes) {
  if (M < 0 || N < 0 || K < 0) return PET_ATTN_EINVAL;
  if (M == 0 || N == 0) return PET_ATTN_OK;
  if (K == 0) return PET_ATTN_EINVAL;
  if (int64_t((M + 63) / 64) * ((N + 63) / 64) >= (int64_t(1) << 31)) return PET_ATTN_EINDEX;  // 1-D grid of tiles
  if (K % 32 || lda % 4 || (reinterpret_cast<uintptr_t>(A) & 15) || (reinterpret_cast<uintptr_t>(Bs) & 15))
    return PET_ATTN_EALIGN;
  if (e.act == 2 && N % 2) return PET_ATTN_EINVAL;
  const int64_t ldcin = e.ldcin, ldpre = e.ldpre;
  // A's rows split into the scratch a chunk at a time (as many rows as it
  // holds, a multiple of 128), each chunk's product from the pairs
  const int64_t chunk = scratch ? int64_t(scratch_bytes / (size_t(K) * 4 + 4)) / 128 * 128 : 0;
  const bool room = pair_form(K) && N >= kBlocksMinN && chunk >= 128 && (reinterpret_cast<uintptr_t>(scratch) & 15) == 0;
  if (e.pout && !room) return PET_ATTN_EINVAL;  // block pairs out: as many rows of scratch as that path has always asked for
  if (e.pout || (room && N >= kPairsMinN)) {
    for (int64_t r0 = 0; r0 < M; r0 += chunk) {
      const int m = int(std::min<int64_t>(chunk, M - r0));
      Epi ec = e;
      if (ec.row_scale) ec.row_scale += r0;
      if (ec.cin) ec.cin += r0 * ldcin;
      if (ec.pre) ec.pre += r0 * ldpre;
      if (ec.pout) ec.pout += r0 * ec.kgo * 2, ec.pinv += r0;
      int rc = pet_gemm_pair_rows(A + r0 * lda, m, K, lda, scratch, st);
      if (rc == PET_ATTN_OK) rc = pet_gemm_nt_pp(m, N, K, scratch, Bs, C ? C + r0 * ldc : C, ldc, ec, st);
      if (rc != PET_ATTN_OK) return rc;
    }
    return PET_ATTN_OK;
  }
  if (pair_form(K)) return pet_gemm_nt_rows(M, N, K, A, lda, kRowsExact, 0, Bs, 2, C, ldc, e, st, 0);
  auto go = [&](auto kern, int bm, int bn, int threads) {  // a 1-D grid of every tile
    const int64_t tiles = int64_t((M + bm - 1) / bm) * ((N + bn - 1) / bn);
    hipLaunchKernelGGL(kern, dim3(unsigned(tiles)), dim3(threads), 0, st, M, N, K, A, lda, static_cast<const u4*>(Bs), C,
                       ldc, e, static_cast<const float*>(nullptr), int64_t(0), 1);
    tally(1, M, N, K);
  };
  // measured on MI355X: 128 x 128 tiles of 8 waves where there are many
  // (131072 x 1536 x 512: 1200-1213 us against 1394-1418 for 128 x 64 and
  // 1535 for 64 x 64; 256 x 128 and 128 x 256 tiles of 16 waves were no
  // faster), 64 x 64 otherwise (27318 x 128 x 128: 16.1 against 18.4 us); one
  // LDS buffer beat two in every shape
  const int64_t tiles128 = int64_t((M + 127) / 128) * ((N + 63) / 64);
  if (N >= 128 && tiles128 >= 2048)
    go(gemm_nt_split_kernel<128, 128, 2, 4>, 128, 128, 512);
  else if (tiles128 >= 2048)
    go(gemm_nt_split_kernel<128, 64>, 128, 64, 256);
  else
    go(gemm_nt_split_kernel<64, 64>, 64, 64, 256);
  return hipGetLastError() == hipSuccess ? PET_ATTN_OK : PET_ATTN_ELAUNCH;
}

int pet_gemm_nt_split(int M, int N, int K, const float* A, int64_t lda, const void* Bs, float* C, int64_t ldc,
                      const float* row_scale, const float* bias, const float* cin, int64_t ldcin, float beta,
                      float* pre, int64_t ldpre, int act, hipStream_t st, void* scratch, size_t scratch_bytes) {
  Epi e;
  e.row_scale = row_scale, e.bias = bias, e.cin = cin, e.ldcin = ldcin, e.beta = beta, e.pre = pre, e.ldpre = ldpre;
  e.act = act;
  return split_impl(M, N, K, A, lda, Bs, C, ldc, e, st, scratch, scratch_bytes);
}

// The output columns of a product of N columns under activation act.
static int out_cols(int N, int act) { return act == 2 ? N / 2 : act == 4 ? 2 * N : N; }

// Block pairs out: the split-product GEMM's output epi(A B^T) as fp16 pairs
// scaled per (row, 128-column tile of the product) into pout -- M rows of
// out_cols(N, act) / 8 k groups (pair_act_kernel's layout), then the inverse
// scales [out_cols(N, act) / kb][M] -- for a product that reads them as its A
// (pet_gemm_nt_pp_blocks with that kb, returned in *kb: 64 for SwiGLU, 256
// for its backward, 128 otherwise). N a multiple of 128, the output's columns
// of 32, every epilogue operand 16-byte aligned with leading dimensions of 4.
int pet_gemm_nt_split_pairs(int M, int N, int K, const float* A, int64_t lda, const void* Bs, void* pout,
                            const float* row_scale, const float* bias, const float* cin, int64_t ldcin, float beta,
                            float* pre, int64_t ldpre, int act, hipStream_t st, void* scratch, size_t scratch_bytes,
                            int* kb) {
  auto a16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const int no = out_cols(N, act);
  if (!pout || !a16(pout) || N % 128 || no % 32 || (bias && !a16(bias)) || (cin && (!a16(cin) || ldcin % 4)) ||
      (pre && (!a16(pre) || ldpre % 4)))
    return PET_ATTN_EINVAL;
  Epi e;
  e.row_scale = row_scale, e.bias = bias, e.cin = cin, e.ldcin = ldcin, e.beta = beta, e.pre = pre, e.ldpre = ldpre;
  e.act = act;
  e.pout = static_cast<u4*>(pout), e.kgo = no / 8, e.ldinv = M;
  e.pinv = reinterpret_cast<float*>(e.pout + int64_t(M) * e.kgo * 2);
  if (kb) *kb = out_cols(128, act);
  return split_impl(M, N, K, A, lda, Bs, nullptr, 0, e, st, scratch, scratch_bytes);
}

// The same product from fp32 B [N, K] (ld ldb), split as it is staged: for
// callers with no room to keep a split copy of the weights (the op-level
// attention()'s output linear). K a multiple of 32; A and B 16-byte aligned
// rows.
int pet_gemm_nt_split_f32b(int M, int N, int K, const float* A, int64_t lda, const float* B, int64_t ldb, float* C,
                           int64_t ldc, const float* bias, const float* cin, int64_t ldcin, float beta, hipStream_t st) {
  if (M < 0 || N < 0 || K < 0) return PET_ATTN_EINVAL;
  if (M == 0 || N == 0) return PET_ATTN_OK;
  if (K == 0) return PET_ATTN_EINVAL;
  if (int64_t((M + 63) / 64) * ((N + 63) / 64) >= (int64_t(1) << 31)) return PET_ATTN_EINDEX;
  if (K % 32 || lda % 4 || ldb % 4 || (reinterpret_cast<uintptr_t>(A) & 15) || (reinterpret_cast<uintptr_t>(B) & 15))
    return PET_ATTN_EALIGN;
  Epi e;
  e.bias = bias, e.cin = cin, e.ldcin = ldcin, e.beta = beta;
  auto go = [&](auto kern, int bm, int bn, int threads) {
    const int64_t tiles = int64_t((M + bm - 1) / bm) * ((N + bn - 1) / bn);
    hipLaunchKernelGGL(kern, dim3(unsigned(tiles)), dim3(threads), 0, st, M, N, K, A, lda, nullptr, C, ldc, e, B,
                       ldb, 1);
    tally(1, M, N, K);
  };
  const int64_t t128 = int64_t((M + 127) / 128) * ((N + 63) / 64);
  if (N >= 128 && t128 >= 2048)
    go(gemm_nt_split_kernel<128, 128, 2, 4, true>, 128, 128, 512);
  else if (t128 >= 2048)
    go(gemm_nt_split_kernel<128, 64, 2, 2, true>, 128, 64, 256);
  else
    go(gemm_nt_split_kernel<64, 64, 2, 2, true>, 64, 64, 256);
  return hipGetLastError() == hipSuccess ? PET_ATTN_OK : PET_ATTN_ELAUNCH;
}

// B [N, K] as split rows, from W = B (transposed false: W [N, K]) or W = B^T
// (transposed true: W [K, N]); K a multiple of 32, out 16-byte aligned. alt: pairs
// with steps of either sign (pair_rows_kernel), for the products of a model and
// of the layer level, whose errors' mean adds up over a structure's atoms.
int pet_gemm_split_weights(const float* W, int N, int K, int64_t ldw, bool transposed, bool alt, void* out,
                           hipStream_t st) {
  if (N < 0 || K < 0 || K % 32 || (reinterpret_cast<uintptr_t>(out) & 15)) return PET_ATTN_EINVAL;
  const int64_t n = int64_t(N) * (K / 8);
  if (n == 0) return PET_ATTN_OK;
  if (pair_form(K))
    hipLaunchKernelGGL(pair_rows_kernel<2>, dim3(unsigned(N)), dim3(256), 0, st, W, N, K, ldw, transposed, alt,
                       static_cast<u4*>(out));
  else if (transposed)
    hipLaunchKernelGGL(split_rows_t_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, W, N, K, ldw,
                       static_cast<u4*>(out));
  else
    hipLaunchKernelGGL(split_rows_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, W, N, K, ldw,
                       static_cast<u4*>(out));
  return hipGetLastError() == hipSuccess ? PET_ATTN_OK : PET_ATTN_ELAUNCH;
}

extern "C" int pet_linear_split_weights(const float* W, int N, int K, int64_t ldw, void* out, void* stream) {
  if (N < 0 || K < 0 || K % 32 || ldw < K || ((N > 0 && K > 0) && (!W || !out))) return PET_ATTN_EINVAL;
  if (reinterpret_cast<uintptr_t>(out) & 15) return PET_ATTN_EALIGN;
  const int64_t n = int64_t(N) * (K / 8);
  if (n == 0) return PET_ATTN_OK;
  return pet_gemm_split_weights(W, N, K, ldw, false, false, out, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int pet_linear_split_weights_transposed(const float* W, int N, int K, int64_t ldw, void* out,
                                                   void* stream) {
  if (N < 0 || K < 0 || K % 32 || ldw < N || ((N > 0 && K > 0) && (!W || !out))) return PET_ATTN_EINVAL;
  if (reinterpret_cast<uintptr_t>(out) & 15) return PET_ATTN_EALIGN;
  return pet_gemm_split_weights(W, N, K, ldw, true, false, out, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int pet_linear_fused_split(int M, int N, int K, const float* A, int64_t lda, const void* Wsplit, float* C,
                                      int64_t ldc, const float* row_scale, const float* bias, const float* cin,
                                      int64_t ldcin, float beta, float* pre, int64_t ldpre, int act, void* stream) {
  if ((M > 0 && N > 0) && (!A || !Wsplit || !C || lda < K || !epi_args_ok(N, C, ldc, row_scale, cin, ldcin, pre,
                                                                              ldpre, act)))
    return PET_ATTN_EINVAL;
  return pet_gemm_nt_split(M, N, K, A, lda, Wsplit, C, ldc, row_scale, bias, cin, ldcin, beta, pre, ldpre, act,
                           reinterpret_cast<hipStream_t>(stream), nullptr, 0);
}

extern "C" int pet_linear_fused_split_ws(int M, int N, int K, const float* A, int64_t lda, const void* Wsplit,
                                         float* C, int64_t ldc, const float* row_scale, const float* bias,
                                         const float* cin, int64_t ldcin, float beta, float* pre, int64_t ldpre,
                                         int act, void* scratch, size_t scratch_bytes, void* stream) {
  if ((M > 0 && N > 0) && (!A || !Wsplit || !C || lda < K || !epi_args_ok(N, C, ldc, row_scale, cin, ldcin, pre,
                                                                              ldpre, act)))
    return PET_ATTN_EINVAL;
  if (scratch_bytes && !scratch) return PET_ATTN_EINVAL;
  return pet_gemm_nt_split(M, N, K, A, lda, Wsplit, C, ldc, row_scale, bias, cin, ldcin, beta, pre, ldpre, act,
                           reinterpret_cast<hipStream_t>(stream), scratch, scratch_bytes);
}

// fp16-pair rows of an activation X [M, K] into out (M K 4 + M 4 bytes,
// 16-byte aligned): the A operand of pet_gemm_nt_pp. Pair-form K only.
int pet_gemm_pair_rows(const float* X, int M, int K, int64_t ldx, void* out, hipStream_t st) {
  if (M < 0 || K < 0 || !pair_form(K) || K % 32 || ldx % 4 || (reinterpret_cast<uintptr_t>(X) & 15) ||
      (reinterpret_cast<uintptr_t>(out) & 15))
    return PET_ATTN_EINVAL;
  if (M == 0) return PET_ATTN_OK;
  const dim3 grid(unsigned((M + 3) / 4));
  u4* o = static_cast<u4*>(out);
  if (K <= 512)
    hipLaunchKernelGGL(pair_act_kernel<1>, grid, dim3(256), 0, st, X, M, K, ldx, o);
  else if (K <= 1024)
    hipLaunchKernelGGL(pair_act_kernel<2>, grid, dim3(256), 0, st, X, M, K, ldx, o);
  else if (K <= 2048)
    hipLaunchKernelGGL(pair_act_kernel<4>, grid, dim3(256), 0, st, X, M, K, ldx, o);
  else
    hipLaunchKernelGGL(pair_act_kernel<0>, grid, dim3(256), 0, st, X, M, K, ldx, o);
  return hipGetLastError() == hipSuccess ? PET_ATTN_OK : PET_ATTN_ELAUNCH;
}

// C = epi(A B^T) from the pairs of A (pet_gemm_pair_rows) and of B
// (pet_gemm_split_weights), K of the pair form.
int pet_gemm_nt_pp(int M, int N, int K, const void* Ap, const void* Bs, float* C, int64_t ldc, const Epi& e,
                   hipStream_t st) {
  if (M < 0 || N < 0 || !pair_form(K) || K % 32) return PET_ATTN_EINVAL;
  if (M == 0 || N == 0) return PET_ATTN_OK;
  return pet_gemm_nt_rows(M, N, K, Ap, 0, kRowsPairs, K, Bs, 2, C, ldc, e, st, 0);
}

// Block pairs out (as pet_gemm_nt_split_pairs) from A already as pair rows
// (pet_gemm_pair_rows' layout, K of the pair form): gemm_rows_kernel from
// pairs alone, every row at once.
int pet_gemm_nt_pp_to_blocks(int M, int N, int K, const void* Ap, const void* Bs, void* pout, const float* bias,
                             const float* cin, int64_t ldcin, float beta, float* pre, int64_t ldpre, int act,
                             hipStream_t st, int* kb) {
  auto a16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const int no = out_cols(N, act);
  if (!pout || !a16(pout) || N % 128 || no % 32 || (bias && !a16(bias)) || (cin && (!a16(cin) || ldcin % 4)) ||
      (pre && (!a16(pre) || ldpre % 4)) || act < 0 || act > 4 || (act == 2 && N % 2))
    return PET_ATTN_EINVAL;
  Epi e;
  e.bias = bias, e.cin = cin, e.ldcin = ldcin, e.beta = beta, e.pre = pre, e.ldpre = ldpre, e.act = act;
  e.pout = static_cast<u4*>(pout), e.kgo = no / 8, e.ldinv = M;
  e.pinv = reinterpret_cast<float*>(e.pout + int64_t(M) * e.kgo * 2);
  if (kb) *kb = out_cols(128, act);
  return pet_gemm_nt_pp(M, N, K, Ap, Bs, nullptr, 0, e, st);
}

constexpr int kMaxBlocks = 32;  // (the interface's limit, of its callers' too; the kernel takes any number)

// C = epi(A B^T) with A as block pairs (pet_gemm_nt_split_pairs' pout: M
// rows of pairs, then the inverse scales [K / kb][M]) and B's pair rows; kb 32,
// 64, 128 or 256, dividing K, at most 32 blocks.
int pet_gemm_nt_pp_blocks(int M, int N, int K, const void* Ap, int kb, const void* Bs, float* C, int64_t ldc,
                          const float* row_scale, const float* bias, const float* cin, int64_t ldcin, float beta,
                          float* pre, int64_t ldpre, int act, hipStream_t st) {
  if (M < 0 || N < 0 || K <= 0 || K % 32 || !(kb == 32 || kb == 64 || kb == 128 || kb == 256) || K % kb ||
      K / kb > kMaxBlocks || (act == 2 && N % 2))
    return PET_ATTN_EINVAL;
  if (M == 0 || N == 0) return PET_ATTN_OK;
  Epi e;
  e.row_scale = row_scale, e.bias = bias, e.cin = cin, e.ldcin = ldcin, e.beta = beta, e.pre = pre, e.ldpre = ldpre;
  e.act = act;
  return pet_gemm_nt_rows(M, N, K, Ap, 0, kRowsPairs, kb, Bs, 2, C, ldc, e, st, 0);
}

// B's rows as three fp16 parts (hi, mid, lo: W exactly) at any K (a multiple
// of 32), for the three-part kernels: N K 6 + N 4 bytes.
int pet_gemm_pair_weights(const float* W, int N, int K, int64_t ldw, bool transposed, void* out, hipStream_t st) {
  if (N < 0 || K < 0 || K % 32 || (reinterpret_cast<uintptr_t>(out) & 15)) return PET_ATTN_EINVAL;
  if (N == 0 || K == 0) return PET_ATTN_OK;
  hipLaunchKernelGGL(pair_rows_kernel<3>, dim3(unsigned(N)), dim3(256), 0, st, W, N, K, ldw, transposed, false,
                     static_cast<u4*>(out));
  return hipGetLastError() == hipSuccess ? PET_ATTN_OK : PET_ATTN_ELAUNCH;
}

extern "C" int pet_linear_pair_weights(const float* W, int N, int K, int64_t ldw, void* out, void* stream) {
  if (N < 0 || K < 0 || K % 32 || ldw < K || ((N > 0 && K > 0) && (!W || !out))) return PET_ATTN_EINVAL;
  if (reinterpret_cast<uintptr_t>(out) & 15) return PET_ATTN_EALIGN;
  return pet_gemm_pair_weights(W, N, K, ldw, false, out, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int pet_linear_fused_parts(int M, int N, int K, const float* A, int64_t lda, const void* Wpairs, float* C,
                                      int64_t ldc, const float* row_scale, const float* bias, const float* cin,
                                      int64_t ldcin, float beta, float* pre, int64_t ldpre, int act, void* stream) {
  if ((M > 0 && N > 0) && (!A || !Wpairs || !C || lda < K || !epi_args_ok(N, C, ldc, row_scale, cin, ldcin, pre,
                                                                              ldpre, act)))
    return PET_ATTN_EINVAL;
  if (act == 2 && N % 2) return PET_ATTN_EINVAL;
  Epi e;
  e.row_scale = row_scale, e.bias = bias, e.cin = cin, e.ldcin = ldcin, e.beta = beta, e.pre = pre, e.ldpre = ldpre;
  e.act = act;
  return pet_gemm_nt_p3(M, N, K, A, lda, Wpairs, C, ldc, e, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int pet_linear_fused_smallk(int M, int N, int K, const float* A, int64_t lda, const void* Wpairs, float* C,
                                       int64_t ldc, const float* row_scale, const float* bias, const float* cin,
                                       int64_t ldcin, float beta, float* pre, int64_t ldpre, int act, void* stream) {
  if ((M > 0 && N > 0) && (!A || !Wpairs || !C || lda < K || !epi_args_ok(N, C, ldc, row_scale, cin, ldcin, pre,
                                                                              ldpre, act)))
    return PET_ATTN_EINVAL;
  if (act == 2 && N % 2) return PET_ATTN_EINVAL;
  if (K > 128) return PET_ATTN_EINVAL;
  return pet_linear_fused_parts(M, N, K, A, lda, Wpairs, C, ldc, row_scale, bias, cin, ldcin, beta, pre, ldpre, act,
                                stream);
}

extern "C" int pet_linear_pair_rows(const float* X, int M, int K, int64_t ldx, void* out, void* stream) {
  if (M < 0 || K < 0 || ldx < K || (M > 0 && K > 0 && (!X || !out))) return PET_ATTN_EINVAL;
  return pet_gemm_pair_rows(X, M, K, ldx, out, reinterpret_cast<hipStream_t>(stream));
}

// the epilogue's operands for a product with no C (block pairs out)
static bool epi_args_nc_ok(int N, const float* row_scale, const float* cin, int64_t ldcin, const float* pre,
                           int64_t ldpre, int act) {
  if (act < 0 || act > 4) return false;
  if (act >= 3) return cin && ldcin >= (act == 4 ? 2 * int64_t(N) : N) && !row_scale && !pre;
  return (!cin || ldcin >= N) && (!pre || ldpre >= N);
}

extern "C" int pet_linear_fused_split_blocks(int M, int N, int K, const float* A, int64_t lda, const void* Wsplit,
                                             void* out, const float* row_scale, const float* bias, const float* cin,
                                             int64_t ldcin, float beta, float* pre, int64_t ldpre, int act,
                                             void* scratch, size_t scratch_bytes, int* kb, void* stream) {
  if (!kb || (M > 0 && N > 0 && (!A || !Wsplit || !out || lda < K ||
                                  !epi_args_nc_ok(N, row_scale, cin, ldcin, pre, ldpre, act))))
    return PET_ATTN_EINVAL;
  return pet_gemm_nt_split_pairs(M, N, K, A, lda, Wsplit, out, row_scale, bias, cin, ldcin, beta, pre, ldpre, act,
                                 reinterpret_cast<hipStream_t>(stream), scratch, scratch_bytes, kb);
}

extern "C" int pet_linear_fused_blocks(int M, int N, int K, const void* Ablocks, int kb, const void* Wsplit, float* C,
                                       int64_t ldc, const float* row_scale, const float* bias, const float* cin,
                                       int64_t ldcin, float beta, float* pre, int64_t ldpre, int act, void* stream) {
  if ((M > 0 && N > 0) && (!Ablocks || !Wsplit || !C || !epi_args_ok(N, C, ldc, row_scale, cin, ldcin, pre,
                                                                       ldpre, act)))
    return PET_ATTN_EINVAL;
  return pet_gemm_nt_pp_blocks(M, N, K, Ablocks, kb, Wsplit, C, ldc, row_scale, bias, cin, ldcin, beta, pre, ldpre,
                               act, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int pet_linear_fused_pairs(int M, int N, int K, const void* Apairs, const void* Wsplit, float* C,
                                      int64_t ldc, const float* row_scale, const float* bias, const float* cin,
                                      int64_t ldcin, float beta, float* pre, int64_t ldpre, int act, void* stream) {
  if ((M > 0 && N > 0) && (!Apairs || !Wsplit || !C || !epi_args_ok(N, C, ldc, row_scale, cin, ldcin, pre,
                                                                      ldpre, act)))
    return PET_ATTN_EINVAL;
  if (act == 2 && N % 2) return PET_ATTN_EINVAL;
  Epi e;
  e.row_scale = row_scale, e.bias = bias, e.cin = cin, e.ldcin = ldcin, e.beta = beta, e.pre = pre, e.ldpre = ldpre;
  e.act = act;
  return pet_gemm_nt_pp(M, N, K, Apairs, Wsplit, C, ldc, e, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int pet_gemm_flop_tally(double* flops, int reset) {
  if (!flops) return PET_ATTN_EINVAL;
  for (int c = 0; c < 4; ++c)
    flops[c] = double(reset ? g_flops[c].exchange(0, std::memory_order_relaxed)
                            : g_flops[c].load(std::memory_order_relaxed));
  return PET_ATTN_OK;
}

// What the dense-layer kernels share (gemm.hip, gemm_rows.hip): the epilogue's
// operands and arithmetic, the FLOP tally.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>

#include "split_bf16.h"

namespace pet_gemm {

using pet_split::f4;
using pet_split::u2;
using pet_split::u4;

// The hardware's exp and reciprocal, with one Newton step on the reciprocal
// (its own ulp of error has a mean that a model's activations add up).
__device__ __forceinline__ float sig_fast(float x) {
  const float d = fminf(1.0f + __expf(-x), 3.0e38f), r = __builtin_amdgcn_rcpf(d);
  return fmaf(fmaf(-d, r, 1.0f), r, r);
}

struct Epi {
  const float* row_scale = nullptr;  // [M]
  const float* bias = nullptr;       // [N]
  const float* cin = nullptr;        // [M, N] (ld ldcin), scaled by beta
  int64_t ldcin = 0;
  float beta = 0.f;
  float* pre = nullptr;              // [M, N] (ld ldpre): v before the activation
  int64_t ldpre = 0;
  int act = 0;                       // 0 none, 1 SiLU, 2 SwiGLU (C has N/2 columns),
                                     // 3 / 4 the backward of SiLU / SwiGLU (below)
  // Block pairs in place of C (the row kernels only): the output row i as
  // fp16 pairs in pair_act_kernel's layout (kgo k groups of 8 a row, each
  // group's hi then lo 16 bytes), scaled per (row, column tile) -- the tile's
  // output columns are one K block of the product that reads them -- with the
  // block's inverse scale at pinv[block ldinv + i].
  u4* pout = nullptr;
  float* pinv = nullptr;
  int64_t ldinv = 0;
  int kgo = 0;
};

// FLOPs (2 M N K) of the products this library's dense kernels have launched,
// by the instructions that run them: 0 the fp32 fused kernel (fp32 matrix
// cores), 1 split-fp32 as three bf16 parts (six bf16 products), 2 fp16 pairs
// (three fp16 products), 3 the three-part kernels (five fp16 products). A
// measurement aid, process-wide (pet_gemm_flop_tally).
extern std::atomic<uint64_t> g_flops[4];  // gemm.hip
inline void tally(int cls, int64_t M, int64_t N, int64_t K) {
  g_flops[cls].fetch_add(uint64_t(2) * uint64_t(M) * uint64_t(N) * uint64_t(K), std::memory_order_relaxed);
}

// epi_elem's arithmetic, in its order, for four consecutive output columns
// j .. j + 3 of row i (j a multiple of 4; a SwiGLU pair in one lane), with
// 16-byte accesses where vec (every pointer 16-byte aligned, every leading
// dimension and N multiples of 4), element by element otherwise.
template <bool vec, bool bwd>
__device__ __forceinline__ void epi_quad(float (&v)[4], int i, int j, int M, int N, float* C, int64_t ldc,
                                         const Epi& epi, const float4* bq = nullptr) {
  if (i >= M || j >= N) return;
  if constexpr (bwd) {
    const float* z = epi.cin + int64_t(i) * epi.ldcin;
    if constexpr (vec) {  // z, bias and C rows 16-byte aligned, N a multiple of 4
      if (epi.act == 3) {
        const float4 z4 = *reinterpret_cast<const float4*>(z + j);
        const float4 b4 = epi.bias ? *reinterpret_cast<const float4*>(epi.bias + j) : make_float4(0.f, 0.f, 0.f, 0.f);
        const float xs[4] = {z4.x + b4.x, z4.y + b4.y, z4.z + b4.z, z4.w + b4.w};
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float sg = sig_fast(xs[e]);
          o[e] = v[e] * (sg * (1.0f + xs[e] * (1.0f - sg)));
        }
        *reinterpret_cast<float4*>(C + int64_t(i) * ldc + j) = make_float4(o[0], o[1], o[2], o[3]);
      } else {  // (value, gate) pairs 2 j .. 2 j + 7
        float zz[8];
        *reinterpret_cast<float4*>(zz) = *reinterpret_cast<const float4*>(z + 2 * j);
        *reinterpret_cast<float4*>(zz + 4) = *reinterpret_cast<const float4*>(z + 2 * j + 4);
        if (epi.bias) {
          const float4 b0 = *reinterpret_cast<const float4*>(epi.bias + 2 * j);
          const float4 b1 = *reinterpret_cast<const float4*>(epi.bias + 2 * j + 4);
          zz[0] += b0.x, zz[1] += b0.y, zz[2] += b0.z, zz[3] += b0.w;
          zz[4] += b1.x, zz[5] += b1.y, zz[6] += b1.z, zz[7] += b1.w;
        }
        float o[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float u = zz[2 * e], sg = sig_fast(zz[2 * e + 1]);
          o[2 * e] = v[e] * sg;
          o[2 * e + 1] = v[e] * u * sg * (1.0f - sg);
        }
        float* cr = C + int64_t(i) * ldc + 2 * j;
        *reinterpret_cast<float4*>(cr) = make_float4(o[0], o[1], o[2], o[3]);
        *reinterpret_cast<float4*>(cr + 4) = make_float4(o[4], o[5], o[6], o[7]);
      }
      return;
    }
    if (epi.act == 3) {
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (!vec && j + e >= N) break;
        const float x = z[j + e] + (epi.bias ? epi.bias[j + e] : 0.f), sg = sig_fast(x);
        o[e] = v[e] * (sg * (1.0f + x * (1.0f - sg)));
        if (!vec) C[int64_t(i) * ldc + j + e] = o[e];
      }
      if (vec) *reinterpret_cast<float4*>(C + int64_t(i) * ldc + j) = make_float4(o[0], o[1], o[2], o[3]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (j + e >= N) break;
        const int jj = j + e;
        const float u = z[2 * jj] + (epi.bias ? epi.bias[2 * jj] : 0.f);
        const float sg = sig_fast(z[2 * jj + 1] + (epi.bias ? epi.bias[2 * jj + 1] : 0.f));
        *reinterpret_cast<float2*>(C + int64_t(i) * ldc + 2 * jj) = make_float2(v[e] * sg, v[e] * u * sg * (1.0f - sg));
      }
    }
    return;
  }
  const int ne = vec ? 4 : min(4, N - j);
  if (epi.row_scale) {
    const float rs = epi.row_scale[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] *= rs;
  }
  if (epi.bias) {
    if (vec) {
      const float4 b4 = bq ? *bq : *reinterpret_cast<const float4*>(epi.bias + j);
      v[0] += b4.x, v[1] += b4.y, v[2] += b4.z, v[3] += b4.w;
    } else {
      for (int e = 0; e < ne; ++e) v[e] += epi.bias[j + e];
    }
  }
  if (epi.cin) {
    const float* ci = epi.cin + int64_t(i) * epi.ldcin + j;
    if (vec) {
      const float4 c4 = *reinterpret_cast<const float4*>(ci);
      v[0] += epi.beta * c4.x, v[1] += epi.beta * c4.y, v[2] += epi.beta * c4.z, v[3] += epi.beta * c4.w;
    } else {
      for (int e = 0; e < ne; ++e) v[e] += epi.beta * ci[e];
    }
  }
  if (epi.pre) {
    float* pr = epi.pre + int64_t(i) * epi.ldpre + j;
    if (vec) {
      *reinterpret_cast<float4*>(pr) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
      for (int e = 0; e < ne; ++e) pr[e] = v[e];
    }
  }
  float* ci = C + int64_t(i) * ldc;
  if (epi.act == 2) {  // N even: pairs (j, j + 1), (j + 2, j + 3)
    const float o0 = v[0] * sig_fast(v[1]), o1 = v[2] * sig_fast(v[3]);
    if (vec) {
      *reinterpret_cast<float2*>(ci + j / 2) = make_float2(o0, o1);
    } else {
      ci[j / 2] = o0;
      if (ne > 2) ci[j / 2 + 1] = o1;
    }
    return;
  }
  if (epi.act == 1) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = v[e] * sig_fast(v[e]);
  }
  if (vec) {
    *reinterpret_cast<float4*>(ci + j) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    for (int e = 0; e < ne; ++e) ci[j + e] = v[e];
  }
}

// The K loop's barrier: no memory fence, since any fence, even one on LDS
// alone, makes the compiler wait for every global-to-LDS load in flight (the
// prefetches too). The loop's own vmcnt wait before it covers the step's
// loads; an explicit lgkmcnt(0) wait (vmcnt and expcnt left at their maxima)
// makes every LDS read a wave issued in the step before complete before it
// passes, so no wave's global_load_lds can overwrite a stage another is still
// reading, whatever order the compiler gives the products; the empty asm
// keeps the compiler from moving memory accesses across it.
__device__ __forceinline__ void ring_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}


// 16 bytes a lane from global memory into LDS, a wave's 64 lanes filling
// dst .. dst + 1 KB in lane order (dst wave-uniform). A device function: the
// builtin, called in a lambda of a kernel, stops the host side from emitting
// the kernel.
__device__ __forceinline__ void ring_load(const u4* src, u4* dst) {
  __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
}

// s_waitcnt on the vector-memory counter alone (gfx9 encoding: vmcnt in bits
// 3:0 and 15:14; expcnt 7 and lgkmcnt 15 wait for nothing).
template <int n>
__device__ __forceinline__ void wait_vm() {
  __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
}

}  // namespace pet_gemm

// gemm_rows.hip: C = epilogue(A B^T) from three-part weights (pet_gemm_pair_weights)
int pet_gemm_nt_p3(int M, int N, int K, const float* A, int64_t lda, const void* Bp, float* C, int64_t ldc,
                   const pet_gemm::Epi& e, hipStream_t st);
// ... and on the row kernels, P parts of weights a value; as: how A comes
enum { kRowsOnline = 0, kRowsExact = 1, kRowsPairs = 2 };
int pet_gemm_nt_rows(int M, int N, int K, const void* A, int64_t lda, int as, int kb, const void* Bp, int P, float* C,
                     int64_t ldc, const pet_gemm::Epi& e, hipStream_t st, int cfg);
